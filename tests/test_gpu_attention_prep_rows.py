"""GPU test of the launches that bring queries, keys and values of many rows from their projections to the attention: rows on both sides of the line at 64, rotations
shorter and longer than 128 channels, value channels on and off the grid of eight and of a workgroup's 64 -- one-layer models against the float64 oracle, the same bound as
the model's other tests."""
import numpy as np
import pytest

from tests import febivik_oracle as fo
from tests.test_gpu_febivik import TOL, engine, model_folder, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('H,G,D,V,rot', [(4, 2, 32, 24, 16), (6, 3, 136, 72, 136), (3, 1, 16, 20, 0), (2, 1, 160, 8, 144)])
def test_rows(cuda, tmp_path, H, G, D, V, rot, dtype):
    cfg = fo.make_config(48, 61, [fo.attention_layer(H, G, D, V, D ** -0.5, 300, 5, rot, 3000.0, 2.0)])
    folder, w = model_folder(tmp_path, cfg, 4)
    rng = np.random.default_rng(D)
    eng = engine(folder, dtype, max_prefill_token_num=1100, cache_blocks=40)
    for lens in ((63,), (64,), (511, 512), (512, 512), (340, 350, 345)):
        reqs = [rng.integers(0, 61, n).tolist() for n in lens]
        sess = [eng.open_session() for _ in reqs]
        got = eng.step_tokens([(s, r, list(range(len(r)))) for s, r in zip(sess, reqs)])
        for s in sess:
            eng.close_session(s)
        assert rel_err(got, np.concatenate([fo.forward(cfg, w, r) for r in reqs])) <= TOL[dtype], lens
    eng.close()
