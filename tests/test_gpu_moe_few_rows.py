"""GPU tests of routed experts over few tokens on both sides of the row tiles that an expert's product takes: all tokens at the same experts, so that one
expert holds exactly as many rows as there are tokens, and spread ones -- the stream behind a one-layer model against the float64 oracle."""
import numpy as np
import pytest

from tests import febivik_oracle as fo
from tests.test_gpu_febivik import TOL, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('n', [1, 16, 17, 32, 33, 64, 65])
@pytest.mark.parametrize('same', [False, True])
def test_rows_of_an_expert(tmp_path, cuda, n, same, dtype):
    experts = 5 if dtype == 'float32' else 3
    cfg = fo.make_config(64, 97, [fo.lightning_layer(2, 8, 8, [0.9, 0.9], fo.moe(experts, 2 if dtype == 'float32' else experts, 40, 1.0, 24))])
    w = fo.random_weights(cfg, n)
    folder = str(tmp_path / 'm')
    fo.write_checkpoint(folder, cfg, w)
    rng = np.random.default_rng(n)
    reqs = [[7, 7, 7] if same else rng.integers(0, 97, 3).tolist() for _ in range(n)]
    eng = engine(folder, dtype, max_batch_size=n, cache_blocks=n + 2)
    sess = [eng.open_session() for _ in reqs]
    got = [eng.step_tokens([(s, r[i:i + 1], [0]) for s, r in zip(sess, reqs)]).reshape(n, -1) for i in range(3)]
    ref = np.stack([fo.forward(cfg, w, r) for r in reqs], axis=1)
    assert np.abs(np.stack(got) - ref).max() <= TOL[dtype] * np.abs(ref).max()
    eng.close()
