"""GPU test of the launches that bring queries, keys and values of many rows from their projections to the attention: rows on both sides of a workgroup's 64 and of the line at a
million values, rotations shorter and longer than 128 channels, value channels on and off the grid of eight and of a workgroup's 64 -- one-layer models against the float64
oracle, the same bound as the model's other tests."""
import functools

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


@functools.lru_cache(None)
def _million(H, G, D, V, rot, rows):
    """(model, requests side by side in a forward, their logits)"""
    cfg = fo.make_config(48, 61, [fo.attention_layer(H, G, D, V, D ** -0.5, 300, 5, rot, 3000.0, 2.0)])
    w, rng = fo.random_weights(cfg, 4), np.random.default_rng(D)
    steps = [[rng.integers(0, 61, n).tolist() for n in lens] for lens in ((rows - 1, ), (511, rows - 511))]
    return cfg, w, steps, [np.concatenate([fo.forward(cfg, w, r) for r in reqs]) for reqs in steps]


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('H,G,D,V,rot,rows', [(42, 42, 8, 24, 8, 993), (14, 14, 136, 72, 136, 993), (16, 8, 16, 128, 16, 977), (17, 17, 8, 60, 0, 981)])
def test_a_million_values(cuda, tmp_path, H, G, D, V, rot, rows, dtype):
    """from as many rows on the values have a launch of their own (the last model's, not made of pieces of eight, never)"""
    cfg, w, steps, refs = _million(H, G, D, V, rot, rows)
    folder = str(tmp_path / 'm')
    fo.write_checkpoint(folder, cfg, w)
    eng = engine(folder, dtype, max_prefill_token_num=1100, cache_blocks=40, session_len=1024)
    for reqs, ref in zip(steps, refs):
        sess = [eng.open_session() for _ in reqs]
        got = eng.step_tokens([(s, r, list(range(len(r)))) for s, r in zip(sess, reqs)])
        for s in sess:
            eng.close_session(s)
        assert rel_err(got, ref) <= TOL[dtype], len(reqs)
    eng.close()
