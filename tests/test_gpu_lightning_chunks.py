"""GPU test of lightning attention's prompt portions on the matrix cores: portions that end on, before and behind the chunks of 16 tokens, with decoded
tokens in between, and head sizes on every row-tile count of the chunk kernels, against the float64 model of tests/febivik_oracle.py."""
import numpy as np
import pytest

from tests import febivik_oracle as fo
from tests.gpu_helpers import release_all
from tests.test_gpu_febivik import TOL, engine, model_folder

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('heads,dim,vdim', [(2, 12, 20), (3, 33, 16), (1, 64, 65), (2, 100, 128), (1, 200, 48), (1, 256, 17)])
def test_portions_around_the_chunks(cuda, tmp_path, heads, dim, vdim, dtype):
    cfg = fo.make_config(48, 61, [fo.lightning_layer(heads, dim, vdim, [0.99, 0.5, 0.9][:heads])])
    sizes = [15, 2, 1, 16, 17, 1, 1, 33, 31]
    toks = np.random.default_rng(6).integers(0, 61, sum(sizes)).tolist()
    folder, w = model_folder(tmp_path, cfg, 7)
    ref = fo.forward(cfg, w, toks, True)[1][0]
    eng = engine(folder, dtype)
    eng.stop_after(1)
    s, at = eng.open_session(), 0
    for n in sizes:
        eng.step_tokens([(s, toks[at:at + n], [])])
        got = eng.fetch_residual(n)
        assert np.abs(got - ref[at:at + n]).max() <= TOL[dtype] * 3 * np.abs(ref).max(), (at, n)   # the tolerance of the one-layer models there
        at += n
    eng.close_session(s)
    eng.close()


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('heads,dim,vdim', [(2, 12, 20), (3, 33, 16), (1, 64, 65), (2, 100, 128), (1, 128, 96)])
def test_portions_around_the_line_between_the_walks(cuda, tmp_path, heads, dim, vdim, dtype):
    """48 tokens are walked without LDS, 49 through it; a state that the one leaves is the other's"""
    cfg = fo.make_config(48, 61, [fo.lightning_layer(heads, dim, vdim, [0.99, 0.5, 0.9][:heads])])
    sizes = [48, 49, 1, 47, 64, 1, 65, 100, 16]
    toks = np.random.default_rng(8).integers(0, 61, sum(sizes)).tolist()
    folder, w = model_folder(tmp_path, cfg, 7)
    ref = fo.forward(cfg, w, toks, True)[1][0]
    eng = engine(folder, dtype, session_len=512, cache_blocks=8)
    eng.stop_after(1)
    s, at = eng.open_session(), 0
    for n in sizes:
        eng.step_tokens([(s, toks[at:at + n], [])])
        assert np.abs(eng.fetch_residual(n) - ref[at:at + n]).max() <= TOL[dtype] * 3 * np.abs(ref).max(), (at, n)
        at += n
    eng.close()


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_small_heads_that_fill_the_chip(cuda, tmp_path, dtype):
    """heads of few channels: the walk without LDS at any length from 1024 of them on"""
    cfg = fo.make_config(48, 61, [fo.lightning_layer(64, 8, 8, [0.9 + 0.001 * h for h in range(64)])])
    rng = np.random.default_rng(9)
    folder, w = model_folder(tmp_path, cfg, 5)
    reqs = [rng.integers(0, 61, 60 + s).tolist() for s in range(16)]
    ref = np.concatenate([fo.forward(cfg, w, r, True)[1][0] for r in reqs])
    eng = engine(folder, dtype, max_batch_size=16, cache_blocks=40, max_prefill_token_num=2048)
    eng.stop_after(1)
    eng.step_tokens([(eng.open_session(), r, []) for r in reqs])
    assert np.abs(eng.fetch_residual(len(ref)) - ref).max() <= TOL[dtype] * 3 * np.abs(ref).max()
    eng.close()
