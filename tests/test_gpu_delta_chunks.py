"""GPU test of the delta rule's prompt portions in chunks on the matrix cores: portions on both sides of the chunks of 16 tokens and of the line to the token-by-token
kernel, with decoded tokens in between, head sizes on every row-tile count, a token that comes again and again (what one key writes the next erases, so every
factor of the triangular system counts), against the float64 model of tests/febivik_oracle.py."""
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
@pytest.mark.parametrize('same', [False, True])
@pytest.mark.parametrize('heads,dim', [(2, 12), (3, 33), (1, 64), (2, 100), (1, 128), (1, 200), (1, 256)])
def test_portions_around_the_chunks(cuda, tmp_path, heads, dim, same, dtype):
    cfg = fo.make_config(48, 61, [fo.delta_layer(heads, dim, 8)])
    sizes = [17, 2, 1, 16, 33, 1, 1, 31, 48]
    toks = [7] * sum(sizes) if same else np.random.default_rng(6).integers(0, 61, sum(sizes)).tolist()
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
def test_sequences_of_all_lengths_in_a_launch(cuda, tmp_path, dtype):
    """chunks of a sequence count from its first row; sequences with no whole chunk, one and several"""
    cfg = fo.make_config(48, 61, [fo.delta_layer(2, 72, 8)])
    lens = [5, 40, 2, 16, 17, 64, 100]
    rng = np.random.default_rng(3)
    folder, w = model_folder(tmp_path, cfg, 9)
    reqs = [rng.integers(0, 61, n).tolist() for n in lens]
    ref = np.concatenate([fo.forward(cfg, w, r, True)[1][0] for r in reqs])
    eng = engine(folder, dtype, max_batch_size=len(lens), cache_blocks=20)
    eng.stop_after(1)
    sess = [eng.open_session() for _ in reqs]
    eng.step_tokens([(s, r, []) for s, r in zip(sess, reqs)])
    assert np.abs(eng.fetch_residual(sum(lens)) - ref).max() <= TOL[dtype] * 3 * np.abs(ref).max()
    eng.close()


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_many_heads_are_walked(cuda, tmp_path, dtype):
    """heads x sequences that fill the chip: portions beyond 32 tokens one token after the other, and in chunks again for a single sequence"""
    cfg = fo.make_config(48, 61, [fo.delta_layer(32, 256, 8)])
    rng = np.random.default_rng(4)
    folder, w = model_folder(tmp_path, cfg, 11)
    reqs = [rng.integers(0, 61, n).tolist() for n in (33, 40, 35, 36)]
    eng = engine(folder, dtype, max_batch_size=len(reqs), cache_blocks=20)
    eng.stop_after(1)
    tol = TOL[dtype] * 3

    def check(sess, toks, ref):
        eng.step_tokens([(s, t, []) for s, t in zip(sess, toks)])
        assert np.abs(eng.fetch_residual(len(ref)) - ref).max() <= tol * np.abs(ref).max()
    refs = [fo.forward(cfg, w, r + r[:34], True)[1][0] for r in reqs]
    sess = [eng.open_session() for _ in reqs]
    check(sess, reqs, np.concatenate([f[:len(r)] for f, r in zip(refs, reqs)]))
    check(sess[:1], [reqs[0][:34]], refs[0][33:67])
    eng.close()
