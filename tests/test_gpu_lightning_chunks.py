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
