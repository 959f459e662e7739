"""GPU tests of the launch that routes a few tokens and copies their rows to the experts' order: 64 and 65 tokens, as many choices as its list holds and one more, rows
of one load and several, off the 16-byte grid, one row of a workgroup's four -- one-layer models against the float64 model of tests/febivik_oracle.py."""
import numpy as np
import pytest

from tests import febivik_oracle as fo
from tests.gpu_helpers import release_all
from tests.test_gpu_febivik import TOL, _clear_seed, engine, model_folder

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('dtype,width,experts,top,shared', [
    ('float32', 32, 40, 32, 8), ('float32', 32, 40, 33, 0), ('float32', 1028, 6, 2, 16), ('float32', 1026, 4, 1, 0), ('bfloat16', 2064, 6, 2, 16), ('float32', 2052, 5, 3, 8)])
def test_forwards_of_few_tokens(cuda, tmp_path, dtype, width, experts, top, shared):
    cfg = fo.make_config(width, 61, [fo.lightning_layer(2, 8, 8, [0.9, 0.95], fo.moe(experts, top, 16, 1.3, shared))])
    toks = np.random.default_rng(5).integers(0, 61, 130).tolist()
    folder, w = model_folder(tmp_path, cfg, _clear_seed(cfg, toks, 'float32'))
    ref = fo.forward(cfg, w, toks, True)[1][0]
    eng = engine(folder, dtype)
    eng.stop_after(1)
    s, at = eng.open_session(), 0
    for n in (64, 1, 65):                                     # portions of the same sequence: one launch, one launch, a launch each
        eng.step_tokens([(s, toks[at:at + n], [])])
        got = eng.fetch_residual(n)
        assert np.abs(got - ref[at:at + n]).max() <= TOL[dtype] * 3 * np.abs(ref).max(), (at, n)
        at += n
    eng.close_session(s)
    eng.close()
