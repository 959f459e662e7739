"""GPU tests of the expert routing of a few tokens (masks of tokens per expert) at the borders of its range: 64 and 65 tokens in a forward, experts on
one and on several registers of a lane and just beyond what it serves, one and many choices, with and without the shared rows behind the routed ones, row
widths on and off the 16-byte grid -- one-layer models against the float64 model of tests/febivik_oracle.py."""
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
    ('float32', 32, 64, 3, 0), ('float32', 32, 65, 1, 16), ('float32', 36, 130, 5, 16), ('float32', 32, 256, 7, 0), ('float32', 32, 257, 2, 16),
    ('float32', 30, 1, 1, 16), ('float32', 32, 9, 9, 16), ('bfloat16', 40, 8, 8, 16), ('bfloat16', 44, 5, 5, 8)])
def test_forwards_of_few_tokens(cuda, tmp_path, dtype, width, experts, top, shared):
    cfg = fo.make_config(width, 61, [fo.lightning_layer(2, 8, 8, [0.9, 0.95], fo.moe(experts, top, 16, 1.3, shared))])
    toks = np.random.default_rng(4).integers(0, 61, 130).tolist()
    folder, w = model_folder(tmp_path, cfg, _clear_seed(cfg, toks, 'float32'))
    ref = fo.forward(cfg, w, toks, True)[1][0]
    eng = engine(folder, dtype)
    eng.stop_after(1)
    s, at = eng.open_session(), 0
    for n in (64, 1, 65):                                     # portions of the same sequence: the tables of 64, 1 and 65 tokens
        eng.step_tokens([(s, toks[at:at + n], [])])
        got = eng.fetch_residual(n)
        assert np.abs(got - ref[at:at + n]).max() <= TOL[dtype] * 3 * np.abs(ref).max(), (at, n)
        at += n
    eng.close_session(s)
    eng.close()
