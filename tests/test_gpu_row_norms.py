"""GPU tests of the row norms over an fp32 stream at the borders of their register variants: RMS norm with one and two weight vectors (through
the C-ABI), layer norm with and without the sum into the stream, and the gated output norm of the state mixers in one group and head by head (both
inside one-layer models, against the float64 model of tests/febivik_oracle.py)."""
import numpy as np
import pytest

from lmdeploy_amd import _ffi
from tests import febivik_oracle as fo
from tests.gpu_helpers import dev, release_all, st
from tests.test_gpu_febivik import TOL, act, engine, model_folder, read

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('dtype', [0, 1])
@pytest.mark.parametrize('pair', [True, False])
@pytest.mark.parametrize('H', [4, 1020, 1024, 1028, 2048, 2052, 4096, 4100, 8192, 8196, 1026])
def test_rmsnorm_register_variants(tm, cuda, H, pair, dtype):
    rng = np.random.default_rng(H)
    M, ld = 3, (H + 31) // 32 * 32
    x = rng.normal(0, 3, (M + 2, H)).astype(np.float32)
    w = rng.normal(0, 0.2, (2, H)).astype(np.float32)
    rows = np.asarray([4, 0, 2], np.int32)
    for shift in (0, 1):                                      # an input that starts off the 16-byte grid
        buf = np.concatenate([np.zeros(shift, np.float32), x.ravel()])
        xd, wd, rd = dev(buf), [dev(w[0]), dev(w[1])], dev(rows)
        y = [act(np.full((M, ld), 7.0), dtype) for _ in range(2)]
        _ffi.check(tm.tm_rmsnorm_f32(y[0].data_ptr(), y[1].data_ptr() if pair else None, ld, 2 if dtype == 0 else 4, xd.data_ptr() + 4 * shift,
                                     rd.data_ptr(), wd[0].data_ptr(), wd[1].data_ptr() if pair else None, 1.0, 1e-5, M, H, st()))
        xr = x[rows].astype(np.float64)
        base = xr / np.sqrt((xr * xr).mean(-1, keepdims=True) + 1e-5)
        for i in range(2 if pair else 1):
            ref = base * (1.0 + w[i].astype(np.float64))
            # fp32: a sum of H squares in partial sums of at most 64 terms, a root, three products: under 40 units in the last place; bf16: half of 2^-8
            assert (np.abs(read(y[i], dtype)[:, :H] - ref) <= (2.0 ** -8 if dtype == 0 else 40 * 2.0 ** -24) * np.abs(ref) + 1e-30).all()
            assert (read(y[i], dtype)[:, H:] == 7.0).all()    # nothing behind the row
        if not pair:
            assert (read(y[1], dtype) == 7.0).all()


CASES = {f'width_{H}': (H, lambda: fo.lightning_layer(2, 8, 8, [0.9, 0.95])) for H in (1024, 1028, 2052, 4100, 8196, 1030)}
CASES.update({f'one_group_{h * v}': (32, lambda h=h, v=v: fo.lightning_layer(h, 8, v, [0.9] * h))
              for h, v in ((8, 256), (27, 76), (41, 100), (41, 200), (3, 25))})
CASES.update({f'groups_{h}_of_{d}': (32, lambda h=h, d=d: fo.delta_layer(h, d, 4)) for h, d in ((5, 4), (6, 252), (3, 256), (2, 50), (9, 64))})


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('name', list(CASES))
def test_layer_norm_and_gated_norm_register_variants(cuda, tmp_path, name, dtype):
    width, layer = CASES[name]
    cfg = fo.make_config(width, 61, [layer()])
    toks = np.random.default_rng(2).integers(0, 61, 9).tolist()
    folder, w = model_folder(tmp_path, cfg, 5)
    _, trail = fo.forward(cfg, w, toks, True)
    eng = engine(folder, dtype, session_len=64, max_prefill_token_num=64)
    eng.stop_after(1)
    s = eng.open_session()
    eng.step_tokens([(s, toks, [])])
    got = eng.fetch_residual(len(toks))
    eng.close_session(s)
    eng.close()
    assert np.abs(got - trail[0]).max() <= TOL[dtype] * 3 * np.abs(trail[0]).max()    # the tolerance of the one-layer models there
