"""GPU test of the W4 products of up to 16 rows that keep their rows in LDS and apply scales and zero points to sums (gemm_w4_rows.hip): its four workgroup shapes, column
groups and k-blocks that leave waves without work, slices of unequal length, the two ways the row sums are made, plain and gated results, rows with strides -- against
64-bit results, which it has to be as close to as the kernel that rounds its weights, and the rule that takes it."""
import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from oracle import tm_oracle as o
from tests.gpu_helpers import dev, host, release_all, st
from tests.test_gpu_ops import _QCACHE, _make_linear

pytestmark = pytest.mark.gpu
ROWS = 14


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


def _run(tm, h, x, N, M, shape, splits, gated=0):
    cols = N // 2 if gated else N
    y = torch.full((M + 1, cols + 4), 7.0, dtype=torch.float16, device='cuda')
    ws = torch.zeros(max(1, tm.tm_linear_workspace(h, M)), dtype=torch.uint8, device='cuda')
    _ffi.check(tm.tm_linear_forward(h, dev(x).data_ptr(), x.shape[1], y.data_ptr(), cols + 4, M, gated, 0, splits, 0x200 | shape, ws.data_ptr(), st()))
    y = host(y)
    assert (y[M] == 7.0).all() and (y[:M, cols:] == 7.0).all()
    return y[:M, :cols].astype(np.float64)


# sizes whose shapes are 1 x 8, 2 x 4, 2 x 8 and 4 x 4 waves (column groups of 32 x k-phases) and their neighbours
@pytest.mark.parametrize('K,N,splits,gated', [
    (128, 32, 1, 0), (384, 96, 1, 1), (2048, 4096, 1, 0), (2304, 4128, 2, 0), (2048, 10272, 1, 1), (2048, 2048, 4, 0), (4096, 10240, 1, 1), (4096, 4096, 4, 0),
    (4224, 5152, 4, 0), (2048, 28704, 1, 1), (8192, 2048, 8, 0), (8320, 608, 8, 0), (14336, 512, 4, 0)])
@pytest.mark.parametrize('M', [1, 3, 8, 9, 16])
def test_against_64_bits(tm, cuda, K, N, splits, gated, M):
    rng = np.random.default_rng(K + N + M)
    h, _ = _make_linear(tm, rng, K, N)
    q, s, z = _QCACHE[(K, N)][:3]
    x = rng.standard_normal((M, K + 8)).astype(np.float16)
    x[:, ::7] *= 30
    w = q * np.repeat(s.astype(np.float64), 128, 0) + np.repeat((-z * s).astype(np.float16).astype(np.float64), 128, 0)
    ref = x[:, :K].astype(np.float64) @ w
    if gated:
        ref = ref[:, ::2] / (1 + np.exp(-ref[:, ::2])) * ref[:, 1::2]
    got, other = _run(tm, h, x, N, M, ROWS, splits, gated), _run(tm, h, x, N, M, 0, splits, gated)
    _ffi.check(tm.tm_linear_destroy(h))
    rms = np.sqrt((ref**2).mean())
    assert np.sqrt(((got - ref)**2).mean()) <= 1.02 * np.sqrt(((other - ref)**2).mean())
    assert (np.abs(got - ref) <= 2.0**-11 * np.abs(ref) + 2.0**-9 * rms).all()    # one rounding to fp16; sums of 1039 |x| in fp32 beside results of about 52


@pytest.mark.parametrize('K,N,splits,gated', [(2048, 4096, 1, 0), (2304, 4128, 2, 0), (2048, 2048, 4, 1), (4096, 10240, 1, 1), (2048, 28704, 1, 0)])
@pytest.mark.parametrize('M', [1, 4, 16])
def test_infinities(tm, cuda, K, N, splits, gated, M):
    """a row with infinities has the infinities and NaN that its weights give it, as in the kernel that makes them; the other rows keep their bits"""
    rng = np.random.default_rng(K + N + M)
    h, _ = _make_linear(tm, rng, K, N)
    x = rng.standard_normal((M, K + 8)).astype(np.float16)
    plain = _run(tm, h, x, N, M, ROWS, splits, gated)
    rows = [0] if M == 1 else [1, M - 1]
    x[rows[0], [5, 131]] = np.inf, -np.inf
    for r in rows[1:]:
        x[r, K - 3] = -np.inf
    got, other = _run(tm, h, x, N, M, ROWS, splits, gated), _run(tm, h, x, N, M, 0, splits, gated)
    _ffi.check(tm.tm_linear_destroy(h))
    left = np.setdiff1d(np.arange(M), rows)
    assert np.array_equal(got[left], plain[left]) and not np.isfinite(got[rows]).any()
    if not gated:
        assert np.isinf(got[rows]).any()
    same = np.where(np.isnan(got[rows]), 0, got[rows]) == np.where(np.isnan(other[rows]), 0, other[rows])
    assert same.all()


def test_a_named_shape_runs_or_is_refused(tm, cuda):
    """rows beyond LDS, slices without k-blocks, and a launch whose slices would be dropped for want of a workspace"""
    rng = np.random.default_rng(1)
    for K, M, splits, ws, ok in ((14336, 16, 1, True, False), (14336, 16, 4, True, True), (14336, 16, 4, False, False), (14336, 4, 4, False, True), (2304, 8, 8, True, False)):
        h, _ = _make_linear(tm, rng, K, 64)
        x, y = dev(rng.standard_normal((M, K)).astype(np.float16)), torch.full((M, 64), 7.0, dtype=torch.float16, device='cuda')
        buf = torch.zeros(tm.tm_linear_workspace(h, M), dtype=torch.uint8, device='cuda')
        rc = tm.tm_linear_forward(h, x.data_ptr(), K, y.data_ptr(), 64, M, 0, 0, splits, 0x200 | ROWS, buf.data_ptr() if ws else None, st())
        assert (rc == 0) == ok and (ok or (host(y) == 7.0).all()), (K, M, splits, ws)
        assert tm.tm_linear_forward(h, x.data_ptr(), K, y.data_ptr(), 64, M, 0, 0, splits, 0, buf.data_ptr() if ws else None, st()) == 0    # (no shape named)
        _ffi.check(tm.tm_linear_destroy(h))


def _residual(tm, h, x, N, M, shape, splits):
    rng = np.random.default_rng(M)
    r, g = dev(rng.standard_normal((M, N)).astype(np.float16)), dev(rng.choice([0.5, 1, 2], N).astype(np.float16))
    y, before = torch.zeros((M, N), dtype=torch.float16, device='cuda'), host(r).astype(np.float64)
    ws = torch.zeros(tm.tm_linear_workspace(h, M) + 2 * M * N, dtype=torch.uint8, device='cuda')
    _ffi.check(tm.tm_linear_residual_norm(h, dev(x).data_ptr(), x.shape[1], y.data_ptr(), r.data_ptr(), g.data_ptr(), 1e-5, M, shape, splits, ws.data_ptr(), st()))
    return host(r).astype(np.float64), host(y).astype(np.float64), before, host(g).astype(np.float64)


@pytest.mark.parametrize('K,N,M,splits', [(2304, 2144, 8, 1), (2304, 2144, 8, 2), (2304, 2144, 13, 4), (4096, 512, 1, 4)])
def test_slabs_and_the_norm_behind_them(tm, cuda, K, N, M, splits):
    """the row kernel's slabs through the launch that adds them to the residual stream and makes its norm, as an engine runs them"""
    rng = np.random.default_rng(K + N + M)
    h, _ = _make_linear(tm, rng, K, N)
    q, s, z = _QCACHE[(K, N)][:3]
    x = (3 * rng.standard_normal((M, K))).astype(np.float16)
    r, y, before, g = _residual(tm, h, x, N, M, ROWS, splits)
    _ffi.check(tm.tm_linear_destroy(h))
    ref = before + x.astype(np.float64) @ (q * np.repeat(s.astype(np.float64), 128, 0) + np.repeat((-z * s).astype(np.float16).astype(np.float64), 128, 0))
    rms = np.sqrt((ref**2).mean(1, keepdims=True))
    assert (np.abs(r - ref) <= 2.0**-10 * np.abs(ref) + 2.0**-9 * rms).all()            # the product's rounding to fp16 and the sum's
    norm = r / np.sqrt((r**2).mean(1, keepdims=True) + 1e-5) * g
    assert (np.abs(y - norm) <= 2.0**-9 * np.abs(norm) + 2.0**-14).all()                # two roundings to fp16, a row sum in fp32


def test_the_residual_stream_keeps_its_tile_with_a_line(tm, cuda, tmp_path):
    """a measured line that names the row kernel is the engine's: tm_linear_residual_norm has the bits that it has without one"""
    K, N, M = 2432, 2208, 8
    rng = np.random.default_rng(2)
    h, _ = _make_linear(tm, rng, K, N)
    x = rng.standard_normal((M, K)).astype(np.float16)
    first = _residual(tm, h, x, N, M, -1, 0)
    assert not np.array_equal(first[0], _residual(tm, h, x, N, M, ROWS, 2)[0])          # (or this would show nothing)
    f = tmp_path / 't.txt'
    f.write_text(f'{K} {N} {M} {ROWS} 2\n')
    assert tm.tm_gemm_import(str(f).encode()) == 0
    again = _residual(tm, h, x, N, M, -1, 0)
    _ffi.check(tm.tm_linear_destroy(h))
    assert np.array_equal(first[0], again[0]) and np.array_equal(first[1], again[1])


def test_what_a_launch_takes(tm, cuda):
    def pick(K, N, M):
        sh, sp = _ffi.C.c_int(), _ffi.C.c_int()
        _ffi.check(tm.tm_debug_pick_tiling(K, N, M, 4, _ffi.C.byref(sh), _ffi.C.byref(sp)))
        return sh.value, sp.value
    for K, N, M, want in ((4096, 28672, 1, (ROWS, 1)), (4096, 6144, 8, (ROWS, 2)), (4096, 4096, 16, (ROWS, 4)), (14336, 4096, 8, None), (14336, 4096, 9, (3, 4)), (4096, 6144, 17, (3, 2)),
                          (4096, 768, 4, (ROWS, 4))):
        assert pick(K, N, M) == want if want else pick(K, N, M)[0] == ROWS, (K, N, M)
