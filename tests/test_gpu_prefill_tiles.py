"""GPU test of the 256 x 256 W4 prefill tile (gemm_prefill.hip): row and column counts on both sides of its edges, one k-block, odd and even counts of them,
slices of k, rows of the output that start on 16 bytes and rows that do not, plain and gated; and of the rule that chooses it, against the oracle."""
import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from oracle import tm_oracle as o
from tests.gpu_helpers import dev, host, release_all, st
from tests.test_gpu_ops import _QCACHE, _make_linear

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('K,N', [(128, 256), (256, 32), (384, 288), (640, 544), (1792, 224)])
@pytest.mark.parametrize('M', [65, 255, 256, 257, 600])
@pytest.mark.parametrize('gated', [0, 1])
def test_tile_edges(tm, cuda, K, N, M, gated):
    rng = np.random.default_rng(K + N + M)
    h, (q, s, z) = _make_linear(tm, rng, K, N)
    x = rng.standard_normal((M, K)).astype(np.float16)
    ref = (o.w4a16_linear_gated_silu(x, q, s, z) if gated else x.astype(np.float32) @ _QCACHE[(K, N)][3]).astype(np.float32)
    cols = N // 2 if gated else N
    ws = torch.zeros(max(1, tm.tm_linear_workspace(h, M)), dtype=torch.uint8, device='cuda')
    x_d = dev(x)
    for splits in (1, 2, 3):
        if splits > K // 128:
            continue
        for ldy in (cols, cols + 4, cols + 8):
            y = torch.full((M + 1, ldy), 7.0, dtype=torch.float16, device='cuda')
            _ffi.check(tm.tm_linear_forward(h, x_d.data_ptr(), K, y.data_ptr(), ldy, M, gated, 0, splits, 0x20c, ws.data_ptr(), st()))
            got = host(y).astype(np.float32)
            assert (np.abs(got[:M, :cols] - ref) <= 2e-3 + 2.0**-9 * np.abs(ref)).all(), (splits, ldy)   # the bound of the other prefill tiles
            assert (got[M] == 7.0).all() and (got[:M, cols:] == 7.0).all()
    _ffi.check(tm.tm_linear_destroy(h))


@pytest.mark.parametrize('K,N,M', [(128, 8192, 2049), (256, 6144, 2604), (256, 16384, 257), (128, 512, 4100), (256, 4096, 4096)])
def test_picked_prefill_tile(tm, cuda, K, N, M):
    """sizes where the rule takes 128 x 256, 128 x 512 and 256 x 256 tiles: the same sums"""
    rng = np.random.default_rng(K + N + M)
    h, _ = _make_linear(tm, rng, K, N)
    x = rng.standard_normal((M, K)).astype(np.float16)
    ws = torch.zeros(max(1, tm.tm_linear_workspace(h, M)), dtype=torch.uint8, device='cuda')
    y = torch.zeros((M, N), dtype=torch.float16, device='cuda')
    _ffi.check(tm.tm_linear_forward(h, dev(x).data_ptr(), K, y.data_ptr(), N, M, 0, 0, 0, 0, ws.data_ptr(), st()))
    ref = x.astype(np.float32) @ _QCACHE[(K, N)][3]
    assert (np.abs(host(y).astype(np.float32) - ref) <= 2e-3 + 2.0**-9 * np.abs(ref)).all()
    _ffi.check(tm.tm_linear_destroy(h))


@pytest.mark.parametrize('K,N,M,shape', [(512, 8192, 2048, 12), (512, 6144, 2604, 5)])
def test_reported_tile_runs(tm, cuda, K, N, M, shape):
    """The tile that is reported for a size is the one that runs there, and an explicit shape runs that shape wherever the rule would take the other: the 256 x 256
    tile adds the 32 channels of a step in another order than the 128 x 512 tile, so their results differ in single roundings."""
    rng = np.random.default_rng(N)
    h, _ = _make_linear(tm, rng, K, N)
    sh, sp = _ffi.C.c_int(-1), _ffi.C.c_int(-1)
    _ffi.check(tm.tm_debug_pick_tiling(K, N, M, 2, _ffi.C.byref(sh), _ffi.C.byref(sp)))
    assert (sh.value, sp.value) == (shape, 1)
    x = rng.standard_normal((M, K)).astype(np.float16)
    ws = torch.zeros(max(1, tm.tm_linear_workspace(h, M)), dtype=torch.uint8, device='cuda')
    x_d, ys = dev(x), []
    for code in (0, 0x205, 0x20c):
        y = torch.zeros((M, N), dtype=torch.float16, device='cuda')
        _ffi.check(tm.tm_linear_forward(h, x_d.data_ptr(), K, y.data_ptr(), N, M, 0, 0, 1 if code else 0, code, ws.data_ptr(), st()))
        ys.append(y)
    ref = x.astype(np.float32) @ _QCACHE[(K, N)][3]
    for y in ys:
        assert (np.abs(host(y).astype(np.float32) - ref) <= 2e-3 + 2.0**-9 * np.abs(ref)).all()
    assert not torch.equal(ys[1], ys[2])
    assert torch.equal(ys[0], ys[1] if shape == 5 else ys[2])
    _ffi.check(tm.tm_linear_destroy(h))
