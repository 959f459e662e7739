"""GPU test of the few-row products whose workgroups cover 96 columns (gemm_stream.h): column counts that leave a part of the last workgroup, one and several
slices of k, one, two and four row tiles, three number formats, with the bounds of the other stream kernels' tests."""
import ctypes as C

import pytest
import torch

from lmdeploy_amd import _ffi
from tests.gpu_helpers import release_all, st
from tests.test_gpu_stream import check

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('dtype', [0, 1])
@pytest.mark.parametrize('K,N', [(520, 20010), (1024, 21504), (96, 24500)])
def test_one_slice(tm, cuda, dtype, K, N):
    g = torch.Generator('cuda').manual_seed(K + N)
    w = torch.randn(N, K, generator=g, device='cuda').bfloat16()
    h = C.c_void_p()
    _ffi.check(tm.tm_dense_create(C.byref(h), K, N, dtype, w.data_ptr(), st()))
    T = torch.bfloat16 if dtype == 0 else torch.float32
    ldx = (K + 31) // 32 * 32
    for M in (9, 17, 33, 64):
        x = torch.zeros((M, ldx), device='cuda', dtype=T)
        x[:, :K] = torch.randn(M, K, generator=g, device='cuda').to(T)
        ref, size = x[:, :K].double() @ w.double().t(), x[:, :K].double().abs() @ w.double().abs().t()
        y = torch.full((M + 1, N + 3), -3.0, device='cuda', dtype=T)
        _ffi.check(tm.tm_dense_forward(h, x.data_ptr(), ldx, y.data_ptr(), N + 3, M, 0, 1.0, st()))
        check(y[:M, :N], ref, size, K, dtype == 0)
        assert bool((y[M] == -3.0).all()) and bool((y[:M, N:] == -3.0).all())
    _ffi.check(tm.tm_dense_destroy(h))


@pytest.mark.parametrize('K,N', [(4096, 6144), (4096, 6112), (2048, 12288), (1024, 20480)])
def test_slices_fp16(tm, cuda, K, N):
    g = torch.Generator('cuda').manual_seed(K + N)
    w = (torch.randn(K, N, generator=g, device='cuda') / K ** 0.5).half()
    h = C.c_void_p()
    _ffi.check(tm.tm_linear_create(C.byref(h), K, N, 1, 128))
    _ffi.check(tm.tm_linear_prepare(h, w.data_ptr(), None, None, st()))
    for M in (8, 24, 40, 64):
        x = torch.randn(M, K, generator=g, device='cuda').half()
        ref, size = x.double() @ w.double(), x.double().abs() @ w.double().abs()
        ws = torch.zeros(max(1, tm.tm_linear_workspace(h, M)), dtype=torch.uint8, device='cuda')
        y = torch.full((M + 1, N), -3.0, device='cuda', dtype=torch.half)
        _ffi.check(tm.tm_linear_forward(h, x.data_ptr(), K, y.data_ptr(), N, M, 0, 0, 0, 0, ws.data_ptr(), st()))
        # fp32 sums of K products in any order, one rounding to fp16
        assert bool(((y[:M].double() - ref).abs() <= K * 2.0 ** -24 * size + 2.0 ** -11 * ref.abs() + 2.0 ** -24).all())
        assert bool((y[M] == -3.0).all())
    _ffi.check(tm.tm_linear_destroy(h))
