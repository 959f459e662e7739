"""GPU test of products whose last columns go to a launch of smaller tiles (gemm_stream.h): rows that fill a round of 256 x 256 tiles with a column tile or two
left over, a remainder of rows and of columns, every epilogue family, bf16 and fp16, with the bounds of the other stream kernels' tests."""
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


@pytest.mark.parametrize('K,N,M', [(512, 8448, 2040), (1024, 8450, 2048), (1024, 16640, 1030), (992, 33024, 500)])
def test_dense(tm, cuda, K, N, M):
    g = torch.Generator('cuda').manual_seed(K + N)
    w = torch.randn(N, K, generator=g, device='cuda').bfloat16()
    h = C.c_void_p()
    _ffi.check(tm.tm_dense_create(C.byref(h), K, N, 0, w.data_ptr(), st()))
    x = torch.randn(M, K, generator=g, device='cuda').bfloat16()
    ref, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    y = torch.full((M + 1, N + 6), -3.0, device='cuda', dtype=torch.bfloat16)
    _ffi.check(tm.tm_dense_forward(h, x.data_ptr(), K, y.data_ptr(), N + 6, M, 0, 1.0, st()))
    check(y[:M, :N], ref, size, K, True)
    assert bool((y[M] == -3.0).all()) and bool((y[:M, N:] == -3.0).all())
    r = torch.randn(M + 1, N, generator=g, device='cuda')
    keep, want = r[M].clone(), r[:M].double() + 0.25 * ref
    _ffi.check(tm.tm_dense_forward(h, x.data_ptr(), K, r.data_ptr(), N, M, 2, 0.25, st()))
    # fp32 sums of K products in any order, one multiplication and one addition
    assert bool(((r[:M].double() - want).abs() <= 0.25 * K * 2.0 ** -24 * size + 2.0 ** -22 * want.abs() + 2.0 ** -24 * ref.abs()).all()) and bool((r[M] == keep).all())
    _ffi.check(tm.tm_dense_destroy(h))


@pytest.mark.parametrize('K,N,M', [(512, 8448, 2040), (1024, 16672, 1030)])
@pytest.mark.parametrize('gated', [0, 1])
def test_fp16(tm, cuda, K, N, M, gated):
    g = torch.Generator('cuda').manual_seed(K + N)
    w = (torch.randn(K, N, generator=g, device='cuda') / K ** 0.5).half()
    h = C.c_void_p()
    _ffi.check(tm.tm_linear_create(C.byref(h), K, N, 1, 128))
    _ffi.check(tm.tm_linear_prepare(h, w.data_ptr(), None, None, st()))
    x = torch.randn(M, K, generator=g, device='cuda').half()
    ref = x.double() @ w.double()
    err = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs())
    if gated:
        a, b, ea, eb = ref[:, 0::2], ref[:, 1::2], err[:, 0::2], err[:, 1::2]
        ref = a / (1 + torch.exp(-a)) * b
        err = 1.1 * ea * b.abs() + a.abs() * eb + ea * eb + 2.0 ** -20 * ref.abs()     # (|silu'| <= 1.1, |silu(a)| <= |a|)
    n = ref.shape[1]
    ws = torch.zeros(max(1, tm.tm_linear_workspace(h, M)), dtype=torch.uint8, device='cuda')
    y = torch.full((M + 1, n), -3.0, device='cuda', dtype=torch.half)
    _ffi.check(tm.tm_linear_forward(h, x.data_ptr(), K, y.data_ptr(), n, M, gated, 0, 0, 0, ws.data_ptr(), st()))
    assert bool(((y[:M].double() - ref).abs() <= err + 2.0 ** -11 * ref.abs() + 2.0 ** -24).all()) and bool((y[M] == -3.0).all())
    _ffi.check(tm.tm_linear_destroy(h))
