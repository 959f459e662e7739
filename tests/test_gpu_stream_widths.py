"""GPU test of the few-row products whose workgroups cover 96 columns (gemm_stream.h): column counts that leave a part of the last workgroup, one, two and four row
tiles, three number formats, in one slice of k and in several -- slabs that a launch adds, and slices that meet inside the launch of an engine -- with the bounds of
the other stream kernels' tests.  Every size says what it is meant to run: (kernel, column tiles a workgroup, row tiles, slices)."""
import ctypes as C

import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from tests import layered_oracle as lo
from tests.gpu_helpers import release_all, st
from tests.test_gpu_layered import TOL, _layer, engine_for, rel_err
from tests.test_gpu_stream import check
from tests.test_host import stream_plan

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('dtype,K,N,rows', [(0, 520, 20010, (24, 33, 64)), (0, 1024, 21504, (9, 16, 17, 32, 33, 64)), (0, 96, 24500, (64, )),
                                            (1, 520, 20010, (16, 32)), (1, 1024, 21504, (9, 16, 24, 32, 64)), (1, 256, 24500, (9, 17, 48, 64)), (1, 96, 24500, (16, 32))])
def test_one_slice(tm, cuda, dtype, K, N, rows):
    g = torch.Generator('cuda').manual_seed(K + N)
    w = torch.randn(N, K, generator=g, device='cuda').bfloat16()
    h = C.c_void_p()
    _ffi.check(tm.tm_dense_create(C.byref(h), K, N, dtype, w.data_ptr(), st()))
    T = torch.bfloat16 if dtype == 0 else torch.float32
    ldx = (K + 31) // 32 * 32
    for M in rows:
        assert stream_plan(dtype, K, N, M, 0)[:4] == (2, 6, 1 if M <= 16 else 2 if M <= 32 else 4, 1)
        x = torch.zeros((M, ldx), device='cuda', dtype=T)
        x[:, :K] = torch.randn(M, K, generator=g, device='cuda').to(T)
        ref, size = x[:, :K].double() @ w.double().t(), x[:, :K].double().abs() @ w.double().abs().t()
        y = torch.full((M + 1, N + 3), -3.0, device='cuda', dtype=T)
        _ffi.check(tm.tm_dense_forward(h, x.data_ptr(), ldx, y.data_ptr(), N + 3, M, 0, 1.0, st()))
        check(y[:M, :N], ref, size, K, dtype == 0)
        assert bool((y[M] == -3.0).all()) and bool((y[:M, N:] == -3.0).all())
    _ffi.check(tm.tm_dense_destroy(h))


@pytest.mark.parametrize('K,N,plans', [(4096, 6144, {24: (2, 4, 2, 2), 40: (2, 6, 4, 4), 64: (2, 6, 4, 4)}),
                                       (4096, 6112, {8: (1, 1, 1, 1), 16: (2, 6, 1, 4), 24: (2, 6, 2, 4), 64: (2, 6, 4, 4)}),
                                       (2048, 12288, {8: (2, 4, 1, 1), 64: (2, 4, 4, 1)}), (1024, 20480, {8: (2, 6, 1, 1), 24: (2, 6, 2, 1), 64: (2, 6, 4, 1)})])
def test_slices_fp16(tm, cuda, K, N, plans):
    g = torch.Generator('cuda').manual_seed(K + N)
    w = (torch.randn(K, N, generator=g, device='cuda') / K ** 0.5).half()
    h = C.c_void_p()
    _ffi.check(tm.tm_linear_create(C.byref(h), K, N, 1, 128))
    _ffi.check(tm.tm_linear_prepare(h, w.data_ptr(), None, None, st()))
    for M, plan in plans.items():
        assert stream_plan(2, K, N, M)[:4] == plan
        x = torch.randn(M, K, generator=g, device='cuda').half()
        ref, size = x.double() @ w.double(), x.double().abs() @ w.double().abs()
        ws = torch.zeros(max(1, tm.tm_linear_workspace(h, M)), dtype=torch.uint8, device='cuda')
        y = torch.full((M + 1, N), -3.0, device='cuda', dtype=torch.half)
        _ffi.check(tm.tm_linear_forward(h, x.data_ptr(), K, y.data_ptr(), N, M, 0, 0, 0, 0, ws.data_ptr(), st()))
        # fp32 sums of K products in any order, one rounding to fp16
        assert bool(((y[:M].double() - ref).abs() <= K * 2.0 ** -24 * size + 2.0 ** -11 * ref.abs() + 2.0 ** -24).all())
        assert bool((y[M] == -3.0).all())
    _ffi.check(tm.tm_linear_destroy(h))


@pytest.mark.parametrize('dtype,width,rows', [('bfloat16', 2080, (32, 33, 64)), ('float32', 2048, (9, 17, 64))])
def test_slices_that_meet_in_the_launch(cuda, dtype, width, rows):
    """the head of an engine: 6000 columns, three and four slices whose last workgroup of a column group adds them; the same rows again give the same bits"""
    cfg = lo.make_config(width, 6000, [_layer(heads=2, kv_heads=1, dim=8, vdim=8, ff=24)])
    w = lo.make_weights(cfg, 3)
    eng = engine_for(cfg, w, dtype, max_batch_size=64, cache_blocks=70)
    rng = np.random.default_rng(width)
    for n in rows:
        assert stream_plan(0 if dtype == 'bfloat16' else 1, width, 6000, n)[:4] == (2, 6, 1 if n <= 16 else 2 if n <= 32 else 4, 3 if dtype == 'bfloat16' else 4)
        toks, outs = rng.integers(0, 6000, n), []
        for _ in range(2):
            sess = [eng.open_session() for _ in range(n)]
            outs.append(eng.step_tokens([(s, toks[i:i + 1], [0]) for i, s in enumerate(sess)]).reshape(n, -1))
            for s in sess:
                eng.close_session(s)
        assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
        ref = np.concatenate([lo.forward(cfg, w, [int(t)])[0] for t in toks])
        assert rel_err(outs[0], ref) <= TOL[dtype] and rel_err(np.roll(ref, 96, axis=1), ref) > 10 * TOL[dtype]
    eng.close()
