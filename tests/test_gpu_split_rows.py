"""GPU tests of fp32 products (bf16 weights, fp32 rows that the kernels split into three bf16 parts, gemm_stream.h): the kernels of few rows, row blocks beside each other and both tiles, at
their edges, with a bound that needs every part and the short runs of steps; rows with infinities, NaN and numbers near the largest."""
import ctypes as C

import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from tests import layered_oracle as lo
from tests.gpu_helpers import release_all, st
from tests.test_gpu_layered import _layer, engine_for
from tests.test_host import stream_plan

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


def product(tm, w, x):
    N, K = w.shape
    M, ldx = x.shape
    h = C.c_void_p()
    _ffi.check(tm.tm_dense_create(C.byref(h), K, N, 1, w.data_ptr(), st()))
    y = torch.full((M + 1, N), -3.0, device='cuda')
    _ffi.check(tm.tm_dense_forward(h, x.data_ptr(), ldx, y.data_ptr(), N, M, 0, 1.0, st()))
    _ffi.check(tm.tm_dense_destroy(h))
    assert bool((y[M] == -3.0).all())
    return y[:M]


@pytest.mark.parametrize('sign', ['both', 'one'])
@pytest.mark.parametrize('K,N,rows', [
    (32, 130, (1, 16, 17, 64, 65, 129)),            # one step
    (264, 2052, (3, 33, 64, 200, 257, 700)),        # a run of eight steps and one of one, ragged columns
    (2080, 1030, (2, 31, 48, 90, 300)),             # slices of k are not to be had here: blocks of rows beside each other, 64 x 64 tiles
    (1024, 4100, (5, 2500)),                        # 128 x 128 tiles with ragged edges
    (8448, 260, (4, 40, 70))])
def test_every_part_counts(tm, cuda, K, N, rows, sign):
    """Products are exact, so the error is that of the sums: every run of eight steps is cut off 24 times at most, by 2^-23 of what it holds, and the runs, the waves' sums and the
    parts' sums are added in fp32: less than (48 + K / 256 + 24) 2^-24 sum |x w|.  A product that left the low part out would be off by 2^-17 |x w| a term"""
    g = torch.Generator('cuda').manual_seed(K + N)
    w = torch.randn(N, K, generator=g, device='cuda')
    w = (w.abs() if sign == 'one' else w).bfloat16()
    ldx = (K + 31) // 32 * 32 + 4
    for M in rows:
        x = torch.full((M, ldx), 5.0, device='cuda')
        x[:, :K] = torch.randn(M, K, generator=g, device='cuda').abs() + 0.01
        if sign == 'both':
            x[:, :K:2] *= -1
        ref, size = x[:, :K].double() @ w.double().t(), x[:, :K].double().abs() @ w.double().abs().t()
        err = (product(tm, w, x).double() - ref).abs()
        assert bool((err <= (72 + K / 256) * 2.0 ** -24 * size).all()), (M, float((err / size).max()) * 2 ** 24)
        if sign == 'one' and K >= 1024:      # ... and the mean shows no drift of long sums: each run's cuts are 24 of at most 2^-23, half of that each on average
            assert float((err / size).mean()) <= (24 + K / 256) * 2.0 ** -24, M


SLICED = {   # (K, N): rows and the plan they have in an engine: weight stream, column tiles a workgroup, row tiles, slices
    (2048, 250): {16: (2, 4, 1, 8), 17: (2, 4, 2, 8), 40: (2, 4, 4, 8), 65: (2, 4, 4, 8), 129: (2, 4, 4, 8), 256: (2, 4, 4, 8)},
    (2048, 770): {40: (2, 4, 4, 8), 90: (2, 4, 4, 8), 129: (2, 6, 4, 8), 200: (2, 4, 4, 4)},
    (8192, 2050): {3: (2, 6, 1, 8), 16: (2, 6, 1, 11), 24: (2, 6, 2, 11), 64: (2, 6, 4, 11), 90: (2, 6, 4, 11), 129: (2, 6, 4, 11), 200: (2, 6, 4, 8)}}


@pytest.mark.parametrize('sign', ['both', 'one'])
@pytest.mark.parametrize('K,N', SLICED)
def test_every_part_counts_in_slices(cuda, K, N, sign):
    """The head's product of an engine, which has scratch for slices of k: the logits of rows that are their embedding's norm.  As above, and the norm's own errors: its mean of squares within
    K / 256 + 8 roundings, half of that in its root, and four of each number"""
    cfg = lo.make_config(K, N, [_layer(heads=1, kv_heads=1, dim=8, vdim=8, ff=0)], logit_scale=1.0)
    w = lo.make_weights(cfg, K + N)
    w['l0.mix.o'][:] = 0
    if sign == 'one':
        w['embed'], w['head'], w['final.norm'] = (np.abs(w[k]) for k in ('embed', 'head', 'final.norm'))
    eng = engine_for(cfg, w, 'float32', max_batch_size=2)
    rng = np.random.default_rng(K)
    for M, plan in SLICED[K, N].items():
        assert stream_plan(1, K, N, M)[:4] == plan, (M, stream_plan(1, K, N, M))
        toks, got = rng.integers(0, N, M), []
        for _ in range(2):      # (arrival counters are back at zero)
            s = eng.open_session()
            got.append(eng.step_tokens([(s, toks, list(range(M)))]))
            eng.close_session(s)
        assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
        x = lo.rms_norm(w['embed'][toks], w['final.norm'], cfg['eps'], cfg['offset'])
        err, size = np.abs(got[0] - x @ w['head'].T), np.abs(x) @ np.abs(w['head']).T
        assert (err <= (80 + K / 128) * 2.0 ** -24 * size).all(), (M, (err / size).max() * 2 ** 24)
        if sign == 'one':
            assert (err / size).mean() <= (24 + K / 128) * 2.0 ** -24, (M, (err / size).mean() * 2 ** 24)
    eng.close()


@pytest.mark.parametrize('K,N,M', [(96, 200, 3), (520, 260, 20), (520, 260, 40), (520, 1000, 300), (1024, 4100, 2500)])
def test_rows_that_are_not_finite(tm, cuda, K, N, M):
    """an infinity times finite weights other than zero is an infinity of the sum, as in fp32; a NaN is one in its row only; numbers up to 3.3e38 are split without an overflow"""
    g = torch.Generator('cuda').manual_seed(M)
    w = torch.randn(N, K, generator=g, device='cuda').bfloat16()
    w[w == 0] = 1
    x = torch.zeros(M, (K + 31) // 32 * 32, device='cuda')
    x[:, :K] = torch.randn(M, K, generator=g, device='cuda')
    plain = product(tm, w, x)
    x[0, 5], x[M // 2, K - 1], x[M - 1, 3] = float('inf'), float('-inf'), float('nan')
    y = product(tm, w, x)
    assert torch.equal(y[0], torch.sign(w[:, 5].float()) * float('inf')) and torch.equal(y[M // 2], torch.sign(w[:, K - 1].float()) * -float('inf'))
    assert bool(torch.isnan(y[M - 1]).all())
    keep = [m for m in range(M) if m not in (0, M // 2, M - 1)]
    assert torch.equal(y[keep], plain[keep])
    x[:, :K] = torch.rand(M, K, generator=g, device='cuda') * 3.3e38
    w = (w.float().abs() / 2.0 ** 14).bfloat16()
    ref = x[:, :K].double() @ w.double().t()
    assert float((product(tm, w, x).double() / ref - 1).abs().max()) <= (72 + K / 256) * 2.0 ** -24


@pytest.mark.parametrize('K,N,M', [(96, 200, 3), (520, 260, 20), (520, 260, 40), (520, 1000, 300), (1024, 4100, 2500)])
@pytest.mark.parametrize('bits', [0x7F800001, -0x7FFFFF, 0x7F80FFFF, 0x7FC00000])
def test_every_nan_is_one(tm, cuda, K, N, M, bits):
    """also those whose payload the leading bf16 part does not hold"""
    g = torch.Generator('cuda').manual_seed(M)
    w = torch.randn(N, K, generator=g, device='cuda').bfloat16()
    x = torch.zeros(M, (K + 31) // 32 * 32, device='cuda')
    x[:, :K] = torch.randn(M, K, generator=g, device='cuda')
    plain = product(tm, w, x)
    x.view(torch.int32)[M // 3, 7] = bits
    y = product(tm, w, x)
    assert bool(torch.isnan(y[M // 3]).all())
    keep = [m for m in range(M) if m != M // 3]
    assert torch.equal(y[keep], plain[keep])


def test_kernels_of_the_sizes_above():
    """what the sizes of the first test run: the narrow kernel, the weight stream with one and several blocks of rows, both tiles"""
    for K, N, M, plan in ((264, 2052, 3, 1), (1024, 4100, 5, 1), (8448, 260, 40, 1), (2080, 1030, 90, 6), (264, 2052, 257, 6), (1024, 4100, 2500, 5)):
        assert stream_plan(1, K, N, M, 0)[0] == plan, (K, N, M, stream_plan(1, K, N, M, 0))
    assert stream_plan(1, 2048, 1024, 90)[:1] == (2, ) and stream_plan(1, 2048, 32000, 48)[0] == 6 and stream_plan(1, 8448, 2048, 3)[0] == 2
