"""GPU test of the decode attention's rule for how many key splits a row uses (attention_general.hip): rows that one split finishes, rows at the edge of a
second one and rows with as many splits as the launch has, side by side in one launch, for launches of few and of many workgroups; and of what the partial results need of
their workspace."""
import ctypes as C

import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from tests.gpu_helpers import release_all, st
from tests.test_gpu_febivik import Paged, _rounded, attend, row_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('splits', [2, 8])
@pytest.mark.parametrize('window,keep', [(0, 0), (300, 5)])
@pytest.mark.parametrize('seqs,heads,kv_heads,D,V', [(70, 8, 4, 32, 48), (18, 24, 8, 64, 16), (5, 40, 2, 40, 24), (3, 2, 1, 16, 136)])
def test_rows_of_one_and_of_many_splits(tm, cuda, seqs, heads, kv_heads, D, V, window, keep, splits):
    rng = np.random.default_rng(seqs)
    spec = dict(heads=heads, kv_heads=kv_heads, dim=D, vdim=V, scale=0.2, window=window, keep=keep)
    edges = [0, 1023, 256, 255, 63, 64, 511, 128, 512, 1024]
    lens = (edges + rng.integers(1, 300, 70).tolist())[:seqs]
    cache = Paged(0, kv_heads, D, V, [n + 1 for n in lens], rng)
    K = [_rounded(rng.normal(0, 1, (n + 1, kv_heads, D)), 0) for n in lens]
    W = [_rounded(rng.normal(0, 1, (n + 1, kv_heads, V)), 0) for n in lens]

    def call(lo, hi, kernel, prefill, n):
        rs = np.repeat(np.arange(seqs), np.subtract(hi, lo))
        rp = np.concatenate([np.arange(a, b) for a, b in zip(lo, hi)]).astype(int)
        q = _rounded(rng.normal(0, 1, (len(rs), heads * D)), 0)
        kn, vn = (np.stack([c[s][p].reshape(-1) for s, p in zip(rs, rp)]) for c in (K, W))
        cu = np.concatenate([[0], np.cumsum(np.subtract(hi, lo))])
        return q, attend(tm, 0, spec, cache, q, kn, vn, rs, rp, cu, hi, kernel, n, prefill)

    call([0] * seqs, lens, 2, 1, 1)                           # fills the cache
    for kernel in (3, 1):                                     # the matrix-core kernel, the row kernel: both share the rule and the merge
        q, got = call(lens, [n + 1 for n in lens], kernel, 0, splits)
        for s, n in enumerate(lens):
            ref = row_oracle(spec, q[s], K[s][:n + 1], W[s][:n + 1], n)
            # weights and results are rounded to bf16, 2^-9 of each: 3e-2 of the largest value leaves the same room as the kernels' other tests
            assert np.abs(got[s] - ref).max() <= 3e-2 * max(1.0, np.abs(ref).max()), (kernel, s, n)


@pytest.mark.parametrize('splits', [1, 3])
@pytest.mark.parametrize('D,V', [(8, 8), (128, 128), (128, 136), (120, 128), (192, 64), (192, 72), (256, 16), (256, 192), (248, 192), (136, 256), (256, 256)])
def test_sizes_of_either_load_order(tm, cuda, D, V, splits):
    """sizes whose keys and values are asked for at once and sizes whose values follow, with and without channels short of the instantiation's; waves with
    no block, one and two; three heads a key head: rows of the tile without a head"""
    rng = np.random.default_rng(D + V)
    lens = [0, 62, 63, 64, 255, 256, 700]
    spec = dict(heads=6, kv_heads=2, dim=D, vdim=V, scale=D ** -0.5, window=0, keep=0)
    cache = Paged(0, 2, D, V, [n + 1 for n in lens], rng)
    K = [_rounded(rng.normal(0, 1, (n + 1, 2, D)), 0) for n in lens]
    W = [_rounded(rng.normal(0, 1, (n + 1, 2, V)), 0) for n in lens]

    def call(lo, hi, kernel, prefill, n):
        rs = np.repeat(np.arange(len(lens)), np.subtract(hi, lo))
        rp = np.concatenate([np.arange(a, b) for a, b in zip(lo, hi)]).astype(int)
        q = _rounded(rng.normal(0, 1, (len(rs), 6 * D)), 0)
        kn, vn = (np.stack([c[s][p].reshape(-1) for s, p in zip(rs, rp)]) for c in (K, W))
        return q, attend(tm, 0, spec, cache, q, kn, vn, rs, rp, np.concatenate([[0], np.cumsum(np.subtract(hi, lo))]), hi, kernel, n, prefill)

    call([0] * len(lens), lens, 1, 1, 1)                      # fills the cache
    q, got = call(lens, [n + 1 for n in lens], 3, 0, splits)
    for s, n in enumerate(lens):
        ref = row_oracle(spec, q[s], K[s][:n + 1], W[s][:n + 1], n)
        # a weight and a result are rounded to bf16, 2^-9 of each; scores are sums of exact products of bf16 numbers in fp32, off by D 2^-24 of some 10
        assert np.abs(got[s] - ref).max() <= (2 ** -8 + D * 2 ** -19) * max(1.0, np.abs(W[s][:n + 1]).max()), (s, n)


@pytest.mark.parametrize('dtype,D,V', [(0, 128, 128), (0, 64, 136), (0, 256, 192), (1, 128, 128), (1, 64, 132), (1, 256, 192)])
def test_a_workspace_needs_the_alignment_of_its_floats(tm, cuda, D, V, dtype):
    """partial results leave several at a time; the same bits from a workspace that starts between multiples of eight and of sixteen bytes, and nothing around it is written"""
    rng = np.random.default_rng(D + V)
    B, H, G, n, splits = 3, 6, 2, 700, 3
    eb, T = (2, torch.bfloat16) if dtype == 0 else (4, torch.float32)
    blocks = (n + 63) // 64
    size = G * 64 * (D + V)
    pool = torch.from_numpy(rng.normal(0, 1, (B * blocks, size)).astype(np.float32)).cuda().to(T)
    q = torch.from_numpy(rng.normal(0, 1, (B, H * D)).astype(np.float32)).cuda().to(T)
    ptrs = (torch.arange(B * blocks, device='cuda') * (size * eb) + pool.data_ptr()).contiguous()
    ints = [torch.tensor(v, dtype=torch.int32, device='cuda') for v in (list(range(B)), [n - 1] * B, list(range(B + 1)), [n] * B)]
    need = tm.tm_general_attention_workspace(B, H, V, splits) // 4
    out = []
    for shift in range(4):
        ws = torch.full((need + 8, ), -3.0, device='cuda')
        y = torch.empty(B, H * V, device='cuda', dtype=T)
        a = _ffi.GeneralAttn()
        for k, v in dict(q=q.data_ptr(), out=y.data_ptr(), ldq=H * D, ldo=H * V, rows=B, row_seq=ints[0].data_ptr(), row_pos=ints[1].data_ptr(), block_ptrs=ptrs.data_ptr(),
                         block_stride=blocks, v_offset=G * 64 * D * eb, elem_bytes=eb, q_heads=H, kv_heads=G, dim=D, vdim=V, scale=D ** -0.5, splits=splits,
                         workspace=ws.data_ptr() + 4 * shift, kernel=0, nseq=B, max_q_len=1, cu_q=ints[2].data_ptr(), k_len=ints[3].data_ptr()).items():
            setattr(a, k, v)
        _ffi.check(tm.tm_general_attention(C.byref(a), st()))
        out.append(y.float().cpu().numpy())
        assert bool((ws[:shift] == -3.0).all()) and bool((ws[shift + need:] == -3.0).all())
    assert np.isfinite(out[0]).all() and all(np.array_equal(out[0], o) for o in out[1:])
