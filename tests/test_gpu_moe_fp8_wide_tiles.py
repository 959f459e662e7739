"""GPU tests of the 256 x 256 tile of the grouped fp8 products at the borders of its rows, columns and k-blocks: experts without rows, with one, with exactly
one tile and one row more, a last column tile that is not full, one k-block and several -- against the oracle; and of the line from which on the rule takes it.
Table lines name the tile (these products are too small for the rule); the results are of order one."""
import math

import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from oracle import tm_oracle as o
from tests.gpu_helpers import dev, host, release_all, st

pytestmark = pytest.mark.gpu
f16 = np.float16


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


def _bucket(T):
    return T if T <= 256 else max(512, 1 << (T - 1).bit_length())


def _tile(tm, tmp_path, H, I, T, rows):
    f = tmp_path / 't.txt'
    f.write_text(f'G 34 0 {H} {2 * I} {_bucket(T)} {rows} 0 0 0\nG 34 0 {I} {H} {_bucket(T)} {rows} 0 0 0\n')
    _ffi.check(tm.tm_gemm_import(str(f).encode()))


def _blocks(rng, K, N):
    """weights whose 128 x 128 blocks differ in size, so that a block's scale in another's place shows"""
    f = 2.0 ** ((np.arange(-(-K // 128))[:, None] + 2 * np.arange(-(-N // 128))) % 3 - 1)
    return rng.standard_normal((K, N)) / math.sqrt(K) * f.repeat(128, 0).repeat(128, 1)[:K, :N]


def near(got, ref):
    """An fp32 sum in another order turns an fp16 unit of a gated row now and then and with it an e4m3 code: an eighth of one of the channels of that row.  The
    outputs have the size of a sum of 128 or more such channels, and few rows have a turned code at all."""
    err, most = np.abs(got - ref), np.abs(ref).max()
    rows = (err <= 2.0**-8 * most).all(axis=1)
    return err.max() <= 2.0**-4 * most and rows.mean() >= 0.7


@pytest.mark.parametrize('H,I,counts', [(384, 128, (256, 257, 0, 399)), (128, 384, (1, 512, 511, 0)), (640, 256, (1000, 3, 9, 12)), (256, 128, (0, 0, 0, 900))])
def test_rows_and_columns(tm, cuda, tmp_path, H, I, counts):
    rng = np.random.default_rng(H + I)
    E, T = len(counts), sum(counts)
    x = (rng.standard_normal((T, H)) * 2.0 ** (np.arange(H) // 128 % 3 - 1)).astype(f16)
    x[:, :E] = 0
    x[np.arange(T), rng.permutation(np.repeat(np.arange(E), counts))] = 4.0   # the router takes an expert's rows from the first channels
    gate = np.zeros((H, E), f16)
    gate[np.arange(E), np.arange(E)] = 2.0
    h, experts = _ffi.C.c_void_p(), []
    _ffi.check(tm.tm_moe_create(_ffi.C.byref(h), H, I, E, 1, 2, 1, 1.0))
    _ffi.check(tm.tm_moe_set_gate(h, dev(gate).data_ptr(), st()))
    for e in range(E):
        (q1, s1), (q3, s3), (q2, s2) = (o.fp8_quantize_blockwise(_blocks(rng, *shape).astype(f16)) for shape in ((H, I), (H, I), (I, H)))
        q13, s13 = o.interleave_w1w3(q1, q3), np.concatenate([s1, s3], axis=1)
        experts.append(((q13, s13), (q2, s2)))
        _ffi.check(tm.tm_moe_set_expert(h, e, dev(q13).data_ptr(), dev(s13).data_ptr(), None, dev(q2).data_ptr(), dev(s2).data_ptr(), None, st()))
    ws = torch.zeros(tm.tm_moe_workspace(h, T), dtype=torch.uint8, device='cuda')
    ref, ref_ids, _ = o.moe_ffn_fp8(x, gate, experts, 1)
    ref = ref.astype(np.float32)
    assert tuple(np.bincount(ref_ids.ravel(), minlength=E)) == counts
    # what the bound has to tell apart: nothing, a row's neighbour, one k-block of the second product without its scale
    assert np.abs(ref).max() > 1 and not near(0 * ref, ref) and not near(np.roll(ref, 1, axis=0), ref) and not near(np.roll(ref, 32, axis=1), ref)
    for rows in (256, 128):
        _tile(tm, tmp_path, H, I, T, rows)
        out = torch.full((T + 2, H), 7.0, dtype=torch.float16, device='cuda')
        ids = torch.zeros((T, 1), dtype=torch.int32, device='cuda')
        _ffi.check(tm.tm_moe_forward(h, out[1:].data_ptr(), dev(x).data_ptr(), T, ws.data_ptr(), ids.data_ptr(), None, st()))
        assert np.array_equal(host(ids), ref_ids)
        got = host(out).astype(np.float32)
        assert (got[0] == 7).all() and (got[-1] == 7).all()
        assert near(got[1:-1], ref), rows
    _ffi.check(tm.tm_moe_destroy(h))


@pytest.mark.parametrize('E,I,T,rows', [(4, 2432, 700, 256), (4, 2304, 700, 128), (4, 2432, 460, 128), (16, 1280, 1680, 256), (16, 1408, 1600, 128)])
def test_line(tm, cuda, tmp_path, E, I, T, rows):
    """more than about one round of 128-row tiles: 256 rows; fewer, or fewer than 105 rows an expert: 128.  The two add the 128 channels of a block in another
    order, so their bits tell which one ran (the second product has few columns and always the smaller tile)."""
    H, k = 1024, 1
    g = torch.Generator('cuda').manual_seed(E + I)
    h = _ffi.C.c_void_p()
    _ffi.check(tm.tm_moe_create(_ffi.C.byref(h), H, I, E, k, 2, 1, 1.0))
    gate = (torch.randn(H, E, generator=g, device='cuda') / math.sqrt(H)).half()
    _ffi.check(tm.tm_moe_set_gate(h, gate.data_ptr(), st()))
    for e in range(E):
        a, b = ((16 * torch.randn(*s, generator=g, device='cuda')).to(torch.float8_e4m3fn) for s in ((H, 2 * I), (I, H)))
        sa = torch.full((H // 128, 2 * I // 128), 1 / 16 / math.sqrt(H), device='cuda')
        sb = torch.full((I // 128, H // 128), 1 / 16 / math.sqrt(I), device='cuda')
        _ffi.check(tm.tm_moe_set_expert(h, e, a.data_ptr(), sa.data_ptr(), None, b.data_ptr(), sb.data_ptr(), None, st()))
        torch.cuda.synchronize()
    x = torch.randn(T, H, generator=g, device='cuda').half()
    ws = torch.zeros(tm.tm_moe_workspace(h, T), dtype=torch.uint8, device='cuda')
    outs = []
    for r in (0, 128, 256):
        if r:
            f = tmp_path / 't.txt'
            f.write_text(f'G 34 0 {H} {2 * I} {_bucket(T)} {r} 0 0 0\n')
            _ffi.check(tm.tm_gemm_import(str(f).encode()))
        outs.append(torch.empty(T, H, dtype=torch.float16, device='cuda'))
        _ffi.check(tm.tm_moe_forward(h, outs[-1].data_ptr(), x.data_ptr(), T, ws.data_ptr(), None, None, st()))
    torch.cuda.synchronize()
    assert not torch.equal(outs[1], outs[2])
    assert torch.equal(outs[0], outs[1] if rows == 128 else outs[2])
    tm.tm_moe_destroy(h)
