"""GPU tests of the grouped fp8 products at the borders of their row tiles: experts without rows, with one row, with exactly one tile and one row more, all
rows at one expert; token counts on both sides of the lines between 32, 64 and 128 rows a tile, column counts off the eight-tile grid -- against the oracle."""
import math

import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from oracle import tm_oracle as o
from tests.gpu_helpers import dev, host, release_all, st
from tests.test_gpu_moe_fp8_wide_tiles import near

pytestmark = pytest.mark.gpu
f16 = np.float16


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('T,skew', [(1, 0), (32, 0), (33, 0), (63, 3), (64, 0), (100, 0), (130, 3), (190, 0), (230, 3), (257, 0), (513, 3)])
def test_row_tiles(tm, cuda, T, skew):
    rng = np.random.default_rng(T)
    H, I, E, k = 256, 640, 6, 2
    x = rng.standard_normal((T, H)).astype(f16)
    gate = (rng.standard_normal((H, E)) * 0.2).astype(f16)
    if skew:                                                  # two experts take nearly all rows, the others few or none
        x[:, 0], gate[0] = 1.0, np.asarray([skew, skew, -1, -3, -3, -3], f16)
    h, experts = _ffi.C.c_void_p(), []
    _ffi.check(tm.tm_moe_create(_ffi.C.byref(h), H, I, E, k, 2, 1, 1.0))
    _ffi.check(tm.tm_moe_set_gate(h, dev(gate).data_ptr(), st()))
    for e in range(E):
        w1, w3 = ((rng.standard_normal((H, I)) / math.sqrt(H)).astype(f16) for _ in range(2))
        w2 = (2 * rng.standard_normal((I, H)) / math.sqrt(I)).astype(f16)
        (q1, s1), (q3, s3), (q2, s2) = (o.fp8_quantize_blockwise(w) for w in (w1, w3, w2))
        q13, s13 = o.interleave_w1w3(q1, q3), np.concatenate([s1, s3], axis=1)
        experts.append(((q13, s13), (q2, s2)))
        _ffi.check(tm.tm_moe_set_expert(h, e, dev(q13).data_ptr(), dev(s13).data_ptr(), None, dev(q2).data_ptr(), dev(s2).data_ptr(), None, st()))
    torch.cuda.synchronize()
    ws = torch.zeros(tm.tm_moe_workspace(h, T), dtype=torch.uint8, device='cuda')
    out = torch.zeros((T, H), dtype=torch.float16, device='cuda')
    ids = torch.zeros((T, k), dtype=torch.int32, device='cuda')
    wts = torch.zeros((T, k), dtype=torch.float32, device='cuda')
    _ffi.check(tm.tm_moe_forward(h, out.data_ptr(), dev(x).data_ptr(), T, ws.data_ptr(), ids.data_ptr(), wts.data_ptr(), st()))
    ref, ref_ids, ref_w = o.moe_ffn_fp8(x, gate, experts, k)
    assert np.array_equal(host(ids), ref_ids)
    assert np.abs(host(wts) - ref_w).max() <= 1e-5
    # (as near says; results of order one, so that nothing, a row's neighbour and a 32-column group's neighbour lie outside)
    ref = ref.astype(np.float32)
    assert np.abs(ref).max() > 1 and not near(0 * ref, ref) and not near(np.roll(ref, 32, axis=1), ref) and (T == 1 or not near(np.roll(ref, 1, axis=0), ref))
    assert near(host(out).astype(np.float32), ref)
    _ffi.check(tm.tm_moe_destroy(h))


def test_tiles_of_the_measured_dispatch(tm, cuda, tmp_path):
    """a table line decides the tile: 32, 64, 128 and 256 rows give the same result, whatever the rule would take for these 100 tokens"""
    rng = np.random.default_rng(5)
    T, H, I, E, k = 100, 256, 384, 4, 2
    x = rng.standard_normal((T, H)).astype(f16)
    h, experts, gate = _ffi.C.c_void_p(), [], (rng.standard_normal((H, E)) * 0.2).astype(f16)
    _ffi.check(tm.tm_moe_create(_ffi.C.byref(h), H, I, E, k, 2, 1, 1.0))
    _ffi.check(tm.tm_moe_set_gate(h, dev(gate).data_ptr(), st()))
    for e in range(E):
        w1, w3 = ((rng.standard_normal((H, I)) / math.sqrt(H)).astype(f16) for _ in range(2))
        (q1, s1), (q3, s3), (q2, s2) = (o.fp8_quantize_blockwise(w) for w in (w1, w3, (2 * rng.standard_normal((I, H)) / math.sqrt(I)).astype(f16)))
        q13, s13 = o.interleave_w1w3(q1, q3), np.concatenate([s1, s3], axis=1)
        experts.append(((q13, s13), (q2, s2)))
        _ffi.check(tm.tm_moe_set_expert(h, e, dev(q13).data_ptr(), dev(s13).data_ptr(), None, dev(q2).data_ptr(), dev(s2).data_ptr(), None, st()))
    ref = o.moe_ffn_fp8(x, gate, experts, k)[0].astype(np.float32)
    ws, table = torch.zeros(tm.tm_moe_workspace(h, T), dtype=torch.uint8, device='cuda'), tmp_path / 't.txt'
    for rows in (32, 64, 128, 256):
        table.write_text(f'G 34 0 {H} {2 * I} {T} {rows} 0 0 0\nG 34 0 {I} {H} {T} {rows} 0 0 0\n')
        _ffi.check(tm.tm_gemm_import(str(table).encode()))
        out = torch.zeros((T, H), dtype=torch.float16, device='cuda')
        _ffi.check(tm.tm_moe_forward(h, out.data_ptr(), dev(x).data_ptr(), T, ws.data_ptr(), None, None, st()))
        assert near(host(out).astype(np.float32), ref), rows
    _ffi.check(tm.tm_moe_destroy(h))
