"""GPU tests of the 256 x 256 tile of the grouped fp8 products at the borders of its rows, columns and k-blocks: experts without rows, with one, with exactly
one tile and one row more, a last column tile that is not full, one k-block and several -- against the oracle."""
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


@pytest.mark.parametrize('H,I,counts', [(384, 128, (256, 257, 0, 399)), (128, 384, (1, 512, 511, 0)), (640, 256, (1000, 3, 9, 12)), (256, 128, (0, 0, 0, 900))])
def test_rows_and_columns(tm, cuda, H, I, counts):
    rng = np.random.default_rng(H + I)
    E, T = len(counts), sum(counts)
    x = rng.standard_normal((T, H)).astype(f16)
    x[:, :E] = 0
    x[np.arange(T), rng.permutation(np.repeat(np.arange(E), counts))] = 4.0   # the router takes an expert's rows from the first channels
    gate = np.zeros((H, E), f16)
    gate[np.arange(E), np.arange(E)] = 2.0
    h, experts = _ffi.C.c_void_p(), []
    _ffi.check(tm.tm_moe_create(_ffi.C.byref(h), H, I, E, 1, 2, 1, 1.0))
    _ffi.check(tm.tm_moe_set_gate(h, dev(gate).data_ptr(), st()))
    for e in range(E):
        w1, w3 = ((rng.standard_normal((H, I)) * (0.1 / math.sqrt(H))).astype(f16) for _ in range(2))
        (q1, s1), (q3, s3), (q2, s2) = (o.fp8_quantize_blockwise(w) for w in (w1, w3, (rng.standard_normal((I, H)) * (0.1 / math.sqrt(I))).astype(f16)))
        q13, s13 = o.interleave_w1w3(q1, q3), np.concatenate([s1, s3], axis=1)
        experts.append(((q13, s13), (q2, s2)))
        _ffi.check(tm.tm_moe_set_expert(h, e, dev(q13).data_ptr(), dev(s13).data_ptr(), None, dev(q2).data_ptr(), dev(s2).data_ptr(), None, st()))
    ws = torch.zeros(tm.tm_moe_workspace(h, T), dtype=torch.uint8, device='cuda')
    out = torch.full((T + 2, H), 7.0, dtype=torch.float16, device='cuda')
    ids = torch.zeros((T, 1), dtype=torch.int32, device='cuda')
    _ffi.check(tm.tm_moe_forward(h, out[1:].data_ptr(), dev(x).data_ptr(), T, ws.data_ptr(), ids.data_ptr(), None, st()))
    ref, ref_ids, _ = o.moe_ffn_fp8(x, gate, experts, 1)
    assert np.array_equal(host(ids), ref_ids) and tuple(np.bincount(ref_ids.ravel(), minlength=E)) == counts
    got = host(out).astype(np.float32)
    assert (got[0] == 7).all() and (got[-1] == 7).all()
    # as in the tests of the smaller tiles: an fp32 sum in another order can turn an e4m3 code of a gated row
    err, ref = np.abs(got[1:-1] - ref.astype(np.float32)), np.abs(ref.astype(np.float32))
    assert (err <= 4e-3 + 2.0**-6 * ref).all(), err.max()
    _ffi.check(tm.tm_moe_destroy(h))
