"""GPU test of the routing tables of many tokens (a workgroup an expert): token counts on and around one, two and three tokens a thread, one expert, and 64 with eight
choices -- a block over all tokens against the same block over portions of 64, whose tables are the masks'."""
import ctypes as C
import math

import pytest
import torch

from lmdeploy_amd import _ffi
from tests.gpu_helpers import release_all, st

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('experts,top', [(1, 1), (5, 2), (64, 8)])
def test_tables(tm, cuda, experts, top):
    H, I = 128, 128
    g = torch.Generator('cuda').manual_seed(experts)
    h = C.c_void_p()
    _ffi.check(tm.tm_moe_create(C.byref(h), H, I, experts, top, 2, 1, 1.0))
    gate = (torch.randn(H, experts, generator=g, device='cuda') / math.sqrt(H)).half()
    _ffi.check(tm.tm_moe_set_gate(h, gate.data_ptr(), st()))
    for e in range(experts):
        a = (16 * torch.randn(H, 2 * I, generator=g, device='cuda')).to(torch.float8_e4m3fn)
        b = (16 * torch.randn(I, H, generator=g, device='cuda')).to(torch.float8_e4m3fn)
        sa = torch.full((H // 128, 2 * I // 128), 1 / 16 / math.sqrt(H), device='cuda')
        sb = torch.full((I // 128, H // 128), 1 / 16 / math.sqrt(I), device='cuda')
        _ffi.check(tm.tm_moe_set_expert(h, e, a.data_ptr(), sa.data_ptr(), None, b.data_ptr(), sb.data_ptr(), None, st()))
        torch.cuda.synchronize()

    def run(x):
        T = x.shape[0]
        ws = torch.zeros(tm.tm_moe_workspace(h, T), dtype=torch.uint8, device='cuda')
        out = torch.empty(T, H, dtype=torch.float16, device='cuda')
        ids = torch.empty(T, top, dtype=torch.int32, device='cuda')
        _ffi.check(tm.tm_moe_forward(h, out.data_ptr(), x.data_ptr(), T, ws.data_ptr(), ids.data_ptr(), None, st()))
        torch.cuda.synchronize()
        return out.float(), ids

    for T in (65, 1023, 1024, 1025, 2049):
        x = torch.randn(T, H, generator=g, device='cuda').half()
        got, ids = run(x)
        parts = [run(x[i:i + 64].contiguous()) for i in range(0, T, 64)]
        ref = torch.cat([p[0] for p in parts])
        assert torch.equal(ids, torch.cat([p[1] for p in parts]))
        # fp32 sums in another order may turn an e4m3 code of an activation by one step, an eighth of it at most: 1/8 of one of 128 terms
        assert (got - ref).abs().max() <= 0.02 * ref.abs().max(), T
    tm.tm_moe_destroy(h)
