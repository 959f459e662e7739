"""GPU test of the choice of experts: equal scores (the lower index first), experts on one and on several registers of a lane, infinite scores, and numbers that are
none, which only have to leave each token distinct experts."""
import ctypes as C

import pytest
import torch

from lmdeploy_amd import _ffi
from tests.gpu_helpers import release_all, st

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('experts,top', [(1, 1), (5, 3), (8, 8), (64, 7)])
def test_router(tm, cuda, experts, top):
    H, I, T = 128, 128, 9
    h = C.c_void_p()
    _ffi.check(tm.tm_moe_create(C.byref(h), H, I, experts, top, 2, 1, 1.0))
    # a token's only channel picks its row of scores: all equal, two levels, falling, rising, with infinities of both signs, with a NaN
    rows = torch.zeros(T, experts)
    e = torch.arange(experts)
    rows[1], rows[2], rows[3] = (e % 2).float(), -e.float(), e.float()
    rows[4, ::2], rows[5, 1::3] = float('-inf'), float('inf')
    rows[6] = float('-inf')
    rows[7, experts // 2] = float('nan')
    rows[8] = -0.0
    gate = torch.zeros(H, experts)
    gate[:T] = rows
    gate = gate.half().cuda()
    x = torch.zeros(T, H, dtype=torch.float16, device='cuda')
    for t in range(T):
        x[t, t] = 1
    finite = [0, 1, 2, 3, 8]                     # (0 * inf: with the others' rows every token's scores are NaN or infinite)
    plain = gate.clone()
    plain[[4, 5, 6, 7]] = 0
    gates = [(plain, finite), (gate, range(T))]
    for ex in range(experts):
        w = torch.ones(H, 2 * I, device='cuda').to(torch.float8_e4m3fn)
        s1, s2 = torch.full((1, 2), 1 / 128, device='cuda'), torch.full((1, 1), 1 / 128, device='cuda')
        v = torch.ones(I, H, device='cuda').to(torch.float8_e4m3fn)
        _ffi.check(tm.tm_moe_set_expert(h, ex, w.data_ptr(), s1.data_ptr(), None, v.data_ptr(), s2.data_ptr(), None, st()))
        torch.cuda.synchronize()
    for gt, tokens in gates:
        _ffi.check(tm.tm_moe_set_gate(h, gt.data_ptr(), st()))
        ws = torch.zeros(tm.tm_moe_workspace(h, T), dtype=torch.uint8, device='cuda')
        out = torch.empty(T, H, dtype=torch.float16, device='cuda')
        ids = torch.empty(T, top, dtype=torch.int32, device='cuda')
        _ffi.check(tm.tm_moe_forward(h, out.data_ptr(), x.data_ptr(), T, ws.data_ptr(), ids.data_ptr(), None, st()))
        torch.cuda.synchronize()
        got = ids.cpu().tolist()
        for t in tokens:
            if gt is gate:
                assert len(set(got[t])) == top and 0 <= min(got[t]) and max(got[t]) < experts, (t, got[t])
            else:
                assert got[t] == sorted(range(experts), key=lambda i: (-rows[t, i].item(), i))[:top], (t, got[t])
    tm.tm_moe_destroy(h)
