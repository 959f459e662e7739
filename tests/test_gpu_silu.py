"""GPU test of silu(gate) * up as the gated products' epilogues make it (tm_silu_mul runs the same function): every fp16 gate against 64 bits"""
import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from tests.gpu_helpers import release_all, st

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('up', [1.0, -0.7998046875, 3.14453125e-4, 1000.0])
def test_every_gate(tm, cuda, up):
    """one rounding to fp16 of a product that is off by less than 2^-20 of itself: half a unit of fp16 and 2^-9 of one more"""
    g = torch.arange(65536, dtype=torch.int32, device='cuda').to(torch.int16).view(torch.half)
    gu = torch.cat([g.reshape(64, 1024), torch.full((64, 1024), up, dtype=torch.half, device='cuda')], 1).contiguous()
    y = torch.empty(64, 1024, dtype=torch.half, device='cuda')
    _ffi.check(tm.tm_silu_mul(y.data_ptr(), gu.data_ptr(), 64, 1024, st()))
    y, z = y.reshape(-1).double().cpu().numpy(), g.double().cpu().numpy()
    nan = np.isnan(z)
    assert np.isnan(y[nan]).all()
    with np.errstate(over='ignore', invalid='ignore'):
        ref = z / (1 + np.exp(-z)) * float(torch.tensor(up).half())
    fin = np.isfinite(z)
    big = fin & (np.abs(ref) >= 65520)      # rounds to infinity
    assert (y[big & (np.abs(ref) > 65536)] == np.sign(ref[big & (np.abs(ref) > 65536)]) * np.inf).all()
    ok = fin & ~big
    unit = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ref[ok]), 2.0 ** -14))) - 10)
    assert (np.abs(y[ok] - ref[ok]) <= (0.5 + 2.0 ** -9) * unit).all()
    assert y[np.isposinf(z)] == np.sign(up) * np.inf and not np.isfinite(y[np.isneginf(z)])
