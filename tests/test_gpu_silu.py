"""GPU tests of silu(gate) * up as the gated products' epilogues make it (tm_silu_mul runs the same function): every fp16 gate against 64 bits, and in fp32 and bf16 gates
that are far below zero, whose silu is zero whatever it is multiplied by"""
import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from tests import bedenex_oracle as bo
from tests.gpu_helpers import release_all, st
from tests.test_gpu_bedenex import TOL, engine, rel_err

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


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('rows', [2, 90])                   # products of few rows and tiles
def test_gates_far_below_zero(cuda, tmp_path, dtype, rows):
    """a gate of -64 ... -2^126 times an `up` of some 2^60 stays below 2^-20 of the stream; the model's other gates are ordinary"""
    cfg = bo.make_config(64, 97, [bo.attention_layer(4, 1, 16, 32, 0.5, 33, bo.moe(1, 1, 96))])
    w = bo.make_weights(cfg, 3)
    w['embed'][:, 0], w['l0.norm1'][0], w['l0.mlp.router'][0] = 1.0, 1.0, 0.0     # every row's first channel is positive, its score 1/2
    w['l0.mlp.e0.gate'][32:], w['l0.mlp.e0.up'][32:] = 0.0, w['l0.mlp.e0.up'][32:] * 2.0 ** 60
    w['l0.mlp.e0.gate'][32:, 0] = -2.0 ** np.linspace(8, 127, 64).round()
    folder = str(tmp_path / 'm')
    bo.write_checkpoint(folder, cfg, w)
    toks = np.random.default_rng(rows).integers(0, 97, rows)
    with np.errstate(over='ignore'):
        ref = bo.forward(cfg, w, toks)
    eng = engine(folder, dtype)
    s = eng.open_session()
    got = eng.step_tokens([(s, toks, list(range(rows)))])
    eng.close_session(s)
    eng.close()
    assert rel_err(got, ref) <= TOL[dtype]
