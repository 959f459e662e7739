"""GPU test of the prefill kernel over staged cache blocks where the sign of the scale decides which of its forms may run: plain scores keep their scale in the exponent, which needs
the largest score to have the largest weight.  Bound as in test_gpu_attention_staged."""
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


@pytest.mark.parametrize('D,V', [(64, 64), (128, 128), (256, 192), (96, 40)])      # (the last: attn_tiles_kernel)
@pytest.mark.parametrize('scale,temp,cap', [(0.2, 0.0, 0.0), (-0.2, 0.0, 0.0), (0.0, 0.0, 0.0), (1e-30, 0.0, 0.0), (0.2, -0.6, 0.0), (-0.2, 0.3, 4.0), (0.2, 0.0, 1e-3), (30.0, 0.0, 0.0)])
def test_scale_of_either_sign(tm, cuda, D, V, scale, temp, cap):
    n, H, chunk = 150, 2, 70      # (a chunk that begins inside a block: rows whose first block holds none of their keys)
    g = torch.Generator('cuda').manual_seed(D)
    pool = torch.randn(3, 64 * (D + V), generator=g, device='cuda').bfloat16()
    q = torch.randn(n, H * D, generator=g, device='cuda').bfloat16()
    out = torch.full((n + 1, H * V), -3.0, device='cuda', dtype=torch.bfloat16)
    ints = [torch.tensor(v, dtype=torch.int32, device='cuda') for v in ([0] * n, list(range(n)), [0, n], [n])]
    ptrs = torch.tensor([pool.data_ptr() + i * 128 * (D + V) for i in range(3)], device='cuda')
    a = _ffi.GeneralAttn()
    for k, v in dict(q=q.data_ptr(), out=out.data_ptr(), ldq=H * D, ldo=H * V, rows=n, row_seq=ints[0].data_ptr(), row_pos=ints[1].data_ptr(), block_ptrs=ptrs.data_ptr(),
                     block_stride=3, v_offset=128 * D, elem_bytes=2, q_heads=H, kv_heads=1, dim=D, vdim=V, scale=scale, softcap=cap, qtemp_coef=temp, qtemp_every=20.0,
                     splits=1, kernel=2, prefill=1, nseq=1, max_q_len=n, cu_q=ints[2].data_ptr(), k_len=ints[3].data_ptr(), chunk=chunk).items():
        setattr(a, k, v)
    _ffi.check(tm.tm_general_attention(C.byref(a), st()))
    K, W = pool[:, :64 * D].reshape(-1, D)[:n].double(), pool[:, 64 * D:].reshape(3, V, 64).transpose(1, 2).reshape(-1, V)[:n].double()
    i = torch.arange(n, device='cuda')
    hide = (i[None, :] > i[:, None]) | (i[None, :] < (i // chunk * chunk)[:, None])
    for h in range(H):
        x = q[:, h * D:(h + 1) * D].double() @ K.t() * scale * (1 + temp * torch.log(torch.floor((i.double() + 1) / 20) + 1))[:, None]
        x = cap * torch.tanh(x / cap) if cap else x
        w = torch.softmax(x.masked_fill(hide, -math.inf), 1)
        ref, size = w @ W, w @ W.abs()
        slack = 1e-3 + 2.0 ** -20 * float(x.abs().max())      # fp32 errors of the largest scores, as errors of a weight
        assert bool(((out[:n, h * V:(h + 1) * V].double() - ref).abs() <= (2.0 ** -8 + slack) * size + 2.0 ** -8 * ref.abs() + 1e-6).all()), h
    assert bool((out[n] == -3.0).all())
