"""GPU tests of the prefill kernel that brings cache blocks into LDS (attention_general.hip): every size it serves, portions that start and end around
its row tiles and cache blocks, and every modifier that a score, a row's range or an output can have, against 64 bits.

Bound: soft-max weights are rounded to bf16 (2^-9 of each), the result once more; scores carry fp32 errors (1e-5 of a weight, 64 scores an exponent)."""
import ctypes as C
import math

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


SIZES = [(64, 64), (64, 128), (128, 128), (256, 128), (256, 192), (256, 256)]
# (rows of the launch, context including them) of each sequence: one row, the edges of 32- and 128-row tiles, portions inside a block
PORTIONS = [[(1, 1), (33, 33), (130, 130)], [(31, 95), (64, 64), (257, 300), (2, 700)], [(128, 128), (5, 64), (1, 65)]]


def run(tm, D, V, portions, H=4, G=2, cap=0.0, sink=False, window=0, keep=0, chunk=0, bias=False, table=0, gate=False, out_f32=False, space=0,
        k_heads=0, v_heads=0, temp=0.0, seed=0):
    g = torch.Generator('cuda').manual_seed(seed)
    kh, vh = k_heads or G, v_heads or G
    n = len(portions)
    blocks = [(k + 63) // 64 for _, k in portions]
    elems = kh * 64 * D + vh * V * 64
    pool = (torch.randn(sum(blocks), elems, generator=g, device='cuda')).bfloat16()
    order, ptrs, at = np.random.default_rng(seed).permutation(sum(blocks)), np.zeros((n, max(blocks)), np.int64), 0
    for s, b in enumerate(blocks):
        for i in range(b):
            ptrs[s, i] = pool.data_ptr() + int(order[at + i]) * elems * 2
        at += b
    lens = [q for q, _ in portions]
    rows, ldq, hs = sum(lens), H * D + 8, V + space
    q = torch.randn(rows, ldq, generator=g, device='cuda').bfloat16()
    ldo = H * hs + 3
    out = torch.full((rows + 1, ldo), -3.0, device='cuda', dtype=torch.float32 if out_f32 else torch.bfloat16)
    t = {k: torch.from_numpy(np.asarray(v)).cuda() for k, v in dict(
        ptrs=ptrs, seq=np.repeat(np.arange(n), lens).astype(np.int32), cu=np.cumsum([0] + lens).astype(np.int32),
        pos=np.concatenate([np.arange(k - m, k) for m, k in portions]).astype(np.int32), klen=np.asarray([k for _, k in portions], np.int32)).items()}
    sk, r1, r2 = (torch.randn(H, generator=g, device='cuda').abs() + 0.1 for _ in range(3))
    tab, gt = torch.randn(H, max(1, table), generator=g, device='cuda'), torch.randn(rows, H + 2, generator=g, device='cuda')
    a = _ffi.GeneralAttn()
    for k, v in dict(q=q.data_ptr(), out=out.data_ptr(), ldq=ldq, ldo=ldo, rows=rows, row_seq=t['seq'].data_ptr(), row_pos=t['pos'].data_ptr(),
                     block_ptrs=t['ptrs'].data_ptr(), block_stride=max(blocks), v_offset=kh * 64 * D * 2, elem_bytes=2, q_heads=H, kv_heads=G, dim=D,
                     vdim=V, scale=1.5 / math.sqrt(D), softcap=cap, qtemp_coef=temp, qtemp_every=40.0, splits=1, kernel=2, prefill=1, nseq=n,
                     max_q_len=max(lens), cu_q=t['cu'].data_ptr(), k_len=t['klen'].data_ptr(), window=window, keep_first=keep, chunk=chunk,
                     k_heads=k_heads, v_heads=v_heads, out_f32=int(out_f32), out_head_stride=hs if space else 0).items():
        setattr(a, k, v)
    if sink:
        a.sink = sk.data_ptr()
    if bias:
        a.dist_r1, a.dist_r2 = r1.data_ptr(), r2.data_ptr()
    if table:
        a.dist_table, a.dist_table_len = tab.data_ptr(), table
    if gate:
        a.out_gate, a.ld_gate = gt.data_ptr(), H + 2
    _ffi.check(tm.tm_general_attention(C.byref(a), st()))
    torch.cuda.synchronize()
    row, at = 0, 0
    for s, (m, k) in enumerate(portions):
        blk = pool[torch.from_numpy(order[at:at + blocks[s]].copy()).cuda()].double()
        at += blocks[s]
        p, j = torch.arange(k - m, k, device='cuda'), torch.arange(k, device='cuda')
        d = p[:, None] - j[None, :]
        hide = d < 0
        if window:
            hide |= (d >= window) & (j[None, :] >= keep)
        if chunk:
            hide |= j[None, :] < (p // chunk * chunk)[:, None]
        for h in range(H):
            grp = h // (H // G)
            K = blk[:, :kh * 64 * D].reshape(-1, kh, 64, D)[:, grp % kh].reshape(-1, D)[:k]
            Vv = blk[:, kh * 64 * D:].reshape(-1, vh, V, 64)[:, grp % vh].transpose(1, 2).reshape(-1, V)[:k]
            x = q[row:row + m, h * D:(h + 1) * D].double() @ K.t() * (1.5 / math.sqrt(D))
            if temp:
                x = x * (1 + temp * torch.log(torch.floor((p.double() + 1) / 40) + 1))[:, None]
            x = cap * torch.tanh(x / cap) if cap else x
            if bias:
                x = x - r1[h].double() * torch.log(1 + r2[h].double() * d.clamp(min=0))
            if table:
                x = x + tab[h].double()[d.clamp(0, table - 1)]
            x = x.masked_fill(hide, -math.inf)
            if sink:
                x = torch.cat([x, sk[h].double().expand(m, 1)], 1)
            w = torch.softmax(x, 1)[:, :k]
            w = w * torch.sigmoid(gt[row:row + m, h].double())[:, None] if gate else w
            ref, size = w @ Vv, w @ Vv.abs()
            got = out[row:row + m, h * hs:h * hs + V].double()
            assert bool(((got - ref).abs() <= (2.0 ** -8 + 1e-3) * size + (0 if out_f32 else 2.0 ** -8) * ref.abs() + 1e-6).all()), (s, h)
        row += m
    assert bool((out[rows] == -3.0).all()) and bool((out[:rows, H * hs:] == -3.0).all())


@pytest.mark.parametrize('D,V', SIZES)
@pytest.mark.parametrize('portions', range(len(PORTIONS)))
def test_sizes_and_portions(tm, cuda, D, V, portions):
    run(tm, D, V, PORTIONS[portions], seed=portions)


@pytest.mark.parametrize('D,V', [(64, 128), (128, 128), (256, 192)])
@pytest.mark.parametrize('kw', [
    dict(cap=9.0, sink=True, temp=0.35), dict(window=70, keep=3), dict(window=1, keep=0), dict(window=64, keep=130, sink=True), dict(chunk=48),
    dict(chunk=256, bias=True, gate=True), dict(table=50, out_f32=True, space=8), dict(H=8, G=4, k_heads=4, v_heads=2), dict(H=5, G=5, cap=30.0),
    dict(H=16, G=1, k_heads=1, v_heads=1), dict(H=6, G=2, k_heads=1, v_heads=2, table=9, cap=20.0, window=100, keep=2),
], ids=str)
def test_modifiers(tm, cuda, D, V, kw):
    run(tm, D, V, PORTIONS[1], seed=3, **kw)


def test_long_context_keeps_every_far_key(tm, cuda):
    run(tm, 128, 128, [(700, 3000), (1, 2049)], H=2, G=1, seed=5)
