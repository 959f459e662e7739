"""GPU tests of the fp32 attention kernel whose workgroups hold the query heads of a key head as a tile (attention_general.hip): sizes on both sides of its channel
steps, groups of heads around its tile of sixteen, rows around its blocks, waves and key splits, every modifier, against 64 bits and the row kernel.

Bound: a score is a sum of `dim` fp32 products and, with a cap, a tanhf (2^-24 of every product a step, 8 more for the modifiers), its error moves a weight by as
much of itself, twice with the denominator; the output is a sum over the keys with one rounding each."""
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


# (rows, context including them) of each sequence: one row, block and 16-key edges, portions inside a block, decoded rows
PORTIONS = [[(1, 1), (3, 17), (66, 130)], [(1, 16), (1, 64), (1, 65), (1, 700), (1, 129)]]


def run(tm, D, V, portions, H, G, kernel=0, splits=1, cap=0.0, sink=False, window=0, keep=0, chunk=0, bias=False, table=0, gate=False, space=0, k_heads=0, v_heads=0,
        temp=0.0, unseen=False):
    g = torch.Generator('cuda').manual_seed(D + H)
    kh, vh = k_heads or G, v_heads or G
    n = len(portions)
    blocks = [(k + 63) // 64 for _, k in portions]
    elems = kh * 64 * D + vh * V * 64
    pool = torch.randn(sum(blocks), elems, generator=g, device='cuda')
    order, ptrs, at = np.random.default_rng(D).permutation(sum(blocks)), np.zeros((n, max(blocks)), np.int64), 0
    for s, b in enumerate(blocks):
        for i in range(b):
            ptrs[s, i] = pool.data_ptr() + int(order[at + i]) * elems * 4
        last = pool[int(order[at + b - 1])]
        behind = (portions[s][1] - 1) % 64 + 1      # entries behind a sequence's own hold what they may
        last[:kh * 64 * D].view(kh, 64, D)[:, behind:] = float('nan')
        last[kh * 64 * D:].view(vh, V, 64)[:, :, behind:] = float('nan')
        if unseen:                                  # and so do those that no row of the portion sees any more
            lo = portions[s][1] - portions[s][0]
            lo = lo // chunk * chunk if chunk else max(0, lo - window + 1)
            for i in range(keep, lo):
                e = pool[int(order[at + i // 64])]
                e[:kh * 64 * D].view(kh, 64, D)[:, i % 64] = float('nan')
                e[kh * 64 * D:].view(vh, V, 64)[:, :, i % 64] = float('inf')
        at += b
    lens = [q for q, _ in portions]
    rows, ldq, hs = sum(lens), H * D + 3, V + space
    q = torch.randn(rows, ldq, generator=g, device='cuda')
    ldo = H * hs + 3
    out = torch.full((rows + 1, ldo), -3.0, device='cuda')
    t = {k: torch.from_numpy(np.asarray(v)).cuda() for k, v in dict(
        ptrs=ptrs, seq=np.repeat(np.arange(n), lens).astype(np.int32), cu=np.cumsum([0] + lens).astype(np.int32),
        pos=np.concatenate([np.arange(k - m, k) for m, k in portions]).astype(np.int32), klen=np.asarray([k for _, k in portions], np.int32)).items()}
    sk, r1, r2 = (torch.randn(H, generator=g, device='cuda').abs() + 0.1 for _ in range(3))
    tab, gt = torch.randn(H, max(1, table), generator=g, device='cuda'), torch.randn(rows, H + 2, generator=g, device='cuda')
    ws = torch.zeros(max(1, tm.tm_general_attention_workspace(rows, H, V, splits) // 4), device='cuda')
    a, scale = _ffi.GeneralAttn(), 1.5 / math.sqrt(D)
    for k, v in dict(q=q.data_ptr(), out=out.data_ptr(), ldq=ldq, ldo=ldo, rows=rows, row_seq=t['seq'].data_ptr(), row_pos=t['pos'].data_ptr(),
                     block_ptrs=t['ptrs'].data_ptr(), block_stride=max(blocks), v_offset=kh * 64 * D * 4, elem_bytes=4, q_heads=H, kv_heads=G, dim=D,
                     vdim=V, scale=scale, softcap=cap, qtemp_coef=temp, qtemp_every=40.0, splits=splits, workspace=ws.data_ptr(), kernel=kernel,
                     prefill=int(splits == 1), nseq=n, max_q_len=max(lens), cu_q=t['cu'].data_ptr(), k_len=t['klen'].data_ptr(), window=window, keep_first=keep,
                     chunk=chunk, k_heads=k_heads, v_heads=v_heads, out_head_stride=hs if space else 0).items():
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
    ref, bound = torch.full((rows + 1, ldo), -3.0, device='cuda', dtype=torch.float64), torch.zeros((rows + 1, ldo), device='cuda', dtype=torch.float64)
    row, at = 0, 0
    for s, (m, k) in enumerate(portions):
        blk = pool[torch.from_numpy(order[at:at + blocks[s]].copy()).cuda()].double()
        at += blocks[s]
        if unseen:
            blk = blk.nan_to_num(0.0, 0.0, 0.0)
        p, j = torch.arange(k - m, k, device='cuda'), torch.arange(k, device='cuda')
        d = p[:, None] - j[None, :]
        hide = d < 0
        if window:
            hide |= (d >= window) & (j[None, :] >= keep)
        if chunk:
            hide |= j[None, :] < (p // chunk * chunk)[:, None]
        for h in range(H):
            gr = h // (H // G)
            K = blk[:, :kh * 64 * D].view(-1, kh, 64, D)[:, gr % kh].reshape(-1, D)[:k]
            Vv = blk[:, kh * 64 * D:].view(-1, vh, V, 64)[:, gr % vh].transpose(1, 2).reshape(-1, V)[:k]
            qq = q[row:row + m, h * D:(h + 1) * D].double()
            f = scale * (1 + temp * torch.log(torch.floor((p + 1) / 40.0) + 1))[:, None].double()
            sc, size = qq @ K.t() * f, qq.abs() @ K.abs().t() * f
            if cap:
                sc, size = cap * torch.tanh(sc / cap), size + cap
            if bias:
                e = r1[h].double() * torch.log1p(r2[h].double() * d.clamp(min=0))
                sc, size = sc - e, size + e
            if table:
                sc = sc + tab[h].double()[d.clamp(0, table - 1)]
            sc = sc.masked_fill(hide, -math.inf)
            full = torch.cat([sc, sk[h].double().expand(m, 1)], 1) if sink else sc
            w = torch.softmax(full, 1)[:, :k]
            err = 2.0 ** -24 * (D + 8) * size.masked_fill(hide, 0).max(1).values + 2.0 ** -22 * (8 + sc.masked_fill(hide, 0).abs().max(1).values)
            gg = torch.sigmoid(gt[row:row + m, h].double())[:, None] if gate else 1.0
            ref[row:row + m, h * hs:h * hs + V] = w @ Vv * gg
            bound[row:row + m, h * hs:h * hs + V] = (2 * err[:, None] + k * 2.0 ** -24) * (w @ Vv.abs()) * gg + 2.0 ** -22
        row += m
    return out, ref, bound


def check(tm, *args, **kw):
    out, ref, bound = run(tm, *args, **kw)
    assert bool(((out.double() - ref).abs() <= bound).all())
    assert float(bound.max()) < 0.01  # (results are sums of numbers of size one)
    return out


@pytest.mark.parametrize('D,V', [(4, 4), (60, 64), (64, 68), (68, 128), (128, 132), (132, 12), (252, 192), (256, 196), (256, 256)])
@pytest.mark.parametrize('rows', [0, 1])
def test_sizes(tm, cuda, D, V, rows):
    out = check(tm, D, V, PORTIONS[rows], 8, 2, splits=1 + 4 * rows)
    assert float((out - run(tm, D, V, PORTIONS[rows], 8, 2, kernel=1)[0]).abs().max()) < 1e-4  # the row kernel's results


@pytest.mark.parametrize('H,G', [(4, 1), (15, 1), (16, 1), (17, 1), (40, 2), (32, 8), (6, 2), (5, 5)])
def test_groups(tm, cuda, H, G):
    for rows in (0, 1):
        check(tm, 64, 32, PORTIONS[rows], H, G, splits=1 + 7 * rows)


FORMS = [dict(cap=3.0), dict(sink=True), dict(window=20), dict(window=70, keep=5), dict(chunk=48), dict(bias=True), dict(table=9), dict(gate=True), dict(space=5),
         dict(k_heads=1, v_heads=2), dict(temp=0.3), dict(cap=3.0, sink=True, window=33, keep=17, bias=True, table=300, gate=True, space=1, temp=0.1)]


@pytest.mark.parametrize('form', FORMS, ids=lambda f: '-'.join(f))
def test_modifiers(tm, cuda, form):
    for rows, splits in ((0, 1), (1, 1), (1, 3)):
        check(tm, 96, 80, PORTIONS[rows], 8, 2, splits=splits, **form)


@pytest.mark.parametrize('form', [dict(window=20), dict(window=70, keep=5), dict(window=17, keep=40), dict(chunk=48)], ids=lambda f: '-'.join(f))
def test_entries_that_are_not_seen(tm, cuda, form):
    """entries before a window or a chunk that no row of a launch sees hold what they may, as those behind a sequence's own do"""
    for portions, splits in (([(1, 1), (3, 170), (20, 130)], 1), ([(1, 64), (1, 65), (1, 700), (1, 129)], 3)):
        check(tm, 96, 80, portions, 8, 2, splits=splits, unseen=True, **form)
