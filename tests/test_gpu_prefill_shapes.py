"""GPU test of the fp16 prefill attention's variants (one or two row tiles a wave; one, two or four query heads of a kv head a workgroup) at the borders of
the rule that chooses them: prompts of 1 to 129 rows, few and many of them, behind no context and behind one that ends inside a 32-key half."""
import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from tests.gpu_helpers import dev, release_all, st

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('heads,kv_heads,batch,longest,hist', [
    (32, 8, 17, 16, 0), (32, 8, 17, 16, 70), (28, 7, 20, 9, 33),        # four heads of a workgroup
    (16, 8, 33, 16, 0), (32, 8, 17, 17, 40), (12, 2, 43, 32, 0),        # two
    (32, 8, 17, 33, 0), (7, 1, 80, 16, 31), (32, 8, 16, 32, 95),        # one, with one row tile ...
    (5, 1, 2, 129, 200), (8, 8, 3, 64, 0), (32, 8, 5, 300, 1),
    (32, 8, 16, 128, 0), (32, 8, 16, 127, 65), (16, 4, 8, 449, 0),      # ... and with two
])
def test_variants(tm, cuda, heads, kv_heads, batch, longest, hist):
    rng = np.random.default_rng(heads + batch + longest + hist)
    q_len = [longest] + [int(n) for n in rng.integers(1, longest + 1, batch - 1)]
    k_len = [n + (hist if b % 3 else 0) for b, n in enumerate(q_len)]
    off = np.concatenate([[0], np.cumsum([(k + 63) // 64 * 64 for k in k_len])]).astype(np.int32)
    cu = np.concatenate([[0], np.cumsum(q_len)]).astype(np.int32)
    g = torch.Generator('cuda').manual_seed(batch)
    q = torch.randn(int(cu[-1]), heads, 128, generator=g, device='cuda').half()
    k = torch.full((kv_heads, int(off[-1]), 128), float('nan'), device='cuda', dtype=torch.half)      # behind a context: masked, not multiplied
    vt = torch.zeros(kv_heads, 128, int(off[-1]), device='cuda', dtype=torch.half)
    out = torch.full_like(q, 7.0)
    for b in range(batch):
        s = slice(int(off[b]), int(off[b]) + k_len[b])
        k[:, s] = torch.randn(kv_heads, k_len[b], 128, generator=g, device='cuda').half()
        vt[:, :, s] = torch.randn(kv_heads, 128, k_len[b], generator=g, device='cuda').half()
    _ffi.check(tm.tm_prefill_attention(out.data_ptr(), q.data_ptr(), heads * 128, k.data_ptr(), vt.data_ptr(), int(off[-1]), dev(cu).data_ptr(),
                                       dev(off).data_ptr(), dev(np.asarray(k_len, np.int32)).data_ptr(), batch, longest, heads, kv_heads, 0.0, st()))
    for b in range(batch):
        s, r = slice(int(off[b]), int(off[b]) + k_len[b]), slice(int(cu[b]), int(cu[b + 1]))
        kk, vv = (x.double().repeat_interleave(heads // kv_heads, 0) for x in (k[:, s], vt[:, :, s]))
        score = torch.matmul(q[r].double().permute(1, 0, 2).contiguous(), kk.permute(0, 2, 1).contiguous()) / 128 ** 0.5
        i = torch.arange(q_len[b], device='cuda')[:, None] + k_len[b] - q_len[b]
        p = torch.softmax(score.masked_fill(torch.arange(k_len[b], device='cuda')[None] > i, -1e300), -1)
        ref = torch.matmul(p, vv.permute(0, 2, 1).contiguous()).permute(1, 0, 2)
        size = torch.matmul(p, vv.abs().permute(0, 2, 1).contiguous()).permute(1, 0, 2)
        # weights and result are rounded to fp16 once (2^-11 each), scores and sums are fp32: a score of 60 is off by 60 * 2^-23 at most
        assert bool(((out[r].double() - ref).abs() <= 2.0 ** -10 * size + 2.0 ** -11 * ref.abs() + 1e-6).all()), b
