"""GPU test of the decode attention's rule for how many key splits a row uses (attention_general.hip): rows that one split finishes, rows at the edge of a
second one and rows with as many splits as the launch has, side by side in one launch, for launches of few and of many workgroups."""
import numpy as np
import pytest

from tests.gpu_helpers import release_all
from tests.test_gpu_febivik import Paged, _rounded, attend, row_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('splits', [2, 8])
@pytest.mark.parametrize('window,keep', [(0, 0), (300, 5)])
@pytest.mark.parametrize('seqs,heads,kv_heads,D,V', [(70, 8, 4, 32, 48), (18, 24, 8, 64, 16), (5, 40, 2, 40, 24), (3, 2, 1, 16, 136)])
def test_rows_of_one_and_of_many_splits(tm, cuda, seqs, heads, kv_heads, D, V, window, keep, splits):
    rng = np.random.default_rng(seqs)
    spec = dict(heads=heads, kv_heads=kv_heads, dim=D, vdim=V, scale=0.2, window=window, keep=keep)
    edges = [0, 1023, 256, 255, 63, 64, 511, 128, 512, 1024]
    lens = (edges + rng.integers(1, 300, 70).tolist())[:seqs]
    cache = Paged(0, kv_heads, D, V, [n + 1 for n in lens], rng)
    K = [_rounded(rng.normal(0, 1, (n + 1, kv_heads, D)), 0) for n in lens]
    W = [_rounded(rng.normal(0, 1, (n + 1, kv_heads, V)), 0) for n in lens]

    def call(lo, hi, kernel, prefill, n):
        rs = np.repeat(np.arange(seqs), np.subtract(hi, lo))
        rp = np.concatenate([np.arange(a, b) for a, b in zip(lo, hi)]).astype(int)
        q = _rounded(rng.normal(0, 1, (len(rs), heads * D)), 0)
        kn, vn = (np.stack([c[s][p].reshape(-1) for s, p in zip(rs, rp)]) for c in (K, W))
        cu = np.concatenate([[0], np.cumsum(np.subtract(hi, lo))])
        return q, attend(tm, 0, spec, cache, q, kn, vn, rs, rp, cu, hi, kernel, n, prefill)

    call([0] * seqs, lens, 2, 1, 1)                           # fills the cache
    for kernel in (3, 1):                                     # the matrix-core kernel, the row kernel: both share the rule and the merge
        q, got = call(lens, [n + 1 for n in lens], kernel, 0, splits)
        for s, n in enumerate(lens):
            ref = row_oracle(spec, q[s], K[s][:n + 1], W[s][:n + 1], n)
            # weights and results are rounded to bf16, 2^-9 of each: 3e-2 of the largest value leaves the same room as the kernels' other tests
            assert np.abs(got[s] - ref).max() <= 3e-2 * max(1.0, np.abs(ref).max()), (kernel, s, n)
