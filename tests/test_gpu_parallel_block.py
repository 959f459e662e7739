"""GPU tests of what a parallel block's fused product leaves behind: the cache entries of many rows bit for bit (rows in several blocks and sequences, a remainder
of rows and of channels, sizes on and off the eight-channel grid), and decode steps on both sides of the most rows whose keys and values the product itself
stores -- against the float64 oracle."""
import numpy as np
import pytest

from tests import layered_oracle as lo
from tests.gpu_helpers import host, release_all
from tests.test_gpu_febivik import Paged, attend
from tests.test_gpu_layered import TOL, _layer, engine_for, rel_err, small_model

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('dtype', [0, 1])
@pytest.mark.parametrize('G,D,V', [(2, 32, 48), (1, 8, 8), (3, 72, 136), (2, 20, 24)])
def test_rows_in_the_cache(tm, cuda, G, D, V, dtype):
    rng = np.random.default_rng(G * D + V)
    starts, counts = [60, 0, 127, 5], [70, 64, 1, 3]          # the first row's position and the rows of every sequence: 138 rows
    cache = Paged(dtype, G, D, V, [a + n for a, n in zip(starts, counts)], rng)
    before, base, size = host(cache.pool).copy().reshape(-1, cache.elems), cache.pool.data_ptr(), cache.elems * cache.eb
    spec = dict(heads=G, kv_heads=G, dim=D, vdim=V, scale=0.2, window=0, keep=0)
    seq = np.repeat(np.arange(4), counts)
    pos = np.concatenate([a + np.arange(n) for a, n in zip(starts, counts)])
    k, v = rng.normal(0, 1, (len(seq), G * D)), rng.normal(0, 1, (len(seq), G * V))
    k, v = (a.astype(np.float32) for a in (k, v))
    attend(tm, dtype, spec, cache, rng.normal(0, 1, (len(seq), G * D)), k, v, seq, pos, np.concatenate([[0], np.cumsum(counts)]),
           [a + n for a, n in zip(starts, counts)], kernel=1)
    def bits(a):
        return lo.to_bf16_bits(a).view(np.int16) if dtype == 0 else a
    want = before
    ptrs = host(cache.ptrs).view(np.uint64)
    for t in range(len(seq)):
        b, ti = int(ptrs[seq[t], pos[t] // 64] - base) // size, pos[t] % 64
        for g in range(G):
            want[b, (g * 64 + ti) * D:(g * 64 + ti) * D + D] = bits(k[t, g * D:g * D + D])
            at = G * 64 * D + (g * V + np.arange(V)) * 64 + ti
            want[b, at] = bits(v[t, g * V:g * V + V])
    assert np.array_equal(host(cache.pool).reshape(want.shape).view(np.uint8), want.view(np.uint8))


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('n', [64, 65])
def test_decode_rows_around_the_line(cuda, n, dtype):
    cfg, w = small_model(1)
    rng = np.random.default_rng(n)
    reqs = [rng.integers(0, cfg['vocab'], 6).tolist() for _ in range(n)]
    eng = engine_for(cfg, w, dtype, cache_blocks=n + 2, max_batch_size=n)
    sess = [eng.open_session() for _ in reqs]
    got = [eng.step_tokens([(s, r[:3], [0, 1, 2]) for s, r in zip(sess, reqs)]).reshape(n, 3, -1)]
    for i in range(3, 6):
        got.append(eng.step_tokens([(s, r[i:i + 1], [0]) for s, r in zip(sess, reqs)]).reshape(n, 1, -1))
    got = np.concatenate(got, axis=1)
    for r in (0, 1, n // 2, n - 1):
        assert rel_err(got[r], lo.forward(cfg, w, reqs[r])[0]) <= TOL[dtype], r
    eng.close()


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_weight_bytes(cuda, dtype):
    """the reported bytes are those of the weights (columns in whole groups of 128, bf16 in either type), not of the memory between tiles or between the parts of the fused product"""
    cfg = lo.make_config(2048, 203, [_layer(dim=8, vdim=8, ff=24)])
    eng = engine_for(cfg, lo.make_weights(cfg, 0), dtype)
    # [q | k | v], up: 2048 to 64 and 24 columns; [o | down]: 32 + 24 to 2048; head
    assert eng.stats()['weight_bytes'] == 2 * (2048 * (128 + 128) + 64 * 2048 + 2048 * 256)
    eng.close()
