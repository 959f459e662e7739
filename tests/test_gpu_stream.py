"""GPU tests of the unquantised products (gemm_stream.h) where their kernels can go wrong: row counts around the tile heights, columns around
the tile widths, one to three steps of k and odd counts of them, every kernel of the dispatch; slices of k that meet across workgroups; items whose
row tiles are one list.  Bounds: a sum of K products in fp32 in any order is within K 2^-24 sum|x w| of the exact one, a bf16 result adds 2^-8 |y|."""
import ctypes as C

import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from tests import bedenex_oracle as bo
from tests import febivik_oracle as fo
from tests import layered_oracle as lo
from tests import roravik_oracle as ro
from tests.gpu_helpers import release_all, st
from tests.test_gpu_bedenex import engine as bedenex_engine
from tests.test_gpu_bedenex import model_folder as bedenex_folder
from tests.test_gpu_febivik import engine, model_folder
from tests.test_gpu_febivik import rel_err as rel_err_febivik
from tests.test_gpu_layered import TOL, _layer, engine_for, rel_err
from tests.test_gpu_roravik import engine as roravik_engine
from tests.test_gpu_roravik import model_folder as roravik_folder
from tests.test_host import stream_plan

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


def check(got, ref, size, K, bf16):
    bound = K * 2.0 ** -24 * size + (2.0 ** -8 if bf16 else 2.0 ** -22) * ref.abs() + 1e-30
    assert bool(((got.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize('dtype', [0, 1])
@pytest.mark.parametrize('K,N,rows', [
    (32, 130, (1, 63, 64, 65, 127, 256, 257)),      # one step, a ragged last column tile
    (96, 4100, (2, 16, 17, 129, 1500)),             # three steps; 256 x 128 tiles with a ragged edge on both sides
    (1056, 2304, (3, 33, 300, 2100)),               # 33 steps, 256 x 256 tiles
    (2080, 2048, (5, 48, 255)),
    (200, 512, (70, 511, 513)),
    (9000, 130, (2, 20, 40)),                       # waves that take several chunks of a long k, up to a ragged end
])
def test_products_at_the_edges_of_tiles(tm, cuda, dtype, K, N, rows):
    g = torch.Generator('cuda').manual_seed(K + N)
    w = torch.randn(N, K, generator=g, device='cuda').bfloat16()
    h = C.c_void_p()
    _ffi.check(tm.tm_dense_create(C.byref(h), K, N, dtype, w.data_ptr(), st()))
    T = torch.bfloat16 if dtype == 0 else torch.float32
    ldx = (K + 31) // 32 * 32 + 32
    for M in rows:
        x = torch.full((M, ldx), 5.0, device='cuda', dtype=T)
        x[:, :K] = torch.randn(M, K, generator=g, device='cuda').to(T)
        ref, size = x[:, :K].double() @ w.double().t(), x[:, :K].double().abs() @ w.double().abs().t()
        for ldy in (N, N + 5, (N + 7) // 8 * 8 + 8):      # rows that start on 16 bytes and rows that do not
            y = torch.full((M + 1, ldy), -3.0, device='cuda', dtype=T)
            _ffi.check(tm.tm_dense_forward(h, x.data_ptr(), ldx, y.data_ptr(), ldy, M, 0, 1.0, st()))
            check(y[:M, :N], ref, size, K, dtype == 0)
            assert bool((y[M] == -3.0).all()) and bool((y[:M, N:] == -3.0).all())      # nothing is written beyond
        y = torch.randn(M, N, generator=g, device='cuda')
        old = y.double()
        _ffi.check(tm.tm_dense_forward(h, x.data_ptr(), ldx, y.data_ptr(), N, M, 2, 0.25, st()))
        check(y, old + 0.25 * ref, 0.25 * size + old.abs(), K, False)
    _ffi.check(tm.tm_dense_destroy(h))


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('rows', [3, 20, 40, 64])
def test_slices_of_k_meet_in_any_order(cuda, dtype, rows):
    """decode steps of an engine, whose products may be cut along k: widths and feed-forwards of 33 and 130 (bf16) and 66 and 260 (fp32) steps,
    one, two and four row tiles; the same step again gives the same bits (slices are added in their own order)"""
    cfg = lo.make_config(1056, 203, [_layer(heads=8, kv_heads=2, dim=32, vdim=32, ff=4160), _layer(heads=8, kv_heads=2, dim=32, vdim=32, ff=2080)], mult=0.4)
    w = lo.make_weights(cfg, 5)
    eng = engine_for(cfg, w, dtype, max_batch_size=64, cache_blocks=70)
    rng = np.random.default_rng(rows)
    toks = rng.integers(0, cfg['vocab'], (rows, 3))
    outs = []
    for _ in range(3):
        s = [eng.open_session() for _ in range(rows)]
        outs.append([eng.step_tokens([(s[i], [int(toks[i, k])], [0]) for i in range(rows)]) for k in range(3)])
        for i in s:
            eng.close_session(i)
    assert all(np.array_equal(a, b) for o in outs[1:] for a, b in zip(o, outs[0]))
    got = np.stack(outs[0], 1)
    for i in range(0, rows, 7):
        assert rel_err(got[i], lo.forward(cfg, w, toks[i].tolist())[0]) <= (3e-5 if dtype == 'float32' else 4e-2)
    eng.close()


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('rows,ff', [(3, 8320), (20, 8320), (65, 4160), (100, 4160), (250, 4160)])
def test_slices_of_k_of_long_sums_and_of_several_row_blocks(cuda, dtype, rows, ff):
    """the same for sums that are cut whatever the format, and for two to four blocks of 64 rows: counters and slabs of every (column group, block)"""
    cfg = lo.make_config(1056, 203, [_layer(heads=8, kv_heads=2, dim=32, vdim=32, ff=ff)], mult=0.4)
    w = lo.make_weights(cfg, 6)
    eng = engine_for(cfg, w, dtype, max_batch_size=256, cache_blocks=260)
    toks = np.random.default_rng(rows).integers(0, cfg['vocab'], (rows, 2))
    outs = []
    for _ in range(3):
        s = [eng.open_session() for _ in range(rows)]
        outs.append([eng.step_tokens([(s[i], [int(toks[i, k])], [0]) for i in range(rows)]) for k in range(2)])
        for i in s:
            eng.close_session(i)
    assert all(np.array_equal(a, b) for o in outs[1:] for a, b in zip(o, outs[0]))
    got = np.stack(outs[0], 1)
    for i in [0, 1, rows // 2, rows - 1] + list(range(0, rows, 13)):
        assert rel_err(got[i], lo.forward(cfg, w, toks[i].tolist())[0]) <= (3e-5 if dtype == 'float32' else 4e-2)
    eng.close()


def test_row_tiles_of_many_items(cuda, tmp_path):
    """prompts through 70 experts (more items than a wave has lanes), most of them with a few rows, some with none"""
    cfg = fo.make_config(64, 97, [fo.attention_layer(2, 1, 8, 8, 0.3, 16, 1, 4, mlp=fo.moe(70, 2, 24, 1.5, 8))])
    toks = np.random.default_rng(1).integers(0, 97, 300).tolist()
    folder, w = model_folder(tmp_path, cfg, 3)
    eng = engine(folder, 'float32')
    s = eng.open_session()
    got = eng.step_tokens([(s, toks, list(range(300)))])
    assert rel_err_febivik(got, fo.forward(cfg, w, toks)) <= 3e-5
    eng.close()


@pytest.mark.parametrize('K,N,gated,rows', [
    (128, 16, 0, (1, 17, 65, 300)),                   # one column tile
    (256, 16, 0, (17, 65, 300)),                      # ... and more than one block of 128 k
    (2048, 16, 0, (1, 65, 300)),
    (256, 4128, 1, (1, 16, 33, 64, 129)),             # a ragged last column group, gated
    (2048, 2080, 0, (8, 16, 31, 64, 200, 257, 1100)),  # slices of k that meet in a reduce launch; tiles of every height
    (4096, 544, 0, (3, 20, 64)),
    (1024, 24576, 1, (16, 17, 64)),                   # both sides of the line to the general kernel
    (512, 9216, 1, (513, 2111)),
    (128, 4096, 0, (256, 257, 512, 513)),             # ... and of the lines at one round of 64 x 64 tiles, or of the general kernel's 64 x 128
    (128, 14336, 0, (16, 17, 64, 65, 128, 129)),
    (128, 32784, 0, (15, 17)),                        # ... and where that has just more than one round for a few rows
])
def test_f16_linears_at_the_edges(tm, cuda, K, N, gated, rows):
    g = torch.Generator('cuda').manual_seed(K + N)
    w = (torch.randn(K, N, generator=g, device='cuda') / K ** 0.5).half()
    h = C.c_void_p()
    _ffi.check(tm.tm_linear_create(C.byref(h), K, N, 1, 128))
    _ffi.check(tm.tm_linear_prepare(h, w.data_ptr(), None, None, st()))
    No = N // 2 if gated else N
    for M in rows:
        ldx = K + 8
        x = torch.randn(M, ldx, generator=g, device='cuda').half()
        ref, size = x[:, :K].double() @ w.double(), x[:, :K].double().abs() @ w.double().abs()
        err = K * 2.0 ** -24 * size
        if gated:       # d silu <= 1.1 d; the product of two values with errors; exp and division within a few fp32 ulps
            s, u = torch.nn.functional.silu(ref[:, 0::2]), ref[:, 1::2]
            err = 1.1 * err[:, 0::2] * (u.abs() + err[:, 1::2]) + s.abs() * err[:, 1::2] + 2.0 ** -20 * (s * u).abs()
            ref = s * u
        bound = err + 2.0 ** -11 * (ref.abs() + err) + 2.0 ** -24      # one rounding to fp16, subnormal results included
        ws = torch.zeros(tm.tm_linear_workspace(h, M) // 4 + 4, device='cuda')
        for work, ldy in ((ws.data_ptr(), No), (None, No + 3), (ws.data_ptr(), No + 8)):
            y = torch.full((M + 1, ldy), -3.0, device='cuda', dtype=torch.half)
            _ffi.check(tm.tm_linear_forward(h, x.data_ptr(), ldx, y.data_ptr(), ldy, M, gated, 0, 0, 0, work, st()))
            assert bool(((y[:M, :No].double() - ref).abs() <= bound).all()), (M, ldy)
            assert bool((y[M] == -3.0).all()) and bool((y[:M, No:] == -3.0).all())
    _ffi.check(tm.tm_linear_destroy(h))


def stream_errs(eng, toks, trail):
    """rms error of every row of the residual stream behind the first layer of a prompt taken in one forward, relative to the stream's size"""
    eng.stop_after(1)
    s = eng.open_session()
    eng.step_tokens([(s, toks, [])])
    d = eng.fetch_residual(len(toks)) - trail[0]
    eng.close_session(s)
    return np.sqrt((d ** 2).mean(-1)) / np.sqrt((trail[0] ** 2).mean())


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('rows,right_heads', [(2048, 5), (3000, 5), (3000, 4)])
def test_segments_that_begin_at_odd_multiples_of_128(cuda, tmp_path, dtype, rows, right_heads):
    """the projections of a parallel pair of mixers are one product whose columns read six inputs of a row: borders at 2048, 2688, 3328, 3968 and 4608, of
    which 2688 and 3968 lie in the middle of 256 columns (four heads: all at multiples of 256), at row counts where a product of one input takes
    256-column tiles.  bf16 rounds the mixed rows, the
    queries, keys, values and weights of the window, the joined heads and the matrices' inputs, 2^-9 each, and a norm behind the sum scales a small
    row up: within 4e-2 of the stream's size; a projection of the wrong input is 0.3 off in every row"""
    cfg = ro.make_config(128, 97, [ro.parallel_layer(8, 4, 128, 128, 64, right_heads, 128)])
    toks = np.random.default_rng(rows).integers(0, 97, rows).tolist()
    folder, w = roravik_folder(tmp_path, cfg, 3)
    eng = roravik_engine(folder, dtype, max_batch_size=1, session_len=3072, cache_blocks=64, max_prefill_token_num=3072)
    errs = stream_errs(eng, toks, ro.forward(cfg, w, toks, True)[1])
    eng.close()
    assert errs.max() <= (3e-5 if dtype == 'float32' else 4e-2), np.sort(errs)[-5:]


def _wide_models():
    """one-layer models and row counts at which the products named take 256 x 256 tiles (plan of the bf16 kernels), ragged in rows"""
    ret = dict(heads=2, dim=16, vdim=16, decay=[0.8, 0.99])
    light = dict(heads=2, dim=16, vdim=16, decay=[0.8, 0.99])
    return {
        'gate and up in one tile': (ro, roravik_folder, roravik_engine, ro.make_config(4608, 97, [ro.retention_layer(**ret, mlp=ro.dense(4096))]), 2000),
        'gate and up, row tiles of items': (ro, roravik_folder, roravik_engine,
                                            ro.make_config(4608, 97, [ro.retention_layer(**ret, mlp=ro.moe(2, 2, 2048, 1, 1, 2048))]), 1000),
        'row tiles of items': (fo, model_folder, engine, fo.make_config(512, 97, [fo.lightning_layer(**light, mlp=fo.moe(2, 2, 2048))]), 2990),
        'activation with two numbers': (fo, model_folder, engine, fo.make_config(512, 97, [fo.lightning_layer(**light, mlp=fo.dense(4096))]), 3000),
        'heads as items, gated sum into the stream': (bo, bedenex_folder, bedenex_engine,
                                                      bo.make_config(2816, 97, [bo.latent_layer(8, 128, 16, 64, 512, 0.05)]), 3000),
    }


@pytest.mark.parametrize('name', list(_wide_models()))
def test_epilogues_of_256_column_tiles(cuda, tmp_path, name):
    oracle, folder, build, cfg, rows = _wide_models()[name]
    toks = np.random.default_rng(rows).integers(0, 97, rows).tolist()
    path, w = folder(tmp_path, cfg, 3)
    eng = build(path, 'bfloat16', max_batch_size=1, session_len=3072, cache_blocks=64, max_prefill_token_num=3072)
    errs = stream_errs(eng, toks, oracle.forward(cfg, w, toks, True)[1])
    eng.close()
    # roundings to bf16 (2^-9) of the normed rows, heads, activations and their products' inputs; a column from a wrong place is off by its own size
    assert errs.max() <= 4e-2, np.sort(errs)[-5:]


@pytest.mark.parametrize('dtype,K', [(0, 4096), (0, 8192), (1, 2048), (0, 2048), (0, 4128)])
def test_turned_tiles(tm, cuda, dtype, K):
    """tiles of 128 KB and more (multiples of 64 KB) begin at a step of their own, shorter ones and those of other lengths do not: more than sixteen times 256 columns,
    the last not full, in every kernel"""
    N = 4500
    g = torch.Generator('cuda').manual_seed(K)
    w = torch.randn(N, K, generator=g, device='cuda').bfloat16()
    h = C.c_void_p()
    _ffi.check(tm.tm_dense_create(C.byref(h), K, N, dtype, w.data_ptr(), st()))
    T = torch.bfloat16 if dtype == 0 else torch.float32
    for M in (1, 20, 40, 65, 200, 300, 1100, 2100):
        x = torch.randn(M, K, generator=g, device='cuda').to(T)
        ref, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
        y = torch.full((M + 1, N), -3.0, device='cuda', dtype=T)
        _ffi.check(tm.tm_dense_forward(h, x.data_ptr(), K, y.data_ptr(), N, M, 0, 1.0, st()))
        check(y[:M], ref, size, K, dtype == 0)
        assert bool((y[M] == -3.0).all())
    _ffi.check(tm.tm_dense_destroy(h))


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_turned_tiles_in_slices(cuda, dtype):
    """the same in an engine's decode steps, whose products may be cut along k, and in its prompts"""
    cfg = lo.make_config(4096, 203, [_layer(heads=8, kv_heads=2, dim=32, vdim=32, ff=4160)], mult=0.4)
    w = lo.make_weights(cfg, 5)
    eng = engine_for(cfg, w, dtype, max_batch_size=20, cache_blocks=24)
    rng = np.random.default_rng(3)
    for rows in (3, 20):
        toks = rng.integers(0, cfg['vocab'], (rows, 6))
        sess = [eng.open_session() for _ in range(rows)]
        got = [eng.step_tokens([(s, t[:4], [0, 1, 2, 3]) for s, t in zip(sess, toks)]).reshape(rows, 4, -1)]
        got += [eng.step_tokens([(s, t[i:i + 1], [0]) for s, t in zip(sess, toks)]).reshape(rows, 1, -1) for i in (4, 5)]
        got = np.concatenate(got, axis=1)
        for r in (0, rows - 1):
            assert rel_err(got[r], lo.forward(cfg, w, toks[r].tolist())[0]) <= TOL[dtype]
        for s in sess:
            eng.close_session(s)
    eng.close()


@pytest.mark.parametrize('dtype,width', [('float32', 2048), ('bfloat16', 4096)])
def test_turned_items(tmp_path, cuda, dtype, width):
    """the same in the first product of a mixture's experts: each item's tiles begin where their own columns say, whatever item it is; prompts and decode steps"""
    cfg = fo.make_config(width, 97, [fo.lightning_layer(2, 8, 8, [0.9, 0.9], fo.moe(3, 2 if dtype == 'float32' else 3, 600, 1.0, 0))])
    w = fo.random_weights(cfg, 11)
    folder = str(tmp_path / 'm')
    fo.write_checkpoint(folder, cfg, w)
    rng = np.random.default_rng(2)
    reqs = [rng.integers(0, 97, 132).tolist() for _ in range(2)]
    eng = engine(folder, dtype)
    sess = [eng.open_session() for _ in reqs]
    got = [eng.step_tokens([(s, r[:130], [63, 129]) for s, r in zip(sess, reqs)]).reshape(2, 2, -1)]
    got += [eng.step_tokens([(s, r[i:i + 1], [0]) for s, r in zip(sess, reqs)]).reshape(2, 1, -1) for i in (130, 131)]
    ref = np.stack([fo.forward(cfg, w, r)[[63, 129, 130, 131]] for r in reqs])
    assert rel_err_febivik(np.concatenate(got, axis=1), ref) <= TOL[dtype]
    bad = dict(w)                    # one group of columns that takes its steps from another place than its rows do
    for e in range(3):
        bad[f'l0.mlp.e{e}.up'] = m = np.array(w[f'l0.mlp.e{e}.up'])
        m[256:512] = np.roll(m[256:512], 128, axis=1)
    wrong = np.stack([fo.forward(cfg, bad, r)[[63, 129, 130, 131]] for r in reqs])
    assert rel_err_febivik(wrong, ref) > 2 * TOL[dtype]
    eng.close()


@pytest.mark.parametrize('K,N,M,tile', [(264, 2049, 7990, 3), (264, 2052, 8001, 3), (264, 2299, 4000, 3), (1000, 3000, 2500, 4), (264, 1027, 900, 6)])
@pytest.mark.parametrize('more', [0, 1, 2, 3])              # rows of the stream on and off multiples of 16 bytes, a ragged last column tile
def test_sums_into_the_stream(tm, cuda, K, N, M, tile, more):
    """y += alpha x w, whose old values a 256 x 256 tile reads sixteen together and the smaller ones one by one"""
    assert stream_plan(0, K, N, M, 0)[0] == tile
    g = torch.Generator('cuda').manual_seed(N + more)
    w, x = torch.randn(N, K, generator=g, device='cuda').bfloat16(), torch.zeros(M, (K + 31) // 32 * 32, device='cuda').bfloat16()
    x[:, :K] = torch.randn(M, K, generator=g, device='cuda').bfloat16()
    ldy = N + more
    y = torch.randn(M + 1, ldy, generator=g, device='cuda')
    old = y.double()
    h = C.c_void_p()
    _ffi.check(tm.tm_dense_create(C.byref(h), K, N, 0, w.data_ptr(), st()))
    _ffi.check(tm.tm_dense_forward(h, x.data_ptr(), x.shape[1], y.data_ptr(), ldy, M, 2, 0.5, st()))
    _ffi.check(tm.tm_dense_destroy(h))
    ref, size = old[:M, :N] + 0.5 * (x[:, :K].double() @ w.double().t()), x[:, :K].double().abs() @ w.double().abs().t()
    assert bool(((y[:M, :N].double() - ref).abs() <= K * 2.0 ** -24 * size + 2.0 ** -23 * ref.abs() + 1e-30).all())
    assert torch.equal(y[:M, N:].double(), old[:M, N:]) and torch.equal(y[M].double(), old[M])
