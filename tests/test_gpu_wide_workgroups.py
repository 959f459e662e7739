"""GPU test of few-row products whose workgroups cover 128 columns, on both sides of their rule (column counts that end inside a workgroup and inside a column tile, two
and four row tiles), and of experts whose workgroups cover 96: the bound of the other stream kernels' tests, and the float64 oracle behind a one-layer model."""
import ctypes as C

import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from tests import febivik_oracle as fo
from tests.gpu_helpers import st
from tests.test_gpu_febivik import TOL, engine
from tests.test_gpu_stream import check
from tests.test_host import stream_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N', [24577, 27650, 32768])
def test_one_slice(tm, cuda, N):
    K, g = 4104, torch.Generator('cuda').manual_seed(N)
    w = torch.randn(N, K, generator=g, device='cuda').bfloat16()
    h = C.c_void_p()
    _ffi.check(tm.tm_dense_create(C.byref(h), K, N, 0, w.data_ptr(), st()))
    w = w.double()
    for M in (16, 17, 32, 33, 63, 64):
        assert (stream_plan(0, K, N, M)[:2] == (2, 8)) == (M > 16)
        x = torch.zeros((M, 4128), device='cuda', dtype=torch.bfloat16)
        x[:, :K] = torch.randn(M, K, generator=g, device='cuda').bfloat16()
        ref, size = x[:, :K].double() @ w.t(), x[:, :K].double().abs() @ w.abs().t()
        y = torch.full((M + 1, N + 3), -3.0, device='cuda', dtype=torch.bfloat16)
        _ffi.check(tm.tm_dense_forward(h, x.data_ptr(), 4128, y.data_ptr(), N + 3, M, 0, 1.0, st()))
        check(y[:M, :N], ref, size, K, True)
        assert bool((y[M] == -3.0).all()) and bool((y[:M, N:] == -3.0).all())
    _ffi.check(tm.tm_dense_destroy(h))


@pytest.mark.parametrize('n', [2, 8, 17, 40])
def test_items(tmp_path, cuda, n):
    """nine experts (one shared) of width 2048: 288 workgroups of 64 columns where all of them have rows, 198 of 96"""
    cfg = fo.make_config(2048, 97, [fo.lightning_layer(2, 8, 8, [0.9, 0.9], fo.moe(8, 2, 40, 1.0, 40))])
    w = fo.random_weights(cfg, n)
    folder = str(tmp_path / 'm')
    fo.write_checkpoint(folder, cfg, w)
    rng = np.random.default_rng(n)
    reqs = [rng.integers(0, 97, 2).tolist() for _ in range(n)]
    eng = engine(folder, 'bfloat16', max_batch_size=n, cache_blocks=n + 2)
    sess = [eng.open_session() for _ in reqs]
    got = [eng.step_tokens([(s, r[i:i + 1], [0]) for s, r in zip(sess, reqs)]).reshape(n, -1) for i in range(2)]
    ref = np.stack([fo.forward(cfg, w, r) for r in reqs], axis=1)
    assert np.abs(np.stack(got) - ref).max() <= TOL['bfloat16'] * np.abs(ref).max()
    eng.close()
