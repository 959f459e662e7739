"""GPU test of the tiling rules for W4 products of up to 32 and of 65 to 256 rows (64-column tiles, gemm_decode.hip): sizes on both sides of their lines in
columns, k and rows, k-block counts that leave a short last slice, the fewest and the most rows, through the entry point that picks the tiling itself, against
the oracle."""
import numpy as np
import pytest
import torch

from lmdeploy_amd import _ffi
from tests.gpu_helpers import dev, host, release_all, st
from tests.test_gpu_ops import _QCACHE, _make_linear

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _release():
    yield
    release_all()


@pytest.mark.parametrize('K,N', [(128, 256), (896, 288), (1024, 224), (1152, 256), (2048, 1056), (4096, 5120), (4096, 5152), (4224, 5152), (6144, 7168),
                                 (6272, 7168), (13824, 512)])
@pytest.mark.parametrize('M', [1, 16, 17, 32, 65, 96, 128, 129, 250, 256])
def test_picked_tiling(tm, cuda, K, N, M):
    rng = np.random.default_rng(K + N + M)
    h, _ = _make_linear(tm, rng, K, N)
    x = rng.standard_normal((M, K)).astype(np.float16)
    y = torch.full((M + 1, N), 7.0, dtype=torch.float16, device='cuda')
    ws = torch.zeros(max(1, tm.tm_linear_workspace(h, M)), dtype=torch.uint8, device='cuda')
    _ffi.check(tm.tm_linear_forward(h, dev(x).data_ptr(), K, y.data_ptr(), N, M, 0, 0, 0, 0, ws.data_ptr(), st()))
    ref, got = x.astype(np.float32) @ _QCACHE[(K, N)][3], host(y).astype(np.float32)
    assert (np.abs(got[:M] - ref) <= 2e-3 + 2.0**-10 * np.abs(ref)).all()    # the bound of the W4 products' other tests: one rounding to fp16
    assert (got[M] == 7.0).all()
    _ffi.check(tm.tm_linear_destroy(h))
