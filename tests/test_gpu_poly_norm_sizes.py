"""GPU test of PolyNorm feed-forwards whose rows fill one, several and not all of a workgroup's pieces of four elements, rows that are not made of such pieces, few and
many rows -- a one-layer model against the float64 oracle, the same bound as its other tests."""
import numpy as np
import pytest

from tests import sanozen_oracle as so
from tests.test_gpu_sanozen import TOL, engine, model_folder, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('ff', [4, 30, 2048, 2052, 4100, 9216, 9220, 16388, 24576, 24580, 24578])
@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
def test_row_lengths(tmp_path, cuda, ff, dtype):
    cfg = so.make_config(64, 97, [so.hgrn2_layer(2, 8, 8, so.dense(ff))])
    folder, w = model_folder(tmp_path, cfg, ff)
    rng = np.random.default_rng(ff)
    eng = engine(folder, dtype, max_batch_size=4)
    for lens in ((1, 2), (256, 41)):  # few rows and many
        reqs = [rng.integers(0, 97, n).tolist() for n in lens]
        sess = [eng.open_session() for _ in reqs]
        got = eng.step_tokens([(s, r, list(range(len(r)))) for s, r in zip(sess, reqs)]).reshape(sum(lens), -1)
        for s in sess:
            eng.close_session(s)
        assert rel_err(got, np.concatenate([so.forward(cfg, w, r) for r in reqs])) <= TOL[dtype]
    eng.close()
