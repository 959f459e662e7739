"""GPU test of the launch that ends a pre-norm layer, for widths whose rows fill one, several and not all of a workgroup's pieces of four elements, widths that are not made
of such pieces, few and many rows, and more layers than a thread asks for at once -- small models against the float64 oracle, the same bound as its other tests."""
import numpy as np
import pytest

from tests import sanozen_oracle as so
from tests.test_gpu_sanozen import TOL, engine, model_folder, rel_err

pytestmark = pytest.mark.gpu


SIZES = [(30, 3, 0), (40, 3, 4), (1024, 3, 8), (1028, 2, 0), (2048, 3, 8), (2052, 2, 8), (4096, 3, 0), (4100, 2, 8), (8192, 2, 0), (8196, 2, 8)]
DEEP = [(40, 10, 4), (1024, 9, 8), (2048, 10, 8), (4096, 10, 0), (4100, 6, 8), (8192, 5, 0)]


@pytest.mark.parametrize('width,layers,side,dtype', [(*s, 'float32') for s in SIZES + DEEP] + [(w, 1, s, 'bfloat16') for w, _, s in SIZES])
def test_widths(tmp_path, cuda, width, layers, side, dtype):
    cfg = so.make_config(width, 61, [so.hgrn2_layer(1, 8, 8, so.dense(8))] * layers, side=side)
    folder, w = model_folder(tmp_path, cfg, width)
    rng = np.random.default_rng(width)
    eng = engine(folder, dtype, max_batch_size=4)
    for lens in ((1, 2), (240, 21)):  # few rows and many
        reqs = [rng.integers(0, 61, n).tolist() for n in lens]
        sess = [eng.open_session() for _ in reqs]
        got = eng.step_tokens([(s, r, list(range(len(r)))) for s, r in zip(sess, reqs)]).reshape(sum(lens), -1)
        for s in sess:
            eng.close_session(s)
        ref, tol = np.concatenate([so.forward(cfg, w, r) for r in reqs]), TOL[dtype]
        # Deep models pass roundings on enlarged (2e-5 from one of every weight in fp32 at 10 layers of 40, 0.1 in bf16 at three): a layer's launches round some sixteen
        # times in fp32 and some eight times in bf16, of which one layer is taken
        one = {k: v * (1 + (2.0 ** -25 if dtype == 'float32' else 2.0 ** -10) * rng.normal(0, 1, v.shape)) for k, v in w.items()}
        tol = max(tol, (16 if dtype == 'float32' else 8) * rel_err(np.concatenate([so.forward(cfg, one, r) for r in reqs]), ref))
        assert tol < (1e-3 if dtype == 'float32' else 0.5)
        assert rel_err(got, ref) <= tol
    eng.close()
