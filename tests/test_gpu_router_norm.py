"""GPU test of the layer norm that also makes the router's logits: expert counts around its eight and sixteen, widths that end inside a step and a pass over the row, rows
on both sides of its line -- the logits of a one-layer model against the float64 oracle, rows with a clear choice of experts (see test_gpu_expert_tiles)."""
import numpy as np
import pytest

from tests import febivik_oracle as fo
from tests.test_gpu_expert_tiles import _moe_ff
from tests.test_gpu_febivik import TOL, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('width,experts', [(36, 3), (36, 8), (36, 9), (64, 16), (64, 17), (1028, 8), (2048, 8), (2052, 16), (4096, 5), (4100, 8)])
@pytest.mark.parametrize('rows', [1, 7, 256, 257])
def test_router_behind_the_norm(tmp_path, cuda, monkeypatch, width, experts, rows):
    cfg = fo.make_config(width, 97, [fo.lightning_layer(2, 8, 8, [0.9, 0.9], fo.moe(experts, 2, 24, 1.0, 24))])
    w = fo.random_weights(cfg, experts + width)
    folder = str(tmp_path / 'm')
    fo.write_checkpoint(folder, cfg, w)
    gaps, seed = [], rows
    monkeypatch.setattr(fo, 'moe_ff', lambda *a: _moe_ff(*a, gaps))
    while not (gaps and (np.concatenate(gaps) > 0.05).any()):        # (one row alone may have no clear choice, and would show nothing)
        gaps.clear()
        toks = np.random.default_rng(seed).integers(0, 97, rows).tolist()
        ref = fo.forward(cfg, w, toks)
        seed += 1000
    eng = engine(folder, 'bfloat16', max_batch_size=2, cache_blocks=12, session_len=512, max_prefill_token_num=512)
    got = eng.step_tokens([(eng.open_session(), toks, list(range(rows)))]).reshape(rows, -1)
    clear = np.concatenate(gaps) > 0.05
    assert clear.any() and (rows < 20 or clear.mean() > 0.5) and np.abs(got - ref)[clear].max() <= TOL['bfloat16'] * np.abs(ref).max()
    eng.close()
