"""GPU test of latent attention over whole prompts, whose keys and values every head makes of the latent entries: prompts around the blocks' borders side by side, layers that
read another layer's entries, later portions and decoded tokens over the same cache (attention on the entries), and batches in which only some prompts are whole -- against the
float64 oracle.  In bf16 every row has a bound of its own: a side vector next to zero, which the norm behind it scales up, makes a row here and there as rough as 0.4."""
import functools

import numpy as np
import pytest

from tests import bedenex_oracle as bo
from tests import sanozen_oracle as so
from tests import test_gpu_bedenex
from tests.test_gpu_sanozen import TOL, engine, row_errs

pytestmark = pytest.mark.gpu

SIZES = [(3, 64, 64, 128, 192), (2, 32, 32, 64, 72), (5, 48, 16, 128, 96), (2, 120, 8, 128, 264)]  # heads, dim, rot_dim, vdim, kv_rank


@functools.lru_cache(None)
def _case(H, D, R, V, C, side):
    """(model, weights, sequences, their logits, what each row's bound is in bf16): half the model tests' bound, or eight times the most that a rounding of every weight to bf16 moves
    the row in four draws, where that is more (the five layers round some eight times each: sqrt(40) roundings of such a size, and their spread)"""
    layers = [so.attention_layer(H, D, R, V, C, 40), so.hgrn2_layer(1, 8, 8), so.attention_layer(H + 1, D, R, V, C, 24, kv_from=0), so.attention_layer(H, D, R, V, C, 40),
              so.attention_layer(1, D, R, V, C, 16, kv_from=0)]  # (the last reads entries that another layer has replaced)
    cfg = so.make_config(56, 83, layers, side=side)
    w, rng = so.random_weights(cfg, 5), np.random.default_rng(D)
    seqs = [rng.integers(0, 83, n).tolist() for n in (300, 2, 63, 64, 65, 320, 129)]
    refs = [so.forward(cfg, w, s) for s in seqs]
    own = [np.full(len(s), TOL['bfloat16'] / 2) for s in seqs]
    for _ in range(4):
        one = {k: v * (1 + 2.0 ** -10 * rng.normal(0, 1, v.shape)) for k, v in w.items()}
        own = [np.maximum(a, 8 * row_errs(so.forward(cfg, one, s), r)) for a, s, r in zip(own, seqs, refs)]
    return cfg, w, seqs, refs, own


@pytest.mark.parametrize('dtype', ['float32', 'bfloat16'])
@pytest.mark.parametrize('side', [4, 0])
@pytest.mark.parametrize('H,D,R,V,C', SIZES)
def test_whole_prompts_and_what_follows(cuda, tmp_path, H, D, R, V, C, side, dtype):
    cfg, w, seqs, refs, own = _case(H, D, R, V, C, side)
    folder = str(tmp_path / 'm')
    so.write_checkpoint(folder, cfg, w)
    eng = engine(folder, dtype, max_batch_size=8, max_prefill_token_num=1024, cache_blocks=40)
    cut = [300, 2, 63, 64, 65, 190, 0]                            # whole prompts; the last two go on
    sess = [eng.open_session() for _ in seqs]
    errs = []

    def step(which, lo, hi):
        got = eng.step_tokens([(sess[i], seqs[i][lo[i]:hi[i]], list(range(hi[i] - lo[i]))) for i in which])
        at = 0
        for i in which:
            n = hi[i] - lo[i]
            errs.append(row_errs(got[at:at + n], refs[i][lo[i]:hi[i]]))
            at += n
            assert (errs[-1] <= (own[i][lo[i]:hi[i]] if dtype == 'bfloat16' else TOL[dtype])).all(), (i, lo[i], np.sort(errs[-1])[-8:])
    step(range(6), [0] * 7, cut)
    step([5, 6], cut, [0, 0, 0, 0, 0, 260, 129])                  # a later portion beside a whole prompt
    for t in range(260, 264):
        step([5], [t] * 7, [t + 1] * 7)
    for s in sess:
        eng.close_session(s)
    eng.close()
    errs = np.concatenate(errs)
    assert np.median(errs) <= TOL[dtype] / 4
    assert side or (np.concatenate(own) > TOL['bfloat16']).mean() < 1 / 6      # (without side vectors hardly a row's bound is above the model tests')


@pytest.mark.parametrize('kw', [{}, dict(loop=(0, 1, 2))])
@pytest.mark.parametrize('D,R,V,C', [(64, 64, 128, 192), (32, 32, 64, 104), (48, 80, 128, 136)])
def test_wide_blocks_and_runs_that_borrow_weights(cuda, tmp_path, D, R, V, C, kw):
    cfg = bo.make_config(64, 97, [bo.latent_layer(3, D, R, V, C, (D + R) ** -0.5)], **kw)
    folder, w = test_gpu_bedenex.model_folder(tmp_path, cfg, 3)
    rng = np.random.default_rng(C)
    eng = test_gpu_bedenex.engine(folder, 'bfloat16', max_batch_size=4, max_prefill_token_num=512, cache_blocks=24)
    seqs = [rng.integers(0, 97, n).tolist() for n in (130, 64, 191)]
    sess = [eng.open_session() for _ in seqs]
    got = eng.step_tokens([(s, t, list(range(len(t)))) for s, t in zip(sess, seqs)])
    for s in sess:
        eng.close_session(s)
    eng.close()
    assert test_gpu_bedenex.rel_err(got, np.concatenate([bo.forward(cfg, w, t) for t in seqs])) <= test_gpu_bedenex.TOL['bfloat16']
