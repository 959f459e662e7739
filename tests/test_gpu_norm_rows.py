"""GPU test of decode steps of a few rows of fp16 and W4 models whose products add to the residual stream and make the norm of their rows themselves: a row of one wave and of
several, two rows a wave, widths of one piece a wave to eight, the three shapes of the product, slices of the product ahead that meet in its launch, one row more than
it takes -- engines whose logits the attention or the feed-forward makes, against the oracle's separate sequence."""
import contextlib

import numpy as np
import pytest

from lmdeploy_amd.turbomind.engine import Engine
from lmdeploy_amd.turbomind.loader import export_weights
from oracle import tm_oracle as o
from tests import clear_models

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _norms(f):
    old = o.residual_rmsnorm
    try:
        o.residual_rmsnorm = f
        yield
    finally:
        o.residual_rmsnorm = old


def _mistakes(rows):
    """what a step could do wrong: the sum not kept, a factor of half the channels, another row's factor, channels' weights left out"""
    right = o.residual_rmsnorm
    yield lambda r, h, w, eps: (r, right(r, h, w, eps)[1])
    yield lambda r, h, w, eps: _times(right(r, h, w, eps), lambda inv, half: half / inv)
    if rows > 1:
        yield lambda r, h, w, eps: _times(right(r, h, w, eps), lambda inv, half: np.roll(inv, 1, 0) / inv)
    yield lambda r, h, w, eps: right(r, h, np.ones_like(w), eps)


def _times(result, factor):
    r, y = result
    sums = (r.astype(np.float32)**2).reshape(len(r), 2, -1).sum(2)
    inv, half = ((n / r.shape[1] + 1e-5)**-0.5 for n in (sums.sum(1, keepdims=True), sums[:, :1]))
    return r, (y.astype(np.float32) * factor(inv, half)).astype(np.float16)


@pytest.mark.parametrize('hidden,heads,kv_heads,inter,batch,attention', [
    (512, 2, 1, 256, 1, False), (512, 2, 1, 256, 9, True), (1024, 40, 4, 2304, 3, True), (1024, 4, 2, 2304, 16, False), (1536, 4, 2, 256, 5, False), (2048, 4, 1, 4608, 1, False),
    (2048, 4, 1, 4608, 4, False), (2048, 4, 1, 4608, 5, False), (2048, 4, 1, 256, 16, True), (2048, 2, 1, 8192, 8, False), (4096, 2, 1, 256, 8, True), (4096, 4, 1, 4608, 3, False),
    (4096, 2, 1, 256, 9, False), (512, 2, 1, 256, 17, False), (640, 2, 1, 256, 3, False)])
def test_decode(cuda, hidden, heads, kv_heads, inter, batch, attention):
    taken = hidden % 512 == 0 and (batch <= 8 or batch <= 16 and hidden <= 2048)
    _decode(o.ModelConfig(hidden=hidden, layers=2, q_heads=heads, kv_heads=kv_heads, head_dim=128, inter=inter, vocab=256, kv_bits=16, rope=o.RopeParam(128, 10000.0)),
            batch, attention, False, 1 if taken else 4)


# norms: launches of a step; up to eight rows one (the last), or two where the down product keeps its slices
@pytest.mark.parametrize('hidden,heads,kv_heads,inter,batch,attention,norms', [
    (2048, 16, 2, 2048, 1, False, 1), (2048, 16, 2, 2048, 2, True, 1), (2048, 16, 2, 2048, 5, False, 1), (2048, 16, 2, 2048, 8, True, 2), (2048, 16, 2, 2048, 9, False, 4),
    (2560, 16, 2, 11264, 3, False, 2), (4096, 16, 2, 2048, 7, False, 2), (4096, 16, 1, 11008, 1, False, 1), (4096, 32, 8, 14336, 2, False, 2)])
def test_decode_w4(cuda, hidden, heads, kv_heads, inter, batch, attention, norms):
    _decode(o.ModelConfig(hidden=hidden, layers=2, q_heads=heads, kv_heads=kv_heads, head_dim=128, inter=inter, vocab=256, kv_bits=8, rope=o.RopeParam(128, 10000.0)),
            batch, attention, True, norms)


# gate / up products that are faster behind a norm launch: fp16 whose last round of four-tile workgroups is nearly empty, W4 whose many workgroups would norm many rows each
@pytest.mark.parametrize('hidden,heads,kv_heads,inter,batch,quantized,norms', [
    (2048, 4, 1, 8448, 3, False, 3), (1536, 4, 1, 8960, 12, False, 3), (4096, 16, 2, 11008, 8, True, 4), (2048, 16, 2, 8192, 8, True, 2)])
def test_norm_launches_that_stay(cuda, hidden, heads, kv_heads, inter, batch, quantized, norms):
    _decode(o.ModelConfig(hidden=hidden, layers=2, q_heads=heads, kv_heads=kv_heads, head_dim=128, inter=inter, vocab=256, kv_bits=8 if quantized else 16,
                          rope=o.RopeParam(128, 10000.0)), batch, False, quantized, norms)


def _decode(cfg, batch, attention, quantized, launches):
    hidden = cfg.hidden
    w = clear_models.weights(cfg, batch, quantized=quantized, attention=attention)
    rng = np.random.default_rng(batch)
    w['tok_embeddings'] = (w['tok_embeddings'].astype(np.float32) * 2.0**rng.integers(0, 4, (cfg.vocab, 1))).astype(np.float16)    # (rows whose factors differ)
    for L in w['layers']:
        for n in ('attn_norm', 'ffn_norm'):
            L[n] = (L[n].astype(np.float32) * rng.choice([0.25, 0.5, 1], hidden)).astype(np.float16)
    eng = Engine.from_model_config(cfg, weight_type=0 if quantized else 1, max_batch_size=batch, session_len=64, quant_policy=cfg.kv_bits % 16, max_prefill_token_num=256)
    eng.load_weights(export_weights(cfg, w))
    eng.start()
    prompts = [rng.integers(0, cfg.vocab, 2 + i % 3).astype(np.int32) for i in range(batch)]
    eng.prefill(prompts, max_new_tokens=5)
    got = [eng.fetch_logits()]
    for _ in range(2):
        eng.decode(1)
        got.append(eng.fetch_logits())
    norms = eng.profile_decode(1)['residual_norm'][1]
    got.append(eng.fetch_logits())
    toks = eng.fetch()
    resid = eng.fetch_residual(batch)
    eng.close()
    assert norms == launches
    model = []

    class Kept(o.OracleModel):
        def __init__(self, *a, **k):
            super().__init__(*a, **k)
            model.append(self)
    old, o.OracleModel = o.OracleModel, Kept
    try:
        ref = clear_models.forced(cfg, w, prompts, toks, 3)
    finally:
        o.OracleModel = old
    bound = 2.0**-6    # half a dozen roundings to fp16 a layer of factors of about a hundred
    for m in _mistakes(batch):
        wrong = [np.nan_to_num(x, nan=6e4) for x in clear_models.forced(cfg, w, prompts, toks, 3, decode=lambda: _norms(m))]    # (one may overflow)
        assert clear_models.differ(wrong, ref) > 2 * bound
    assert clear_models.differ(got, ref) <= bound
    assert clear_models.differ([resid], [model[0].last_resid]) <= bound
