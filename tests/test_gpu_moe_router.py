"""GPU tests of the router's launch that also quantises its rows (fp8 experts) and, up to 64 tokens, writes the routing tables: 64 and 65 tokens, one token, 64 experts
with eight choices, expert counts off the eight-expert load, widths that leave a part of a round of 4096 channels -- engines whose logits the mixture makes, against
the oracle model, at a bound that a neighbour's experts, a missing choice and rows in another order are far outside of."""
import numpy as np
import pytest

from lmdeploy_amd.turbomind.engine import Engine
from lmdeploy_amd.turbomind.loader import export_weights
from oracle import tm_oracle as o
from tests import clear_models

pytestmark = pytest.mark.gpu


def planted(cfg, w, prompts, toks):
    """the oracle with a mistake in the tables: every expert's rows to its neighbour; a token's last choice left out; a token's rows from the token before it"""
    yield clear_models.forced(cfg, dict(w, layers=[dict(L, experts=L['experts'][1:] + L['experts'][:1]) for L in w['layers']]), prompts, toks, 2)
    name = 'moe_ffn_fp8' if cfg.weight_format == 'fp8' else 'moe_ffn'
    ffn = getattr(o, name)
    try:
        if cfg.moe_top_k > 1:
            setattr(o, name, lambda x, gate, ex, k, *a: ffn(x, gate, ex, k - 1, *a))
            yield clear_models.forced(cfg, w, prompts, toks, 2)
        setattr(o, name, lambda x, gate, ex, k, *a: (lambda d, i, t: (np.roll(d, 1, axis=0), i, t))(*ffn(x, gate, ex, k, *a)))
        if sum(len(p) for p in prompts) > 1:
            yield clear_models.forced(cfg, w, prompts, toks, 2)
    finally:
        setattr(o, name, ffn)


@pytest.mark.parametrize('fmt,hidden,experts,top,lens', [('fp8', 256, 64, 8, (60, 4)), ('u4', 256, 64, 8, (64, )), ('fp8', 384, 5, 1, (64, 1)),
                                                         ('u4', 256, 3, 3, (1, )), ('fp8', 4352, 7, 2, (2, 9)), ('u4', 256, 8, 5, (40, 23))])
def test_engine(cuda, fmt, hidden, experts, top, lens):
    cfg = o.ModelConfig(hidden=hidden, layers=1, q_heads=2, kv_heads=1, head_dim=128, inter=128, vocab=256, kv_bits=8, rope=o.RopeParam(128, 10000.0),
                        moe_experts=experts, moe_top_k=top, weight_format=fmt, moe_fp8_act=True)
    w = clear_models.weights(cfg, hidden + experts)
    eng = Engine.from_model_config(cfg, weight_type=2 if fmt == 'fp8' else 0, max_batch_size=2, session_len=128, quant_policy=8, max_prefill_token_num=128)
    eng.load_weights(export_weights(cfg, w))
    eng.start()
    rng = np.random.default_rng(hidden + top)
    prompts = [rng.integers(0, cfg.vocab, n).astype(np.int32) for n in lens]
    eng.prefill(prompts, max_new_tokens=4)
    got = [eng.fetch_logits()[:len(lens)]]
    for _ in range(2):
        eng.decode(1)
        got.append(eng.fetch_logits()[:len(lens)])
    toks = eng.fetch()
    eng.close()
    ref = clear_models.forced(cfg, w, prompts, toks, 2)
    # u4: half a dozen roundings to fp16.  fp8: an fp32 sum in another order turns single e4m3 codes, each an eighth of one of 128 channels: 2 - 3 % of the logits
    bound = 2.0**-4 if fmt == 'fp8' else 2.0**-7
    for wrong in planted(cfg, w, prompts, toks):
        assert clear_models.differ(wrong, ref) > 2 * bound
    assert clear_models.differ(got, ref) <= bound
