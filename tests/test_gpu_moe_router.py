"""GPU tests of the router's launch that also quantises its rows (fp8 experts) and, up to 64 tokens, writes the routing tables: 64 and 65 tokens, one token, 64 experts
with eight choices, expert counts off the eight-expert load, widths that leave a part of a round of 4096 channels -- engines against the oracle model."""
import numpy as np
import pytest

from lmdeploy_amd.turbomind.engine import Engine
from lmdeploy_amd.turbomind.loader import export_weights
from oracle import tm_oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('fmt,hidden,experts,top,lens', [('fp8', 256, 64, 8, (60, 4)), ('u4', 256, 64, 8, (64, )), ('fp8', 384, 5, 1, (64, 1)),
                                                         ('u4', 256, 3, 3, (1, )), ('fp8', 4352, 7, 2, (2, 9)), ('u4', 256, 8, 5, (40, 23))])
def test_engine(cuda, fmt, hidden, experts, top, lens):
    cfg = o.ModelConfig(hidden=hidden, layers=2, q_heads=2, kv_heads=1, head_dim=128, inter=128, vocab=256, kv_bits=8, rope=o.RopeParam(128, 10000.0),
                        moe_experts=experts, moe_top_k=top, weight_format=fmt, moe_fp8_act=True)
    w = o.make_synthetic_weights(cfg, seed=hidden + experts)
    eng = Engine.from_model_config(cfg, weight_type=2 if fmt == 'fp8' else 0, max_batch_size=2, session_len=128, quant_policy=8, max_prefill_token_num=128)
    eng.load_weights(export_weights(cfg, w))
    eng.start()
    rng = np.random.default_rng(hidden + top)
    prompts = [rng.integers(0, cfg.vocab, n).astype(np.int32) for n in lens]
    eng.prefill(prompts, max_new_tokens=4)
    got = [eng.fetch_logits()]
    for _ in range(2):
        eng.decode(1)
        got.append(eng.fetch_logits())
    toks = eng.fetch()
    model = o.OracleModel(cfg, w, batch=len(lens), max_ctx=128)
    ref = [model.forward(prompts)[1]] + [model.forward([[int(t)] for t in toks[:, s]])[1] for s in range(2)]
    # the bound of the engine's other mixtures: fp32 sums in another order turn single roundings of the activations
    assert max(np.abs(a.astype(np.float32)[:len(lens)] - b.astype(np.float32)).max() for a, b in zip(got, ref)) <= 3e-2
    eng.close()
