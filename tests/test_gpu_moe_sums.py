"""GPU tests of the norms that sum a mixture's rows themselves, at the borders of their register variants: layer norm over the fp32 stream (with a shared expert and
without, one choice, an odd number of them, widths off the four-channel grid, where the sum is a launch of its own) inside one-layer models, and the
fp16 RMS norm at one and two vectors a thread -- against the oracles."""
import numpy as np
import pytest

from lmdeploy_amd.turbomind.engine import Engine
from lmdeploy_amd.turbomind.loader import export_weights
from oracle import tm_oracle as o
from tests import clear_models
from tests import febivik_oracle as fo
from tests.test_gpu_febivik import TOL, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('width,top,shared', [(1024, 1, 16), (1028, 3, 0), (1026, 2, 16), (2052, 3, 24), (4100, 2, 8), (8192, 2, 0)])
def test_layer_norm(tmp_path, cuda, width, top, shared):
    cfg = fo.make_config(width, 97, [fo.lightning_layer(2, 8, 8, [0.9, 0.9], fo.moe(5, top, 24, 1.3, shared))])
    w = fo.random_weights(cfg, width)
    folder = str(tmp_path / 'm')
    fo.write_checkpoint(folder, cfg, w)
    rng = np.random.default_rng(width)
    reqs = [rng.integers(0, 97, 4).tolist() for _ in range(3)]
    eng = engine(folder, 'float32')
    sess = [eng.open_session() for _ in reqs]
    got = [eng.step_tokens([(s, r[:2], [0, 1]) for s, r in zip(sess, reqs)]).reshape(3, 2, -1)]
    got += [eng.step_tokens([(s, r[i:i + 1], [0]) for s, r in zip(sess, reqs)]).reshape(3, 1, -1) for i in (2, 3)]
    ref = np.stack([fo.forward(cfg, w, r) for r in reqs])
    assert np.abs(np.concatenate(got, axis=1) - ref).max() <= TOL['float32'] * np.abs(ref).max()
    eng.close()


@pytest.mark.parametrize('hidden,top', [(256, 2), (4352, 2), (256, 3), (384, 1)])
def test_rms_norm(cuda, hidden, top):
    """two layers, every expert chosen (the second layer's choices cannot turn): the sum with weights, the stream it joins and its norm for the next layer"""
    cfg = o.ModelConfig(hidden=hidden, layers=2, q_heads=2, kv_heads=1, head_dim=128, inter=128, vocab=256, kv_bits=8, rope=o.RopeParam(128, 10000.0),
                        moe_experts=top, moe_top_k=top, weight_format='u4')
    w = clear_models.weights(cfg, hidden)
    eng = Engine.from_model_config(cfg, weight_type=0, max_batch_size=2, session_len=128, quant_policy=8, max_prefill_token_num=128)
    eng.load_weights(export_weights(cfg, w))
    eng.start()
    rng = np.random.default_rng(hidden)
    prompts = [rng.integers(0, cfg.vocab, n).astype(np.int32) for n in (9, 3)]
    eng.prefill(prompts, max_new_tokens=4)
    got = [eng.fetch_logits()]
    for _ in range(2):
        eng.decode(1)
        got.append(eng.fetch_logits())
    toks = eng.fetch()
    eng.close()
    ref = clear_models.forced(cfg, w, prompts, toks, 2)
    bound = 2.0**-7   # a dozen roundings to fp16
    ffn, pick = o.moe_ffn, o.moe_gate
    try:   # no sum; its channels moved by one; another token's rows; equal weights
        for wrong in (lambda d: 0 * d, lambda d: np.roll(d, 1, axis=1), lambda d: np.roll(d, 1, axis=0)):
            o.moe_ffn = lambda *a: (lambda d, i, t: (wrong(d), i, t))(*ffn(*a))
            assert clear_models.differ(clear_models.forced(cfg, w, prompts, toks, 2), ref) > 2 * bound
        if top > 1:
            o.moe_ffn, o.moe_gate = ffn, lambda *a: (lambda z, i, t: (z, i, 0 * t + 1 / top))(*pick(*a))
            assert clear_models.differ(clear_models.forced(cfg, w, prompts, toks, 2), ref) > 2 * bound
    finally:
        o.moe_ffn, o.moe_gate = ffn, pick
    assert clear_models.differ(got, ref) <= bound
