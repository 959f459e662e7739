"""GPU test of the fp16 [q | k | v] product that rotates and stores a decode step's keys and values itself: rows on both sides of its row tiles, the narrow kernel, the
weight stream with 64 and 96 columns a workgroup, in one slice of k and in several that meet in the launch, one more row than it takes, positions at the start and
across a cache block's border -- engines whose logits the attention makes, against the oracle's unfused sequence."""
import contextlib

import numpy as np
import pytest

from lmdeploy_amd.turbomind.engine import Engine
from lmdeploy_amd.turbomind.loader import export_weights
from oracle import tm_oracle as o
from tests import clear_models
from tests.test_host import stream_plan

pytestmark = pytest.mark.gpu


@contextlib.contextmanager
def _instead(**kw):
    old = {n: getattr(o, n) for n in kw}
    try:
        for n, f in kw.items():
            setattr(o, n, f)
        yield
    finally:
        for n, f in old.items():
            setattr(o, n, f)


def _mistakes():
    """what a decode step could do wrong: keys unrotated, queries and keys unrotated, values not stored, keys and values in each other's place, a place too early"""
    store, turn = o.process_kv, o.rope_apply
    yield dict(process_kv=lambda c, b, l, k, v, cos, sin, t: store(c, b, l, k, v, None, None, t))
    yield dict(rope_apply=lambda x, cos, sin: x, process_kv=lambda c, b, l, k, v, cos, sin, t: store(c, b, l, k, v, None, None, t))
    yield dict(process_kv=lambda c, b, l, k, v, cos, sin, t: store(c, b, l, k, 0 * v, cos, sin, t))
    yield dict(process_kv=lambda c, b, l, k, v, cos, sin, t: store(c, b, l, v, turn(k, cos, sin), None, None, t))
    yield dict(process_kv=lambda c, b, l, k, v, cos, sin, t: store(c, b, l, k, v, cos, sin, t - 1))


# plan: (kernel, column tiles a workgroup, row tiles, slices of k), None where the product keeps its own launch for the store
@pytest.mark.parametrize('hidden,heads,kv_heads,batch,plan', [
    (256, 2, 1, 1, (1, 1, 1, 1)), (256, 4, 2, 17, (1, 1, 2, 1)), (256, 2, 1, 33, (1, 1, 4, 1)), (256, 2, 2, 64, (1, 1, 4, 1)), (256, 2, 1, 65, None),
    (4096, 32, 8, 3, (1, 1, 1, 1)), (4096, 32, 8, 24, (2, 4, 2, 2)), (4096, 32, 8, 48, (2, 6, 4, 4)), (2048, 64, 16, 8, (2, 4, 1, 1)), (1024, 128, 16, 5, (2, 6, 1, 1))])
def test_decode(cuda, hidden, heads, kv_heads, batch, plan):
    p = stream_plan(2, hidden, (heads + 2 * kv_heads) * 128, batch)
    assert p[:4] == plan if plan else p[0] > 2
    cfg = o.ModelConfig(hidden=hidden, layers=2 if hidden == 256 else 1, q_heads=heads, kv_heads=kv_heads, head_dim=128, inter=256, vocab=256, kv_bits=16,
                        rope=o.RopeParam(128, 10000.0))
    w = clear_models.weights(cfg, batch, quantized=False, attention=True)
    eng = Engine.from_model_config(cfg, weight_type=1, max_batch_size=batch, session_len=128, quant_policy=0, max_prefill_token_num=4608)
    eng.load_weights(export_weights(cfg, w))
    eng.start()
    rng = np.random.default_rng(batch)
    prompts = [rng.integers(0, cfg.vocab, 61 + i // 8 % 5 if i % 8 == 1 else 2 + i % 3).astype(np.int32) for i in range(batch)]
    eng.prefill(prompts, max_new_tokens=5)
    got = [eng.fetch_logits()]
    for _ in range(3):
        eng.decode(1)
        got.append(eng.fetch_logits())
    toks = eng.fetch()
    eng.close()
    ref = clear_models.forced(cfg, w, prompts, toks, 3)
    bound = 2.0**-6    # half a dozen roundings to fp16 a layer, those of queries and keys under a soft-max of scores of about ten
    for m in _mistakes():
        assert clear_models.differ(clear_models.forced(cfg, w, prompts, toks, 3, decode=lambda: _instead(**m)), ref) > 2 * bound
    assert clear_models.differ(got, ref) <= bound
