"""GPU test of engines after the start-up tuning, whose timed chains run the engine's own launches -- the mixture's tables by its router's last workgroup and its sum
in the norm behind it, the greedy choice over several workgroups, the fp16 [q | k | v] product that rotates and stores: counters, cache and stream are as before it,
so the same prompts give the oracle's logits, and the same bits a second time."""
import numpy as np
import pytest

from lmdeploy_amd.turbomind.engine import Engine
from lmdeploy_amd.turbomind.loader import export_weights
from oracle import tm_oracle as o
from tests import clear_models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('fmt,experts,kv_bits', [('fp8', 4, 8), ('u4', 5, 8), ('f16', 0, 16)])
def test_tuned(cuda, tmp_path, fmt, experts, kv_bits):
    cfg = o.ModelConfig(hidden=256, layers=2, q_heads=4, kv_heads=2, head_dim=128, inter=256, vocab=20000, kv_bits=kv_bits, rope=o.RopeParam(128, 10000.0),
                        moe_experts=experts, moe_top_k=2, moe_fp8_act=True, **({} if fmt == 'f16' else {'weight_format': fmt}))
    w = clear_models.weights(cfg, 7, quantized=fmt != 'f16', attention=fmt == 'f16')
    eng = Engine.from_model_config(cfg, weight_type={'u4': 0, 'f16': 1, 'fp8': 2}[fmt], max_batch_size=3, session_len=128, quant_policy=0 if kv_bits == 16 else kv_bits,
                                   max_prefill_token_num=128)
    eng.load_weights(export_weights(cfg, w))
    eng.start()
    for M in (3, 70):
        eng.tune_gemm(M, str(tmp_path / 'table.txt'))
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, cfg.vocab, n).astype(np.int32) for n in (40, 9, 21)]
    runs = []
    for _ in range(2):
        eng.prefill(prompts, max_new_tokens=4)
        lg = [eng.fetch_logits()]
        for _ in range(2):
            eng.decode(1)
            lg.append(eng.fetch_logits())
        runs.append((eng.fetch(), lg))
        eng.release()
    eng.close()
    toks, lg = runs[0]
    assert np.array_equal(toks, runs[1][0]) and all(np.array_equal(a.view(np.uint16), b.view(np.uint16)) for a, b in zip(lg, runs[1][1]))
    assert all(np.array_equal(np.argmax(a.astype(np.float32), axis=1), toks[:, s]) for s, a in enumerate(lg))
    # fp16: half a dozen roundings a layer.  fp8: an fp32 sum in another order turns single e4m3 codes, each an eighth of one of 256 channels of a row (2 % of the
    # row's length with the activations' spread, 5 % for a few of them in two layers); another expert or a missing row: 100 %
    assert clear_models.differ(lg, clear_models.forced(cfg, w, prompts, toks, 2)) <= (2.0**-3 if fmt == 'fp8' else 2.0**-7)


@pytest.mark.parametrize('quantized,batch', [(True, 2), (False, 2), (False, 12)])
def test_pairs_are_timed_as_they_run(cuda, tmp_path, capfd, monkeypatch, quantized, batch):
    """products that a decode step runs without a norm launch between them are timed so by the tuner: the choice that an untuned engine would make is measured with the norm in its
    product, others with the norm between the products, and what a tuned engine computes stays within the bound"""
    hidden = 3584 if quantized else 1536
    cfg = o.ModelConfig(hidden=hidden, layers=2, q_heads=16, kv_heads=2, head_dim=128, inter=2304, vocab=256, kv_bits=8 if quantized else 16, rope=o.RopeParam(128, 10000.0))
    w = clear_models.weights(cfg, 3, quantized=quantized)
    eng = Engine.from_model_config(cfg, weight_type=0 if quantized else 1, max_batch_size=batch, session_len=64, quant_policy=cfg.kv_bits % 16, max_prefill_token_num=256)
    eng.load_weights(export_weights(cfg, w))
    eng.start()
    monkeypatch.setenv('TM_GEMM_TUNE_VERBOSE', '1')
    eng.tune_gemm(batch, str(tmp_path / 'table.txt'))
    lines = [x for x in capfd.readouterr().err.splitlines() if f'M={batch} ' in x and '->' not in x]
    for role in ('w_qkv', 'wo ', 'w1w3', 'w2 '):
        own = [x for x in lines if x.startswith(f'[tm tune] {role}')]
        assert any('<- heuristic' in x and '(norm in its product)' in x for x in own), (role, own)
        assert any('(norm between products)' in x for x in own), (role, own)
    rng = np.random.default_rng(3)
    prompts = [rng.integers(0, cfg.vocab, 2 + i % 3).astype(np.int32) for i in range(batch)]
    eng.prefill(prompts, max_new_tokens=4)
    lg = [eng.fetch_logits()]
    for _ in range(2):
        eng.decode(1)
        lg.append(eng.fetch_logits())
    toks = eng.fetch()
    eng.close()
    assert clear_models.differ(lg, clear_models.forced(cfg, w, prompts, toks, 2)) <= 2.0**-6    # (as in the tests of these products)
