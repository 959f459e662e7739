"""GPU tests of a decode step's first and last launch: the tokens are the first largest logits of the rows that the engine hands out, over vocabularies
at the borders of the shared arg-max (one workgroup a row, several, a remainder, rows off the four-column grid), with every largest logit there
several times, and the sequences' lengths, tokens and records go on from step to step."""
import numpy as np
import pytest

from lmdeploy_amd.turbomind.engine import Engine
from lmdeploy_amd.turbomind.loader import export_weights
from oracle import tm_oracle as o
from tests import febivik_oracle as fo
from tests.test_gpu_febivik import engine

pytestmark = pytest.mark.gpu
PERIOD = 7     # logits of columns c and c + PERIOD are equal: ties within a vector, across threads and across workgroups


def check_steps(eng, vocab, prompts, steps):
    n = eng.cfg.max_batch_size
    eng.prefill(prompts, max_new_tokens=steps + 1)
    for s in range(steps + 1):
        lg, toks = eng.fetch_logits()[:len(prompts)], eng.fetch()
        assert toks.shape == (len(prompts), s + 1)
        want = lg[:, :vocab].argmax(1)
        assert (toks[:, s] == want).all() and (want < PERIOD).all(), (vocab, s, toks[:, s], want)
        assert (lg[:, :vocab - PERIOD] == lg[:, PERIOD:vocab]).all()
        if s < steps:
            eng.decode(1)
    batch = eng.fetch()
    eng.release()
    ids = [eng.submit(p, steps + 1) for p in prompts]          # the scheduler's step: the same tokens, slots without a sequence stay where they are
    assert len(prompts) <= n
    active = waiting = 1
    while active or waiting:
        _, active, waiting = eng.step_many(4)
    assert (np.stack([eng.poll(i)[1] for i in ids]) == batch).all()
    eng.release()


@pytest.mark.parametrize('graph', [0, 1])
@pytest.mark.parametrize('vocab', [9, 42, 8192, 8196, 8201, 16420])
def test_layer_list_steps(tmp_path, cuda, vocab, graph):
    cfg = fo.make_config(72, vocab, [fo.attention_layer(6, 2, 24, 40, 0.3, 50, 3, 16, 3000.0, 4.0, fo.dense(88))])
    w = fo.random_weights(cfg, vocab)
    w['head'] = np.asarray(w['head'])[np.arange(vocab) % PERIOD]
    folder = str(tmp_path / 'm')
    fo.write_checkpoint(folder, cfg, w)
    eng = engine(folder, 'float32', use_graph=graph)
    rng = np.random.default_rng(vocab)
    check_steps(eng, vocab, [rng.integers(0, vocab, k).astype(np.int32) for k in (5, 61, 1)], 5)
    eng.close()


@pytest.mark.parametrize('vocab, batch', [(64, 1), (8192, 3), (8256, 2), (24640, 3)])
def test_llama_steps(cuda, vocab, batch):
    cfg = o.ModelConfig(hidden=256, layers=1, q_heads=4, kv_heads=2, head_dim=128, inter=256, vocab=vocab, kv_bits=8, rope=o.RopeParam(128, 10000.0))
    w = o.make_synthetic_weights(cfg, seed=vocab)
    w['output'] = np.ascontiguousarray(w['output'][:, np.arange(vocab) % PERIOD])
    eng = Engine.from_model_config(cfg, max_batch_size=4, session_len=128, quant_policy=8, max_prefill_token_num=128)
    eng.load_weights(export_weights(cfg, w))
    eng.start()
    rng = np.random.default_rng(vocab)
    check_steps(eng, vocab, [rng.integers(0, vocab, 3 + 20 * i).astype(np.int32) for i in range(batch)], 4)
    eng.close()
