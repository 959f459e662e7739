"""Models whose logits are made by the part under test, for engine tests that would see it go wrong.  With the plain synthetic weights a layer adds a few per cent of
a rounding bound to the stream; here the experts (or the attention) outweigh everything else, and every token's router choice is far from a tie, so that a
neighbour's experts, a missing row or an unrotated key move the logits by about their own size.  Scales are powers of two: they change no other rounding."""
import contextlib

import numpy as np

from oracle import tm_oracle as o

f16, f32 = np.float16, np.float32


def _times(W, c):
    for name in ('s', 'bs', 'w'):   # (u4: the zero points count codes)
        if name in W:
            W[name] = (W[name].astype(f32) * c).astype(W[name].dtype)


def weights(cfg, seed, quantized=True, attention=False):
    """attention: queries, keys, values and the output projection are the strong part, else the feed-forward"""
    w = o.make_synthetic_weights(cfg, seed=seed, quantized=quantized)
    rng = np.random.default_rng(seed + 1)
    w['output'] = (w['output'].astype(f32) * 8).astype(f16)
    emb = w['tok_embeddings'].astype(f32)
    for L in w['layers']:
        for part in ([L['w_qkv'], L['wo']] if attention else [x[n] for x in L.get('experts', [L]) for n in ('w1w3', 'w2')]):
            _times(part, 16)
        if cfg.moe_experts:
            g = np.linalg.qr(rng.standard_normal((cfg.hidden, cfg.moe_experts)))[0].astype(f32)
            L['moe_gate'] = g.astype(f16)
            choice = np.argsort(rng.random((cfg.vocab, cfg.moe_experts)), axis=1)[:, :cfg.moe_top_k]
            share = 0.3 * (1 + 0.08 * np.arange(cfg.moe_top_k) / cfg.moe_top_k)   # clear of the experts not chosen, and none the same
            emb += np.einsum('k,vkh->vh', share, g.T[choice]).astype(f32) / np.sqrt(cfg.layers)
    w['tok_embeddings'] = emb.astype(f16)
    return w


def forced(cfg, w, prompts, toks, steps, max_ctx=128, decode=contextlib.nullcontext):
    """the oracle's logits behind the prompts and behind each of `steps` tokens of `toks`; `decode` wraps the steps (a planted mistake)"""
    m = o.OracleModel(cfg, w, batch=len(prompts), max_ctx=max_ctx)
    out = [m.forward(prompts)[1]]
    with decode():
        out += [m.forward([[int(t)] for t in toks[:, s]])[1] for s in range(steps)]
    return [x.astype(f32) for x in out]


def differ(a, b):
    """largest difference of two lists of logits, in units of the largest logit"""
    return max(np.abs(x.astype(f32) - y.astype(f32)).max() for x, y in zip(a, b)) / max(np.abs(y.astype(f32)).max() for y in b)
