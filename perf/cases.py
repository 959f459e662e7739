"""The work that users have this framework do, as cases that can be timed and compared.

A case is one call sequence of a user's program on an engine that the program keeps: a batch of prompts through prefill and greedy decode
(`generate`), a stream of requests of mixed lengths through the scheduler (`serve`), or recorded tokens fed to sessions for their logits
(`replay`).  Models have the layer shapes of real decoders at full width and fewer layers; weights are random, fixed for a model, and drawn
so that a trained model's decisions are there: every token has a clear successor, every router a clear choice.  Prompts come from the seed.

`exact` is the same arithmetic in 64 bits, written from the models' equations on padded batches of whole sequences."""
import math

import numpy as np
import torch

from lmdeploy_amd.turbomind import layered
from lmdeploy_amd.turbomind.checkpoint import ModelConfig, RopeConfig
from lmdeploy_amd.turbomind.engine import Engine

GROUP = 128
CLEAR = 0.4       # how much of a token's embedding is in its successor's row of the head


# ---- the models ---------------------------------------------------------------------------------------------------------------------
def _febivik_json(width, heads, kv_heads, ff, layers, vocab):
    lig = {'heads': heads, 'dim': 128, 'vdim': 128, 'decay': [1.0 - 2.0 ** -(5 + 5 * h / (heads - 1)) for h in range(heads)]}
    att = {'heads': heads, 'kv_heads': kv_heads, 'dim': 128, 'vdim': 128, 'scale': 128 ** -0.5, 'mask': {'size': 2048, 'keep_first': 4},
           'rot': {'base': 10000.0, 'dims': 64, 'scaling': {'factor': 4.0}}}
    dlt = {'heads': heads, 'dim': 128, 'decay_rank': 64}
    dense = {'kind': 'dense', 'ff': ff}
    moe = {'kind': 'moe', 'expert': {'ff': ff // 3}, 'router': {'experts': 8, 'top': 2, 'scale': 1.0}, 'shared': {'ff': ff // 3}}
    four = [{'type': 'lightning', 'mixer': lig, 'mlp': dense}, {'type': 'attention', 'mixer': att, 'mlp': moe},
            {'type': 'lightning', 'mixer': lig, 'mlp': moe}, {'type': 'general_delta', 'mixer': dlt, 'mlp': moe}]
    return {'architecture': 'Febivik', 'width': width, 'vocab': vocab, 'norm': {'eps': 1e-5}, 'layers': [four[i % 4] for i in range(layers)]}


def _sanozen_json(width, heads, ff, layers, vocab):
    lat = {'heads': heads, 'dim': 64, 'rot_dim': 64, 'vdim': 128, 'kv_rank': 192, 'q_rank': width * 3 // 8, 'scale': 128 ** -0.5,
           'rot': {'base': 10000.0, 'dims': 64}}
    dense, out = {'kind': 'dense', 'ff': ff}, []
    for i in range(layers):
        if i % 4 == 2:
            out.append({'type': 'hgrn2', 'mixer': {'heads': heads, 'dim': 128, 'vdim': 128}, 'mlp': dense})
        else:
            out.append({'type': 'latent_attention', 'mixer': dict(lat, kv_from=i // 4 * 4) if i % 4 else lat, 'mlp': dense})
    return {'architecture': 'Sanozen', 'width': width, 'vocab': vocab, 'norm': {'eps': 1e-5}, 'embedding': {'scale': width ** 0.5},
            'token_side': {'dim': 256}, 'layers': out}


def _fokonex_json(width, heads, kv_heads, ff, layers, vocab):
    att = {'heads': heads, 'kv_heads': kv_heads, 'dim': 128, 'vdim': 128, 'scale': 128 ** -0.5, 'softcap': 30.0,
           'q_temp': {'coef': 0.1, 'every': 512.0}}
    return {'architecture': 'Fokonex', 'width': width, 'vocab': vocab, 'norm': {'eps': 1e-5}, 'residual_mult': 0.5, 'logit_scale': 1.0,
            'layers': [{'type': 'attention', 'mixer': att, 'mlp': {'kind': 'dense', 'ff': ff}}] * layers}


LLAMA = {   # the Llama-family decoders this framework serves, some of their layers
    'llama3_8b': dict(weights='u4', layers=8, hidden=4096, q_heads=32, kv_heads=8, inter=14336, vocab=128256, experts=0,
                      rope=RopeConfig(128, 500000.0, 'llama3', 8.0, 1.0, 4.0, 8192)),
    'internlm2_1_8b': dict(weights='f16', layers=12, hidden=2048, q_heads=16, kv_heads=8, inter=8192, vocab=92544, experts=0,
                           rope=RopeConfig(128, 1000000.0)),
    'mixtral_8x7b': dict(weights='fp8', layers=2, hidden=4096, q_heads=32, kv_heads=8, inter=14336, vocab=32000, experts=8,
                         rope=RopeConfig(128, 1000000.0)),
}
LAYERED = {   # layer-list models at the sizes `bench.py --layered` measures
    'fokonex_w4096': _fokonex_json(4096, 32, 8, 21504, 8, 32000),
    'febivik_w2048': _febivik_json(2048, 16, 8, 8448, 8, 32000),
    'sanozen_w2048': _sanozen_json(2048, 16, 8448, 8, 32000),
}


def listed():
    g = dict(kind='generate')
    return [
        # one user's short question and the first words of the answer: nothing but latency
        dict(g, name='chat_w4', model='llama3_8b', kv=8, batch=1, prompt=37, spread=0, new=16),
        # the headline: 64 sequences decoding together, W4A16 with an int8 cache
        dict(g, name='batch_w4', model='llama3_8b', kv=8, batch=64, prompt=160, spread=90, new=128),
        # documents of about a thousand tokens, time to the first token
        dict(g, name='prefill_w4', model='llama3_8b', kv=8, batch=16, prompt=1024, spread=301, new=1),
        # two long documents and an answer each, int4 cache
        dict(g, name='long_w4_kv4', model='llama3_8b', kv=4, batch=2, prompt=8000, spread=999, new=24),
        # a serving load: more requests of all lengths than batch slots, continuous batching
        dict(name='serve_w4', kind='serve', model='llama3_8b', kv=8, batch=80, prompt=200, spread=190, new=40),
        # a small unquantised model, fp16 weights and cache
        dict(g, name='batch_f16', model='internlm2_1_8b', kv=0, batch=8, prompt=333, spread=120, new=48),
        # routed experts with fp8 weights
        dict(g, name='moe_fp8', model='mixtral_8x7b', kv=8, batch=16, prompt=250, spread=77, new=32),
        # layer-list models: prompts of 2048 tokens, 8192 in a forward
        dict(g, name='prefill_fokonex', model='fokonex_w4096', dtype='bfloat16', batch=4, prompt=2048, spread=0, new=1),
        # ... a batch decoding
        dict(g, name='decode_fokonex', model='fokonex_w4096', dtype='bfloat16', batch=32, prompt=101, spread=40, new=96),
        # ... linear attention, delta rule, windowed attention and routed experts, prompts and answers
        dict(g, name='gen_febivik', model='febivik_w2048', dtype='bfloat16', batch=8, prompt=1000, spread=500, new=32),
        # ... latent attention and a forget-gate mixer, long prompts
        dict(g, name='prefill_sanozen', model='sanozen_w2048', dtype='bfloat16', batch=4, prompt=2040, spread=300, new=2),
        # ... recorded tokens through sessions in fp32, logits of every step
        dict(name='replay_sanozen_f32', kind='replay', model='sanozen_w2048', dtype='float32', batch=3, prompt=150, spread=60, new=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the listed ones' ranges, not dearer than the dearest of them."""
    def cost(c):
        w = work(c)
        return max(w['bytes'], w['flops'] / 50)
    most = max(cost(c) for c in listed())
    while True:
        model = rng.choice(sorted(LLAMA) + sorted(LAYERED))
        c = dict(kind='generate', model=model, batch=_log(rng, 1, 64))
        if model in LAYERED:
            c['kind'] = rng.choice(['generate', 'generate', 'replay'])
            c['dtype'] = 'float32' if model == 'sanozen_w2048' and c['kind'] == 'replay' else 'bfloat16'
            c['batch'] = _log(rng, 1, 32)
        else:
            c['kv'] = 0 if LLAMA[model]['weights'] == 'f16' else 8
            if model == 'llama3_8b' and rng.random() < 0.25:
                c.update(kind='serve', kv=8, batch=_log(rng, 20, 100))
        c['prompt'] = _log(rng, 9, 400 if c['kind'] != 'generate' else 8000 if model == 'llama3_8b' else 2048)
        c['spread'] = rng.randrange(0, c['prompt'] * 3 // 4)
        if model == 'llama3_8b' and c['prompt'] >= 2000 and rng.random() < 0.5:
            c['kv'] = 4       # (over a short context a code that rounding turns is seen in the logits: no tolerance would be told from a fault)
        c['new'] = rng.randint(4, 40) if c['kind'] == 'serve' else 1 if rng.random() < 0.25 else _log(rng, 2, 128 if c['kind'] == 'generate' else 16)
        if c['batch'] * (c['prompt'] + c['spread'] // 2 + c['new']) <= 20000 and cost(c) <= 0.95 * most:
            return c


# ---- weights ------------------------------------------------------------------------------------------------------------------------
def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device='cuda', dtype=torch.float32)


def _successors(vocab, gen):
    """a permutation of the vocabulary: the token that clearly follows each token"""
    return torch.randperm(vocab, generator=gen, device='cuda')


def _vocabulary(gen, vocab, width, routers, dtype):
    """(embedding, head, successors): unit-variance rows, part of a token's row in the head's row of its successor; for each router
    [experts, width] the token's two experts' directions are in its row"""
    embed = _randn(gen, vocab, width)
    for r in routers:
        e = torch.randint(0, r.shape[0], (vocab, 2), generator=gen, device='cuda')
        second = (e[:, 0] + 1 + e[:, 1] % (r.shape[0] - 1)) % r.shape[0]
        d = r.float() / r.float().norm(dim=1, keepdim=True)
        embed += 10.0 * d[e[:, 0]] + 7.0 * d[second]
    embed = embed.to(dtype)
    succ = _successors(vocab, gen)
    head = _randn(gen, vocab, width)
    head[succ] += CLEAR * embed.float()
    return embed, (head / math.sqrt(width)).to(dtype), succ


def _linear_llama(gen, kind, K, N, gain, gated=False):
    """one linear of a Llama-family checkpoint in its own format, [K][N]; gated: columns alternate (gate, up)"""
    if kind == 'u4':
        q = torch.randint(-2 ** 31, 2 ** 31, (K, N // 8), generator=gen, device='cuda', dtype=torch.int64).to(torch.int32)
        s = (gain / (4.6 * math.sqrt(K)) * (0.8 + 0.4 * torch.rand(K // GROUP, N, generator=gen, device='cuda'))).half()
        z = torch.randint(7, 9, (K // GROUP, N), generator=gen, device='cuda').half()
        return {'qweight': q, 'scales': s, 'zeros': z}
    if kind == 'fp8':
        w = (16.0 * _randn(gen, K, N)).to(torch.float8_e4m3fn).view(torch.uint8)
        s = gain / (16.0 * math.sqrt(K)) * (0.8 + 0.4 * torch.rand(K // 128, (N + 127) // 128, generator=gen, device='cuda'))
        return {'weight': w, 'scales': s}
    return {'weight': (gain / math.sqrt(K) * _randn(gen, K, N)).half()}


def _llama_layer(name, i):
    """(norms, linears, experts) of layer i; the same numbers each time it is asked for"""
    m = LLAMA[name]
    gen = torch.Generator('cuda').manual_seed(1000 + 17 * i)
    H, I, D = m['hidden'], m['inter'], 128
    out = {'attention_norm': (1 + 0.02 * _randn(gen, H)).half(), 'ffn_norm': (1 + 0.02 * _randn(gen, H)).half()}
    out['attention.w_qkv'] = _linear_llama(gen, m['weights'], H, (m['q_heads'] + 2 * m['kv_heads']) * D, 1.0)
    out['attention.wo'] = _linear_llama(gen, m['weights'], m['q_heads'] * D, H, 0.7)
    if m['experts']:
        out['moe_ffn.gate'] = {'weight': _router_llama(name, i).t().contiguous()}
        for e in range(m['experts']):
            out[f'moe_ffn.experts.{e}.w1w3'] = _linear_llama(gen, m['weights'], H, 2 * I, 1.0, True)
            out[f'moe_ffn.experts.{e}.w2'] = _linear_llama(gen, m['weights'], I, H, 0.7)
    else:
        out['feed_forward.w1w3'] = _linear_llama(gen, m['weights'], H, 2 * I, 1.0, True)
        out['feed_forward.w2'] = _linear_llama(gen, m['weights'], I, H, 0.7)
    return out


def _router_llama(name, i):
    m = LLAMA[name]
    gen = torch.Generator('cuda').manual_seed(500 + i)
    return (0.5 / math.sqrt(m['hidden']) * _randn(gen, m['experts'], m['hidden'])).half()


def _llama_vocabulary(name):
    m = LLAMA[name]
    gen = torch.Generator('cuda').manual_seed(7)
    routers = [_router_llama(name, i) for i in range(m['layers'])] if m['experts'] else []
    return (*_vocabulary(gen, m['vocab'], m['hidden'], routers, torch.float16), (1 + 0.02 * _randn(gen, m['hidden'])).half())


def _layered_config(name):
    j = LAYERED[name]
    read = layered.FAMILIES[j['architecture']]
    return read(j, {}) if j['architecture'] in layered.NEEDS_SHAPES else read(j)


def _layered_weights(name):
    """{tensor name: bf16 tensor} and the successors"""
    j, cfg = LAYERED[name], _layered_config(name)
    gen = torch.Generator('cuda').manual_seed(11)
    out, small = {}, 0.25 if j['architecture'] == 'Febivik' else 0.1
    for tensor, shape in cfg.tensor_shapes().items():
        leaf = tensor.split('.')[-1]
        if tensor in ('embed', 'head'):
            continue
        if j['architecture'] == 'Fokonex' and leaf in ('norm1', 'norm2', 'norm', 'sink'):
            a = 0.1 * _randn(gen, *shape)
        elif leaf in ('norm1', 'norm2') and j['architecture'] == 'Febivik' or tensor.endswith('side.norm'):
            a = small * (1 + 0.1 * _randn(gen, *shape))
        elif leaf in ('norm1', 'norm2', 'norm'):
            a = 1 + 0.1 * _randn(gen, *shape)
        elif leaf == 'b':
            a = (2 + _randn(gen, *shape)) if tensor.endswith('f.b') else 0.1 * _randn(gen, *shape)
        elif leaf == 'w0':
            a = _randn(gen, *shape)
        elif leaf == 'lower':
            a = 0.8 * torch.rand(*shape, generator=gen, device='cuda')
        elif leaf == 'act':
            a = torch.tensor([0.8, 0.4, -0.3, 0.1] if j['architecture'] == 'Sanozen' else [0.5, 0.5], device='cuda') + 0.05 * _randn(gen, *shape)
        elif leaf == 'dwa':
            a = 0.05 * _randn(gen, *shape)
            a[-1] += 0.9
        elif tensor == 'side.embed':
            a = _randn(gen, *shape)
        else:
            gain = 0.5 if leaf in ('o', 'down') else 1.0
            a = gain / math.sqrt(shape[-1]) * _randn(gen, *shape)
        out[tensor] = a.to(torch.bfloat16)
    embed, head, succ = _vocabulary(gen, cfg.vocab, cfg.width, [v for k, v in out.items() if k.endswith('mlp.router')], torch.float32)
    out['embed'] = (embed / cfg.embed_scale).to(torch.bfloat16)
    out['head'] = head.to(torch.bfloat16)
    return out, succ


# ---- engines: one for a model and cache type, kept as a user's program keeps it -----------------------------------------------------
_ENGINES = {}


def _llama_config(name):
    m = LLAMA[name]
    return ModelConfig(hidden=m['hidden'], layers=m['layers'], q_heads=m['q_heads'], kv_heads=m['kv_heads'], head_dim=128, inter=m['inter'],
                       vocab=m['vocab'], rms_eps=1e-5, rope=m['rope'], quantized=m['weights'] != 'f16', weight_format=m['weights'],
                       moe_experts=m['experts'], moe_top_k=2 if m['experts'] else 0)


def _llama_slots(name):
    """the checkpoint's tensors under the engine's slot names, one after the other"""
    embed, head, _, norm = _llama_vocabulary(name)
    yield 'tok_embeddings.weight', embed
    yield 'norm.weight', norm
    yield 'output.weight', head.t().contiguous()
    for i in range(LLAMA[name]['layers']):
        for k, v in _llama_layer(name, i).items():
            if isinstance(v, dict):
                for part, t in v.items():
                    yield f'layers.{i}.{k}.{part}', t
            else:
                yield f'layers.{i}.{k}.weight', v


def _engine(case):
    key = (case['model'], case.get('kv'), case.get('dtype'))
    if key not in _ENGINES:
        if case['model'] in LLAMA:
            eng = Engine.from_model_config(_llama_config(case['model']), weight_type={'u4': 0, 'f16': 1, 'fp8': 2}[LLAMA[case['model']]['weights']],
                                           max_batch_size=64, session_len=9216, quant_policy=case['kv'], cache_blocks=640)
            eng.load_weights({k: t.cpu().numpy() for k, t in _llama_slots(case['model'])})
        else:
            eng = layered.LayeredEngine(_layered_config(case['model']), dtype=case['dtype'], max_batch_size=32, session_len=4096, cache_blocks=640)
            eng.load_weights({k: t.view(torch.int16).cpu().numpy().view(np.uint16) for k, t in _layered_weights(case['model'])[0].items()})
        eng.start()
        _ENGINES[key] = eng
    return _ENGINES[key]


def _vocab(case):
    return LLAMA[case['model']]['vocab'] if case['model'] in LLAMA else LAYERED[case['model']]['vocab']


def _lengths(case):
    """prompt lengths: spread evenly around `prompt`, in a mixed order, so that a case's size does not depend on the seed"""
    n = case['batch']
    return [max(1, case['prompt'] + (case['spread'] * ((i * 7919) % n) // n - case['spread'] // 2 if n > 1 else 0)) for i in range(n)]


def _new_tokens(case):
    """tokens to generate for each request of a serving load: one to twice the mean"""
    return [1 + (case['new'] * ((i * 104729) % 97)) // 48 for i in range(case['batch'])]


def _prompts(case, seed):
    rng = np.random.default_rng(seed)
    return [rng.integers(0, _vocab(case), n).astype(np.int32) for n in _lengths(case)]


def prepare(case, seed):
    state = {'case': case, 'engine': _engine(case), 'prompts': _prompts(case, seed)}
    if case['kind'] == 'replay':
        state['steps'] = np.random.default_rng(seed + 1).integers(0, _vocab(case), (case['new'], case['batch'])).astype(np.int32)
    return state


def run(state):
    case, eng, prompts = state['case'], state['engine'], state['prompts']
    if case['kind'] == 'generate':
        eng.prefill(prompts, max_new_tokens=case['new'])
        if case['new'] > 1:
            eng.decode(case['new'] - 1)
        tokens, logits = eng.fetch(), eng.fetch_logits()
        eng.release()
        return {'tokens': tokens, 'logits': logits}
    if case['kind'] == 'serve':
        ids = [eng.submit(p, n) for p, n in zip(prompts, _new_tokens(case))]
        active = waiting = 1
        while active or waiting:
            _, active, waiting = eng.step_many(8)
        tokens = [eng.poll(i)[1] for i in ids]
        eng.release()
        return {'tokens': np.concatenate(tokens)}
    sessions = [eng.open_session() for _ in prompts]
    logits = [eng.step_tokens([(s, p, [len(p) - 1]) for s, p in zip(sessions, prompts)])]
    for row in state['steps']:
        logits.append(eng.step_tokens([(s, row[i:i + 1], [0]) for i, s in enumerate(sessions)]))
    for s in sessions:
        eng.close_session(s)
    eng.release()
    return {'logits': np.stack(logits)}


# ---- what a pass cannot do without --------------------------------------------------------------------------------------------------
def _sizes(case):
    """(bytes of all layers' weights, of them in experts, multiply-adds a token, head bytes, cache or state reads: list of
    (bytes a token of context, window, multiply-adds a token and token of context) and state bytes a sequence)"""
    if case['model'] in LLAMA:
        m = LLAMA[case['model']]
        H, A = m['hidden'], (m['q_heads'] * 2 + m['kv_heads'] * 2) * 128 * m['hidden']
        F, per = 3 * H * m['inter'], {'u4': 0.53125, 'f16': 2.0, 'fp8': 1.0}[m['weights']]
        entry = m['kv_heads'] * 2 * (128 * (case['kv'] or 16) / 8 + (4 if case['kv'] else 0))
        n = max(1, m['experts'])
        return (m['layers'] * per * (A + n * F), m['layers'] * per * n * F if m['experts'] else 0, m['layers'] * (A + F * (2 if m['experts'] else 1)),
                2.0 * H * m['vocab'], [(entry, 1 << 30, 2 * m['q_heads'] * 128)] * m['layers'], 0)
    cfg, size = _layered_config(case['model']), 2.0     # (weights arrive as bf16 in either type)
    elem = 4 if case['dtype'] == 'float32' else 2
    every = expert = mads = 0
    for k, shape in cfg.tensor_shapes().items():
        if k in ('embed', 'head', 'side.embed') or len(shape) < 2:
            continue
        n, s = math.prod(shape), cfg.layers[int(k[1:].split('.')[0])]
        every += n
        if '.mlp.e' in k:
            expert += n
            mads += n * s.top / s.experts
        else:
            mads += n
    reads, state = [], 0
    for s in cfg.layers:
        if s.mixer == layered.MIXER_ATTENTION:
            reads.append((elem * s.kv_heads * (s.dim + s.vdim), s.window + s.keep_first if s.window else 1 << 30, s.heads * (s.dim + s.vdim)))
        elif s.mixer == layered.MIXER_LATENT:
            reads.append((elem * (s.kv_rank + s.rot_dim), 1 << 30, s.heads * (s.dim + s.rot_dim + s.vdim)))
        else:
            state += s.heads * s.dim * s.vdim * 4 * 2
            mads += 2 * s.heads * s.dim * s.vdim
    return size * every, size * expert, mads, 2.0 * cfg.width * cfg.vocab, reads, state


def work(case):
    weights, expert, mads, head, reads, state = _sizes(case)
    lens, B = _lengths(case), case['batch']
    news = _new_tokens(case) if case['kind'] == 'serve' else [case['new'] - 1 if case['kind'] == 'generate' else case['new']] * B
    tokens = sum(lens) + sum(news)
    # weights: once for the prompts (a forward takes 8192 tokens) and once for each decode step, experts no more than the rows reach
    steps = max(news)
    slots = min(B, 64)
    forwards = -(-sum(lens) // 8192)
    experts = 8 if expert else 1
    reach = min(1.0, 2 * slots / experts) if expert else 1.0
    if case['kind'] == 'serve':
        steps = max(steps, -(-sum(news) // slots))
    moved = forwards * weights + steps * (weights - expert + expert * reach) + (forwards + steps) * head
    flops = 2.0 * mads * tokens + (B + sum(news)) * head
    for n, k in zip(lens, news):
        moved += state * (1 + k)
        for entry, window, m in reads:
            seen = sum(min(window, n + i) for i in range(1, k + 1))
            full = n * n / 2 if window >= n else window * (n - window / 2)
            moved += entry * (n + k + seen)
            flops += 2.0 * m * (full + seen)
    out = 2.0 * B * _vocab(case) if case['kind'] == 'generate' else 4.0 * B * (1 + case['new']) * _vocab(case) if case['kind'] == 'replay' else 0
    return {'bytes': float(moved + out), 'flops': float(flops)}


def tolerance(case):
    """`rel` / `max` about four times the most that the same path shows with its sums in another order: decode attention in three splits
    (int8 and int4 cache, fp16: 1.1e-3 ... 1.5e-3 / 8e-3; fp8, whose activations' codes then turn: 3.1e-3 / 4e-2), prompts in other portions
    (bf16: 1.4e-3 ... 2.7e-3 / 1.3e-2).  A short context makes up for fewer turned codes: 5e-3 against 64 bits for one short prompt and
    an int8 cache.  Tokens follow from clear successors and have no ties."""
    if case['kind'] == 'serve':
        return 'exact'
    if case['model'] in LLAMA:
        return {'rel': 0.02, 'max': 0.2} if LLAMA[case['model']]['weights'] == 'fp8' else {'rel': 0.01, 'max': 0.08}
    return {'rel': 1e-5, 'max': 1e-4} if case['dtype'] == 'float32' else {'rel': 0.011, 'max': 0.06}


# ---- 64 bits ------------------------------------------------------------------------------------------------------------------------
def _rms(x, eps=1e-5):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, w, b, eps=1e-5):
    d = x - x.mean(-1, keepdim=True)
    return _rms(d, eps) * w + b


def _turn(x, freq, pairs):
    """x [B, T, heads, channels]: the first 2 len(freq) channels turn by position * freq; pairs: (2i, 2i + 1), else (i, i + half)"""
    n = len(freq)
    ang = torch.arange(x.shape[1], device=x.device, dtype=torch.float64)[:, None] * freq
    c, s = ang.cos()[None, :, None], ang.sin()[None, :, None]
    u, v = (x[..., 0:2 * n:2], x[..., 1:2 * n:2]) if pairs else (x[..., :n], x[..., n:2 * n])
    a, b = u * c - v * s, v * c + u * s
    y = x.clone()
    if pairs:
        y[..., 0:2 * n:2], y[..., 1:2 * n:2] = a, b
    else:
        y[..., :n], y[..., n:2 * n] = a, b
    return y


def _frequencies(dims, base, scale=1.0):
    return base ** (-torch.arange(0, dims, 2, device='cuda', dtype=torch.float64) / dims) / scale


def _llama3_frequencies(r):
    f = _frequencies(r.dim, r.base)
    if r.type != 'llama3':
        return f
    turns = r.original_max_position_embeddings * f / (2 * math.pi)
    keep = ((turns - r.low_freq_factor) / (r.high_freq_factor - r.low_freq_factor)).clamp(0, 1)
    return keep * f + (1 - keep) * f / r.factor


def _attend(q, k, v, scale, window=0, keep=0, change=None, sink=None):
    """q [B, T, H, d], k [B, T, G, d], v [B, T, G, e] -> [B, T, H e]; change: on the scaled scores [group, T, T]; sink [H]"""
    B, T, H, _ = q.shape
    G = k.shape[2]
    i = torch.arange(T, device=q.device)
    hide = i[None, :] > i[:, None]
    if window:
        hide |= (i[:, None] - i[None, :] >= window) & (i[None, :] >= keep)
    out = torch.empty(B, T, H, v.shape[3], device=q.device, dtype=torch.float64)
    for b in range(B):
        for g in range(G):
            hs = slice(g * (H // G), (g + 1) * (H // G))
            s = torch.matmul(q[b, :, hs].permute(1, 0, 2), k[b, :, g].t().contiguous()) * scale
            s = s if change is None else change(s)
            s.masked_fill_(hide, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[hs, None, None].expand(-1, T, 1)], -1)
            p = torch.softmax(s, -1)[..., :T]
            out[b, :, hs] = torch.matmul(p, v[b, :, g].contiguous()).permute(1, 0, 2)
    return out.reshape(B, T, -1)


def _cached(x, bits):
    """keys or values as a quantised cache holds them: codes between a head's smallest and largest channel"""
    if not bits:
        return x
    lo, hi = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    s = (hi - lo) / (2 ** bits - 1)
    return torch.round((x - lo) / s) * s + lo


def _wide(lin, halves=False):
    """a linear's weights in 64 bits, [K][N]"""
    if 'qweight' in lin:
        q = lin['qweight'].to(torch.int64)
        q = torch.stack([(q >> (4 * j)) & 15 for j in range(8)], -1).reshape(q.shape[0], -1).double()
        rep = q.shape[0] // lin['scales'].shape[0]
        return (q - lin['zeros'].double().repeat_interleave(rep, 0)) * lin['scales'].double().repeat_interleave(rep, 0)
    w = lin['weight']
    if 'scales' not in lin:
        return w.double()
    w, s = w.view(torch.float8_e4m3fn).float().double(), lin['scales'].double().repeat_interleave(128, 0)
    if not halves:
        return w * s.repeat_interleave(128, 1)[:, :w.shape[1]]
    n = s.shape[1] // 2      # gate and up were quantised apart: their columns alternate, their block scales do not
    return w * torch.stack([s[:, :n].repeat_interleave(128, 1), s[:, n:].repeat_interleave(128, 1)], -1).reshape(w.shape)


def _gated(h, w13, w2):
    z = h @ _wide(w13, 'scales' in w13 and 'weight' in w13)
    return (torch.nn.functional.silu(z[..., 0::2]) * z[..., 1::2]) @ _wide(w2)


def _llama_exact(case, ids, last):
    name, m = case['model'], LLAMA[case['model']]
    embed, head, _, norm = _llama_vocabulary(name)
    x, freq = embed[ids].double(), _llama3_frequencies(m['rope'])
    B, T = ids.shape
    Hq, Hk = m['q_heads'], m['kv_heads']
    for i in range(m['layers']):
        L = _llama_layer(name, i)
        h = _rms(x) * L['attention_norm'].double()
        q, k, v = (h @ _wide(L['attention.w_qkv'])).split([Hq * 128, Hk * 128, Hk * 128], -1)
        q, k = _turn(q.reshape(B, T, Hq, 128), freq, True), _turn(k.reshape(B, T, Hk, 128), freq, True)
        x = x + _attend(q, _cached(k, case['kv']), _cached(v.reshape(B, T, Hk, 128), case['kv']), 128 ** -0.5) @ _wide(L['attention.wo'])
        h = _rms(x) * L['ffn_norm'].double()
        if m['experts']:
            h = h.reshape(B * T, -1)
            score, pick = (h @ L['moe_ffn.gate']['weight'].double()).topk(2, -1)
            score, y = torch.softmax(score, -1), torch.zeros_like(h)
            for e in range(m['experts']):
                t, j = (pick == e).nonzero(as_tuple=True)
                y[t] += score[t, j, None] * _gated(h[t], L[f'moe_ffn.experts.{e}.w1w3'], L[f'moe_ffn.experts.{e}.w2'])
            x = x + y.reshape(x.shape)
        else:
            x = x + _gated(h, L['feed_forward.w1w3'], L['feed_forward.w2'])
    x = _rms(x[torch.arange(B, device=x.device)[:, None], last]) * norm.double()
    return x @ head.double().t()


def _recur(T, start, step):
    """outputs [B, T, ...] of a recurrence: state, output = step(t, state)"""
    out = []
    for t in range(T):
        start, o = step(t, start)
        out.append(o)
    return torch.stack(out, 1)


def _febivik_mixer(x, L, w):
    m, (B, T, _) = L['mixer'], x.shape
    H, D = m['heads'], m['dim']
    if L['type'] == 'attention':
        G = m['kv_heads']
        q, k, v = (((x @ w(s).t()) + w(s + '.b')).reshape(B, T, -1, D) for s in 'qkv')
        f = _frequencies(m['rot']['dims'], m['rot']['base'], m['rot']['scaling']['factor'])
        q, k = _turn(_rms(q) * w('q.norm'), f, False), _turn(_rms(k) * w('k.norm'), f, False)
        assert k.shape[2] == G
        return _attend(q, k, v, m['scale'], m['mask']['size'], m['mask']['keep_first']) @ w('o').t()
    S = torch.zeros(B, H, D, D, device=x.device, dtype=torch.float64)
    if L['type'] == 'lightning':
        q, k, v = (torch.nn.functional.silu(x @ w(s).t()).reshape(B, T, H, D) for s in 'qkv')
        d = torch.tensor(m['decay'], device=x.device, dtype=torch.float64)[:, None, None]

        def step(t, S):
            S = torch.addcmul(d * S, k[:, t, :, :, None], v[:, t, :, None, :])
            return S, torch.matmul(q[:, t, :, None, :], S)[:, :, 0]
        o = _rms(_recur(T, S, step).reshape(B, T, -1))
    else:
        r, k, v = ((x @ w(s).t()).reshape(B, T, H, D) for s in 'rkv')
        d = torch.exp(-math.exp(-0.5) * torch.sigmoid(torch.tanh(x @ w('w1').t()) @ w('w2').t() + w('w0'))).reshape(B, T, H, D)
        a = torch.sigmoid(x @ w('a').t() + w('a.b')).reshape(B, T, H, D)
        u = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
        a = a * u

        def step(t, S):
            away = torch.matmul(u[:, t, :, None, :], S)
            S = torch.addcmul(d[:, t, :, :, None] * S, k[:, t, :, :, None], v[:, t, :, None, :]) - a[:, t, :, :, None] * away
            return S, torch.matmul(r[:, t, :, None, :], S)[:, :, 0]
        o = _rms(_recur(T, S, step)).reshape(B, T, -1)
    return (o * w('norm') * torch.sigmoid(x @ w('g').t())) @ w('o').t()


def _febivik_ff(x, f, w):
    if f['kind'] == 'dense':
        z, (p, q) = x @ w('up').t(), torch.nn.functional.softplus(w('act'))
        return torch.where(z > 0, p * z * z, (0.5 + q) * (torch.expm1(z.clamp(max=0)) - z)).add(0.5 * z) @ w('down').t()

    def expert(h, e):
        return torch.relu(h @ w(e + '.up').t()).square() @ w(e + '.down').t()
    h = x.reshape(-1, x.shape[-1])
    score, pick = torch.softmax(h @ w('router').t(), -1).topk(f['router']['top'], -1)
    y = expert(h, 'shared')
    for e in range(f['router']['experts']):
        t, j = (pick == e).nonzero(as_tuple=True)
        y[t] += f['router']['scale'] * score[t, j, None] * expert(h[t], f'e{e}')
    return y.reshape(x.shape)


def _sanozen_mixer(h, L, w, entries, i):
    m, (B, T, _) = L['mixer'], h.shape
    H, D = m['heads'], m['dim']
    if L['type'] == 'hgrn2':
        q = torch.nn.functional.silu(h @ w('q').t()).reshape(B, T, H, D)
        f = (w('lower') + (1 - w('lower')) * torch.sigmoid(h @ w('f').t() + w('f.b'))).reshape(B, T, H, D)
        v = (h @ w('v').t()).reshape(B, T, H, -1)

        def step(t, S):
            S = torch.addcmul(f[:, t, :, :, None] * S, 1 - f[:, t, :, :, None], v[:, t, :, None, :])
            return S, torch.matmul(q[:, t, :, None, :], S)[:, :, 0]
        S = torch.zeros(B, H, D, v.shape[-1], device=h.device, dtype=torch.float64)
        return (_rms(_recur(T, S, step)) * w('norm')).reshape(B, T, -1) @ w('o').t()
    C, freq = m['kv_rank'], _frequencies(m['rot']['dims'], m['rot']['base'])
    if m.get('kv_from') is None:
        c, r = (h @ w('dkv').t()).split([C, m['rot_dim']], -1)
        entries[i] = _rms(c) * w('dkv.norm'), _turn(r[:, :, None], freq, True)
    c, r = entries[m.get('kv_from', i)]
    q = ((_rms(h @ w('dq').t()) * w('dq.norm')) @ w('uq').t()).reshape(B, T, H, -1)
    q = torch.cat([q[..., :D], _turn(q[..., D:], freq, True)], -1)
    k = torch.cat([(c @ w('uk').t()).reshape(B, T, H, D), r.expand(-1, -1, H, -1)], -1)
    return _attend(q, k, (c @ w('uv').t()).reshape(B, T, H, -1), m['scale']) @ w('o').t()


def _layered_exact(case, ids, last):
    j, (w, _) = LAYERED[case['model']], _layered_weights(case['model'])
    wide = {}

    def of(prefix):      # a layer's tensors in 64 bits, as they are asked for
        return lambda leaf: wide.setdefault(prefix + leaf, w[prefix + leaf].double())
    top = of('')
    x = w['embed'][ids].double() * (j.get('embedding') or {}).get('scale', 1.0)
    arch, depth, entries = j['architecture'], [x], {}
    for i, L in enumerate(j['layers']):
        own, mix, ff = of(f'l{i}.'), of(f'l{i}.mix.'), of(f'l{i}.mlp.')
        if arch == 'Fokonex':
            m, (B, T, _) = L['mixer'], x.shape
            h = _rms(x) * (1 + own('norm1'))
            q, k, v = ((h @ mix(s).t()).reshape(B, T, -1, 128) for s in 'qkv')
            at = torch.arange(T, device=x.device, dtype=torch.float64)
            q = q * (1 + m['q_temp']['coef'] * torch.log(torch.floor((at + 1) / m['q_temp']['every']) + 1))[None, :, None, None]
            y = _attend(q, k, v, m['scale'], change=lambda s: m['softcap'] * torch.tanh(s / m['softcap']), sink=mix('sink')) @ mix('o').t()
            z = torch.relu((_rms(x) * (1 + own('norm2'))) @ ff('up').t()).square() @ ff('down').t()
            x = x + j['residual_mult'] * (y + z)
        elif arch == 'Febivik':
            x = x + _layer_norm(_febivik_mixer(x, L, mix), own('norm1'), own('norm1.b'))
            x = x + _layer_norm(_febivik_ff(x, L['mlp'], ff), own('norm2'), own('norm2.b'))
        else:
            x = x + _sanozen_mixer(_layer_norm(x, own('norm1'), own('norm1.b')), L, mix, entries, i)
            z, (a, b, c, e) = _layer_norm(x, own('norm2'), own('norm2.b')) @ ff('up').t(), ff('act')
            x = x + (a * _rms(z) + b * _rms(z ** 2) + c * _rms(z ** 3) + e) @ ff('down').t()
            n = j['token_side']['dim']
            g = torch.nn.functional.gelu(x @ own('side.gate').t(), approximate='tanh') * w['side.embed'][ids][..., i * n:(i + 1) * n].double()
            x = x + _rms(g @ own('side.proj').t()) * own('side.norm')
            depth.append(x)
            x = sum(a * X for a, X in zip(own('dwa'), depth))
        wide.clear()
    x = x[torch.arange(len(ids), device=x.device)[:, None], last]
    x = _rms(x) * (1 + top('final.norm')) if arch == 'Fokonex' else _layer_norm(x, top('final.norm'), top('final.norm.b'))
    return x @ top('head').t()


def exact(case, seed):
    """logits of the places that run() returns logits of; tokens are whole numbers"""
    if case['kind'] == 'serve':
        return None
    prompts, B = _prompts(case, seed), case['batch']
    if case['kind'] == 'replay':
        steps = np.random.default_rng(seed + 1).integers(0, _vocab(case), (case['new'], B)).astype(np.int32)
        seqs = [np.concatenate([p, steps[:, i]]) for i, p in enumerate(prompts)]
        last = [[len(p) - 1 + k for k in range(case['new'] + 1)] for p in prompts]
    else:
        succ = (_llama_vocabulary(case['model'])[2] if case['model'] in LLAMA else _layered_weights(case['model'])[1]).cpu().numpy()
        seqs = []
        for p in prompts:
            p = list(p)
            for _ in range(case['new'] - 1):
                p.append(succ[p[-1]])
            seqs.append(np.asarray(p))
        last = [[len(s) - 1] for s in seqs]
    ids = torch.zeros(B, max(len(s) for s in seqs), dtype=torch.long, device='cuda')
    for i, s in enumerate(seqs):
        ids[i, :len(s)] = torch.from_numpy(np.asarray(s, np.int64))
    logits = (_llama_exact if case['model'] in LLAMA else _layered_exact)(case, ids, torch.tensor(last, device='cuda'))
    if case['kind'] == 'replay':
        return {'logits': logits.transpose(0, 1).contiguous()}
    return {'tokens': None, 'logits': logits[:, 0]}
