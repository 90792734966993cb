"""The work this framework is used for, as cases that can be timed and checked.

A case is one call (or one replay) that a program decoding or serving an int8 Qwen3-shaped model makes:

  linear     `efficientgpt::int8_linear` over `rows` activation rows. 1 row is a decode step's projection, 2-16 rows
             a small batch or a speculative check, more a prompt pass (the op's prefill formula).
  attention  `decode_attention` of one query per batch row over a cache: GQA with the Qwen3 heads in bf16, and the
             multi-head forms in fp16 and fp32.
  quantize   `quantize_weight` of a weight that is on the device (what quantize_model does to each linear).
  step       one decode step of `Qwen3Int8Engine`, the replay of its captured graph at a given position.
  prefill    `Qwen3Int8Engine.prefill` of a prompt, from an empty cache or continuing a filled one.

`step` and `prefill` run a few layers at a model's full widths: each further layer repeats the same launches, and
rounding differences travel through every layer that follows. Their weights are seeded int8 codes and scales in the
engine's packed layout, so a state is made without any of the repository's kernels.
"""

import math

import torch

from efficientgpt_amd.decode_attention import decode_attention
from efficientgpt_amd.int8_linear import int8_linear, quantize_weight
from efficientgpt_amd.qwen3 import Qwen3Config, Qwen3Int8Engine

DEV = 'cuda'
DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.float16, 'fp32': torch.float32}
ELEM = {'bf16': 2, 'fp16': 2, 'fp32': 4}

# widths the repository's configurations, tests and benchmark run
MODELS = {
    '1.7b': dict(vocab=151936, hidden=2048, inter=6144, heads=16, kv_heads=8, head_dim=128, tied=True),
    '8b': dict(vocab=151936, hidden=4096, inter=12288, heads=32, kv_heads=8, head_dim=128, tied=False),
    'tiny': dict(vocab=512, hidden=128, inter=256, heads=4, kv_heads=2, head_dim=32, tied=True),
}
# (K, N) of the linears of those models, and the benchmark's held-out shapes
LINEARS = ((2048, 4096), (2048, 2048), (2048, 12288), (6144, 2048), (4096, 6144), (4096, 4096), (4096, 24576),
           (12288, 4096), (2048, 6144), (2048, 1024), (2048, 151936))
# (query heads, kv heads, head dim)
HEADS = ((16, 8, 128), (32, 8, 128), (6, 6, 64), (8, 1, 64), (4, 2, 32), (8, 8, 128))


def listed():
    return [
        # one token's up projection through the op, the smallest linear call
        dict(name='linear 1 row', kind='linear', rows=1, k=2048, n=6144),
        # the down projection of a batch of 8
        dict(name='linear 8 rows', kind='linear', rows=8, k=6144, n=2048),
        # the gate / up product of a short prompt of odd length
        dict(name='linear 77 rows', kind='linear', rows=77, k=2048, n=12288),
        # the QKV product of a prompt of ordinary length, no multiple of a tile
        dict(name='linear 1000 rows', kind='linear', rows=1000, k=4096, n=6144),
        # the gate / up product of the long-context benchmark's prompt, the largest linear
        dict(name='linear 8192 rows', kind='linear', rows=8192, k=4096, n=24576),
        # attention of one token over a long cache
        dict(name='attention 32 / 8 long', kind='attention', dtype='bf16', batch=1, hq=32, hkv=8, d=128, cap=32768,
             live=30011),
        # a batch of short sequences at positions of their own, multi-head fp16
        dict(name='attention batch fp16', kind='attention', dtype='fp16', batch=24, hq=6, hkv=6, d=64, cap=1024,
             live=0),
        # the largest weight that loading a model quantises
        dict(name='quantize head', kind='quantize', dtype='bf16', n=151936, k=2048),
        # a decode step early in a conversation
        dict(name='step 1.7b', kind='step', model='1.7b', layers=4, pos=300, cap=512),
        # a decode step after a long prompt
        dict(name='step 8b long', kind='step', model='8b', layers=2, pos=8192, cap=8704),
        # the benchmark's prompt
        dict(name='prefill 1.7b short', kind='prefill', model='1.7b', layers=4, rows=128, pos0=0, cap=512),
        # a long prompt, no multiple of a tile
        dict(name='prefill 8b long', kind='prefill', model='8b', layers=2, rows=6001, pos0=0, cap=8192),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(('linear', 'linear', 'linear', 'attention', 'attention', 'quantize', 'step', 'prefill', 'prefill'))
    if kind == 'linear':
        rows = _log_int(rng, 1, 8192)
        if rng.random() < 0.2:  # widths of no model above, odd ones among them
            k, n = _log_int(rng, 64, 8192), _log_int(rng, 64, 8192)
            if rng.random() < 0.7:
                k = -(-k // 64) * 64
            else:
                rows = min(rows, 512)
        else:
            k, n = rng.choice(LINEARS)
            if n > 65536:  # the head runs on the rows whose logits are wanted
                rows = min(rows, 64)
        return dict(kind='linear', rows=rows, k=k, n=n)
    if kind == 'attention':
        hq, hkv, d = rng.choice(HEADS)
        dtype = rng.choice(('bf16', 'bf16', 'fp16', 'fp32'))
        cap = _log_int(rng, 16, 32768)
        most = (1 << 29) // (2 * cap * hkv * d * ELEM[dtype])  # 512 MiB of keys and values
        batch = _log_int(rng, 1, max(1, min(64, most)))
        live = 0 if batch > 1 else rng.randint(max(1, cap // 2), cap)
        return dict(kind='attention', dtype=dtype, batch=batch, hq=hq, hkv=hkv, d=d, cap=cap, live=live)
    if kind == 'quantize':
        k, n = rng.choice(LINEARS) if rng.random() < 0.7 else (_log_int(rng, 64, 8192), _log_int(rng, 64, 16384))
        return dict(kind='quantize', dtype=rng.choice(('bf16', 'bf16', 'fp16', 'fp32')), n=n, k=k)
    model = rng.choice(('1.7b', '1.7b', '8b', '8b', 'tiny'))
    layers = {'1.7b': 4, '8b': 2, 'tiny': 2}[model]
    if kind == 'step':
        pos = _log_int(rng, 1, 16384)
        return dict(kind='step', model=model, layers=layers, pos=pos, cap=pos + rng.randint(1, 512))
    rows = _log_int(rng, 2, 6000)
    pos0 = 0 if rng.random() < 0.7 else rng.randint(1, 2000)
    return dict(kind='prefill', model=model, layers=layers, rows=rows, pos0=pos0, cap=rows + pos0 + rng.randint(1, 512))


# ------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _codes(g, n, k, std=0.02):
    """Int8 codes and fp32 scales of an [n, k] weight N(0, std): a row of k such values has its largest near 3.5 std."""
    step = torch.rand(n, generator=g, device=DEV) * 0.2 + 0.9
    step = step * (3.5 * std / 127)
    q = torch.empty(n, k, dtype=torch.int8, device=DEV)
    for lo in range(0, n, 16384):
        hi = min(n, lo + 16384)
        w = torch.randn(hi - lo, k, generator=g, device=DEV) * std
        q[lo:hi] = torch.round(w / step[lo:hi, None]).clamp_(-127, 127).to(torch.int8)
    return q, step


def _linear_inputs(c, seed):
    g = _gen(seed)
    x = torch.randn(c['rows'], c['k'], generator=g, device=DEV).to(torch.bfloat16)
    q, s = _codes(g, c['n'], c['k'])
    return x, q, s


def _attention_inputs(c, seed):
    g = _gen(seed)
    dt = DTYPES[c['dtype']]
    b = c['batch']
    q = torch.randn(b, c['hq'], 1, c['d'], generator=g, device=DEV).to(dt)
    k = torch.randn(b, c['hkv'], c['cap'], c['d'], generator=g, device=DEV).to(dt)
    v = torch.randn(b, c['hkv'], c['cap'], c['d'], generator=g, device=DEV).to(dt)
    if c['live']:
        pos = torch.full((1,), c['live'] - 1, dtype=torch.long, device=DEV)
    else:
        pos = torch.randint(0, c['cap'], (b,), generator=g, device=DEV)
    return q, k, v, pos


def _quantize_input(c, seed):
    g = _gen(seed)
    w = torch.empty(c['n'], c['k'], dtype=DTYPES[c['dtype']], device=DEV)
    for lo in range(0, c['n'], 16384):
        hi = min(c['n'], lo + 16384)
        w[lo:hi] = torch.randn(hi - lo, c['k'], generator=g, device=DEV) * 0.02
    return w


def _config(c):
    m = MODELS[c['model']]
    return Qwen3Config(vocab=m['vocab'], hidden=m['hidden'], inter=m['inter'], layers=c['layers'], heads=m['heads'],
                       kv_heads=m['kv_heads'], head_dim=m['head_dim'], tied=m['tied'])


def _model_inputs(c, seed):
    """The packed weights, the cache before the call ([layers, Hkv, filled, D] keys and values) and the token ids."""
    m, g = MODELS[c['model']], _gen(seed)
    h, d, inter = m['hidden'], m['head_dim'], m['inter']

    def norm(n):
        return (1 + 0.1 * torch.randn(n, generator=g, device=DEV)).to(torch.bfloat16)

    layers = []
    for _ in range(c['layers']):
        L = {}
        for key, n, k in (('qkv', (m['heads'] + 2 * m['kv_heads']) * d, h), ('o', h, m['heads'] * d),
                          ('gu', 2 * inter, h), ('down', h, inter)):
            L[key + '_q'], L[key + '_s'] = _codes(g, n, k)
        for key, n in (('in_w', h), ('post_w', h), ('qn_w', d), ('kn_w', d)):
            L[key] = norm(n)
        layers.append(L)
    hq, hs = _codes(g, m['vocab'], h)
    # a tied head is an int8 copy of the embedding; an untied one its own
    if m['tied']:
        embed = torch.empty(m['vocab'], h, dtype=torch.bfloat16, device=DEV)
        for lo in range(0, m['vocab'], 16384):
            embed[lo:lo + 16384] = hq[lo:lo + 16384].float() * hs[lo:lo + 16384, None]
    else:
        embed = (torch.randn(m['vocab'], h, generator=g, device=DEV) * 0.02).to(torch.bfloat16)
    packed = {'layers': layers, 'embed': embed, 'norm_w': norm(h), 'head_q': hq, 'head_s': hs}
    filled = c['pos'] if c['kind'] == 'step' else c['pos0']
    rows = 1 if c['kind'] == 'step' else c['rows']
    # keys after the norm and RoPE have unit-variance elements, values those of a projection of normed rows
    kc = torch.randn(c['layers'], m['kv_heads'], filled, d, generator=g, device=DEV).to(torch.bfloat16)
    vc = torch.randn(c['layers'], m['kv_heads'], filled, d, generator=g, device=DEV).to(torch.bfloat16)
    ids = torch.randint(0, m['vocab'], (rows,), generator=g, device=DEV)
    return packed, kc, vc, ids


class _Step:
    """An engine with its step captured, the token to decode and its position."""

    def __init__(self, c, seed):
        packed, kc, vc, ids = _model_inputs(c, seed)
        self.eng = Qwen3Int8Engine(_config(c), packed, c['cap'], device=DEV, packed=True)
        self.eng.k_cache[:, :, :c['pos']] = kc
        self.eng.v_cache[:, :, :c['pos']] = vc
        self.pos = torch.full((1,), c['pos'], dtype=torch.long, device=DEV)
        self.ids = ids
        self.eng.token.copy_(ids)
        self.eng.position.copy_(self.pos)
        self.eng.capture()
        self.k_new = self.eng.k_cache[:, :, c['pos']]
        self.v_new = self.eng.v_cache[:, :, c['pos']]

    def run(self):
        self.eng.token.copy_(self.ids)
        self.eng.position.copy_(self.pos)
        self.eng.replay()
        return {'logits': self.eng.logits, 'k': self.k_new, 'v': self.v_new}


class _Prefill:
    """An engine and a prompt; with pos0 > 0 the cache holds that many earlier tokens."""

    def __init__(self, c, seed):
        packed, kc, vc, ids = _model_inputs(c, seed)
        self.eng = Qwen3Int8Engine(_config(c), packed, c['cap'], device=DEV, packed=True)
        self.pos0, end = c['pos0'], c['pos0'] + c['rows']
        if self.pos0:
            self.eng.k_cache[:, :, :self.pos0] = kc
            self.eng.v_cache[:, :, :self.pos0] = vc
        self.ids = ids
        self.k_new = self.eng.k_cache[:, :, self.pos0:end]
        self.v_new = self.eng.v_cache[:, :, self.pos0:end]

    def run(self):
        logits = self.eng.prefill(self.ids, self.pos0)
        return {'logits': logits, 'k': self.k_new, 'v': self.v_new}


def prepare(case, seed):
    kind = case['kind']
    if kind == 'linear':
        x, q, s = _linear_inputs(case, seed)
        return lambda: int8_linear(x, q, s)
    if kind == 'attention':
        q, k, v, pos = _attention_inputs(case, seed)
        return lambda: decode_attention(q, k, v, pos)
    if kind == 'quantize':
        w = _quantize_input(case, seed)
        return lambda: quantize_weight(w)
    if kind == 'step':
        return _Step(case, seed).run
    return _Prefill(case, seed).run


def run(state):
    return state()


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    c = case
    if c['kind'] == 'linear':
        m, n, k = c['rows'], c['n'], c['k']
        return {'bytes': n * k + 4 * n + 2 * m * k + 2 * m * n, 'flops': 2 * m * n * k}
    if c['kind'] == 'attention':
        live = c['live'] or (c['cap'] + 1) / 2  # positions of their own: uniform over the cache
        kv = 2 * c['batch'] * c['hkv'] * live * c['d'] * ELEM[c['dtype']]
        return {'bytes': kv + 2 * c['batch'] * c['hq'] * c['d'] * ELEM[c['dtype']],
                'flops': 4 * c['batch'] * c['hq'] * live * c['d']}
    if c['kind'] == 'quantize':
        return {'bytes': c['n'] * c['k'] * (ELEM[c['dtype']] + 1) + 4 * c['n'], 'flops': 3 * c['n'] * c['k']}
    m = MODELS[c['model']]
    h, d, inter, hq, hkv = m['hidden'], m['head_dim'], m['inter'], m['heads'], m['kv_heads']
    per_layer = (hq + 2 * hkv) * d * h + h * hq * d + 3 * inter * h
    rows, past = (1, c['pos']) if c['kind'] == 'step' else (c['rows'], c['pos0'])
    weights = c['layers'] * per_layer + m['vocab'] * h
    kv = c['layers'] * hkv * d * 2 * 2 * (past + 2 * rows)  # what came before, and the new rows in and out
    pairs = rows * past + rows * (rows + 1) / 2
    return {'bytes': weights + kv + rows * h * 2 + 2 * m['vocab'],
            'flops': 2 * rows * c['layers'] * per_layer + 2 * m['vocab'] * h + 4 * c['layers'] * hq * d * pairs}


# What the data types give, about four times the error against 64 bits that was measured: a decode linear or an
# attention row is rounded to bf16 once (1.7e-3) and a prompt linear twice (2.3e-3), an fp16 row once (2.1e-4), fp32
# rows differ by the order of their sums (8e-8 to a few 1e-7). Through a few layers every rounding travels on: the
# logits are 0.7e-2 to 2e-2 from their 64-bit value.
def tolerance(case):
    kind = case['kind']
    if kind == 'quantize':
        return 'exact'
    if kind == 'linear':
        return {'rel': 8e-3, 'max': 0.03}
    if kind == 'attention':
        return {'bf16': {'rel': 8e-3, 'max': 0.03}, 'fp16': {'rel': 1e-3, 'max': 4e-3},
                'fp32': {'rel': 1e-5, 'max': 1e-4}}[case['dtype']]
    return {'rel': 0.03, 'max': 0.3}


# ------------------------------------------------------------------ the same in 64 bits


def _mm(x, q, s):
    """x [rows, k] fp64 times the weight q * s, in blocks of rows of q that bound the fp64 copy."""
    out = torch.empty(x.shape[0], q.shape[0], dtype=torch.float64, device=x.device)
    for lo in range(0, q.shape[0], 8192):
        hi = min(q.shape[0], lo + 8192)
        out[:, lo:hi] = (x @ q[lo:hi].double().t()) * s[lo:hi].double()
    return out


def _attend(q, k, v, pos0):
    """Causal attention of q [rows, D] at positions pos0.. over k, v [slots, D], all fp64."""
    out = torch.empty_like(q)
    slots = torch.arange(k.shape[0], device=q.device)
    for lo in range(0, q.shape[0], 2048):
        hi = min(q.shape[0], lo + 2048)
        s = (q[lo:hi] @ k.t()) * q.shape[1] ** -0.5
        s.masked_fill_(slots[None, :] > pos0 + torch.arange(lo, hi, device=q.device)[:, None], -math.inf)
        out[lo:hi] = torch.softmax(s, dim=-1) @ v
    return out


def _rms(x, w, eps=1e-6):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _model_exact(c, seed):
    m = MODELS[c['model']]
    packed, kc, vc, ids = _model_inputs(c, seed)
    d, hq, hkv = m['head_dim'], m['heads'], m['kv_heads']
    pos0, rows = kc.shape[2], ids.numel()
    # the model's RoPE tables are bf16
    inv = 1.0 / (1e6 ** (torch.arange(0, d, 2, dtype=torch.float) / d))
    ang = torch.arange(pos0, pos0 + rows, dtype=torch.float)[:, None] * inv
    ang = torch.cat((ang, ang), dim=-1)
    cos, sin = ang.cos().to(torch.bfloat16).to(DEV).double(), ang.sin().to(torch.bfloat16).to(DEV).double()

    def rope(t):
        return t * cos + torch.cat((-t[:, d // 2:], t[:, :d // 2]), dim=-1) * sin

    x = packed['embed'][ids].double()
    ks, vs = [], []
    for i, L in enumerate(packed['layers']):
        qkv = _mm(_rms(x, L['in_w']), L['qkv_q'], L['qkv_s'])
        out = torch.empty(rows, hq * d, dtype=torch.float64, device=DEV)
        kl, vl = [], []
        for j in range(hkv):
            kn = rope(_rms(qkv[:, (hq + j) * d:(hq + j + 1) * d], L['kn_w']))
            vn = qkv[:, (hq + hkv + j) * d:(hq + hkv + j + 1) * d]
            kl.append(kn)
            vl.append(vn)
            keys, values = torch.cat((kc[i, j].double(), kn)), torch.cat((vc[i, j].double(), vn))
            for a in range(j * (hq // hkv), (j + 1) * (hq // hkv)):
                qn = rope(_rms(qkv[:, a * d:(a + 1) * d], L['qn_w']))
                out[:, a * d:(a + 1) * d] = _attend(qn, keys, values, pos0)
        ks.append(torch.stack(kl))
        vs.append(torch.stack(vl))
        x = x + _mm(out, L['o_q'], L['o_s'])
        gu = _mm(_rms(x, L['post_w']), L['gu_q'], L['gu_s'])
        act = torch.nn.functional.silu(gu[:, :m['inter']]) * gu[:, m['inter']:]
        x = x + _mm(act, L['down_q'], L['down_s'])
    logits = _mm(_rms(x[-1:], packed['norm_w']), packed['head_q'], packed['head_s'])
    k, v = torch.stack(ks), torch.stack(vs)
    if c['kind'] == 'step':
        return {'logits': logits, 'k': k[:, :, 0], 'v': v[:, :, 0]}
    return {'logits': logits[0], 'k': k, 'v': v}


def exact(case, seed):
    c = case
    if c['kind'] == 'linear':
        x, q, s = _linear_inputs(c, seed)
        return _mm(x.double(), q, s)
    if c['kind'] == 'attention':
        q, k, v, pos = _attention_inputs(c, seed)
        out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
        group = c['hq'] // c['hkv']
        for b in range(c['batch']):
            live = int(pos[b if pos.numel() > 1 else 0]) + 1
            for j in range(c['hkv']):
                qs = q[b, j * group:(j + 1) * group, 0].double()
                s = (qs @ k[b, j, :live].double().t()) * c['d'] ** -0.5
                out[b, j * group:(j + 1) * group, 0] = torch.softmax(s, dim=-1) @ v[b, j, :live].double()
        return out
    if c['kind'] == 'quantize':
        w = _quantize_input(c, seed)
        step = torch.cat([w[lo:lo + 16384].double().abs().amax(1) for lo in range(0, c['n'], 16384)]) / 127
        return None, step.clamp_min(1e-12)
    return _model_exact(c, seed)
