"""The work that programs give this framework, as cases that can be timed.

Every case goes through the public entry points: the W8A16 and W8A8 linears,
the decode experts module, the routed experts of a prefill chunk, the router,
the fused MoE layer, and the resident stack (decode step, chunked prefill).
Inputs and weights are drawn on the GPU from the seed alone; weights are
quantized here in plain torch (symmetric absmax, 128-wide K groups), so
`exact` can restate every result in 64 bits without the package.
"""
import math

import numpy as np
import torch

H, I, E, TOP, G = 2048, 512, 256, 8, 128
EPS = 1e-6
DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.float16}

# Shapes [N, K] of dense linears: the projections of a hidden-2048 model whose
# mixers are 4096 wide, the shared expert's three matrices, and one whose N
# is no multiple of any tile.
LINEARS = [(4096, 2048), (2048, 4096), (8192, 2048), (1024, 2048), (512, 2048), (2048, 512),
           (1000, 2048)]
LM_HEAD = (248320, 2048)


def listed():
    return [
        # one projection of one decode step: the smallest dense call
        dict(name='linear_1', kind='linear', m=1, n=4096, k=2048, dtype='bf16'),
        # the same projection for a batch of users or a short prompt
        dict(name='linear_45', kind='linear', m=45, n=4096, k=2048, dtype='bf16'),
        # an output projection (K = 4096) on a medium prompt, in fp16
        dict(name='linear_333_fp16', kind='linear', m=333, n=2048, k=4096, dtype='fp16'),
        # a projection of a whole prefill chunk
        dict(name='linear_2048', kind='linear', m=2048, n=4096, k=2048, dtype='bf16'),
        # the shared expert's fused gate_up + SwiGLU with W8A8, four sequences
        dict(name='w8a8_4', kind='w8a8', m=4, n=1024, k=2048, swiglu=True, dtype='bf16'),
        # W8A8 linear of a medium prompt: quantization and the int8 GEMM
        dict(name='w8a8_700', kind='w8a8', m=700, n=4096, k=2048, swiglu=False, dtype='bf16'),
        # the experts module swapped into a model, one decode token
        dict(name='experts_decode', kind='experts', experts=256, top=8, dtype='bf16'),
        # the routed experts of a prefill chunk with skewed popularity
        dict(name='routed_2048_zipf', kind='routed', tokens=2048, skew=True, dtype='bf16'),
        # the router of a prefill chunk
        dict(name='router_2048', kind='router', tokens=2048, skew=False),
        # one fused layer on a small batch of decoding sequences
        dict(name='layer_24', kind='layer', tokens=24, skew=False),
        # one decode step of a stack, replayed as a graph as a serving loop does
        dict(name='decode_stack', kind='decode', layers=4, skew=False),
        # a 4096-token prompt through a stack, two overlapped chunks
        dict(name='prefill_stack', kind='prefill', tokens=4096, layers=4, skew=False),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(['linear', 'linear', 'w8a8', 'experts', 'routed', 'router', 'layer', 'layer',
                       'decode', 'prefill'])
    dtype = rng.choice(['bf16', 'bf16', 'fp16'])
    skew = rng.random() < 0.4
    if kind == 'linear':
        if rng.random() < 0.12:
            n, k = LM_HEAD
            return dict(kind=kind, m=rng.randint(1, 4), n=n, k=k, dtype=dtype)
        n, k = rng.choice(LINEARS)
        return dict(kind=kind, m=_log_int(rng, 1, 2048), n=n, k=k, dtype=dtype)
    if kind == 'w8a8':
        n, k = rng.choice(LINEARS)
        return dict(kind=kind, m=_log_int(rng, 1, 2048), n=n, k=k, swiglu=rng.random() < 0.5,
                    dtype=dtype)
    if kind == 'experts':
        return dict(kind=kind, experts=rng.randint(32, 256), top=rng.randint(2, 12), dtype=dtype)
    if kind == 'routed':
        return dict(kind=kind, tokens=_log_int(rng, 2, 2048), skew=skew, dtype=dtype)
    if kind == 'router':
        return dict(kind=kind, tokens=_log_int(rng, 1, 2048), skew=skew)
    if kind == 'layer':
        return dict(kind=kind, tokens=_log_int(rng, 2, 2048), skew=skew)
    if kind == 'decode':
        return dict(kind=kind, layers=rng.randint(2, 5), skew=skew)
    return dict(kind=kind, tokens=_log_int(rng, 256, 4096), layers=rng.randint(1, 4), skew=skew)


# ------------------------------------------------------------------ inputs
def _gen(case, seed):
    g = torch.Generator(device='cuda')
    g.manual_seed((seed * 1_000_003 + sum(map(ord, case['kind'])) * 7919) % (2 ** 62))
    return g


def _weights(gen, q, s):
    """Fills q int8 [..., N, K] and s fp32 [..., N, K/128] with quantized N(0, 0.02)."""
    q2, s2 = q.view(-1, q.shape[-1]), s.view(-1, s.shape[-1])
    step = max(1, (1 << 26) // q.shape[-1])
    for r in range(0, q2.shape[0], step):
        part = q2[r:r + step]
        w = torch.randn(part.shape[0], part.shape[1] // G, G, generator=gen, device='cuda') * 0.02
        sc = (w.abs().amax(-1) / 127.0).clamp_min(1e-30)
        part.copy_((w / sc[..., None]).round_().clamp_(-127, 127).view(part.shape))
        s2[r:r + step] = sc


def _bank(gen, e, n, k):
    q = torch.empty((e, n, k), dtype=torch.int8, device='cuda')
    s = torch.empty((e, n, k // G), dtype=torch.float32, device='cuda')
    _weights(gen, q, s)
    return q, s


def _zipf(s=1.1, seed=3):
    """Per-expert logit offset that skews popularity like Zipf(s), fp32 [E]."""
    ranks = np.random.default_rng(seed).permutation(E) + 1
    logp = -s * np.log(ranks.astype(np.float64))
    return (logp - logp.mean()).astype(np.float32)


def _bias(case):
    return torch.from_numpy(_zipf()) if case['skew'] else None


def _route(gen, tokens, skew, experts=E, top_k=TOP):
    """Routing of a chunk as a router hands it over: ids int64 and bf16 weights [T, top_k]."""
    logits = torch.randn(tokens, experts, generator=gen, device='cuda') * 0.9
    if skew:
        logits = logits + torch.from_numpy(_zipf()).to('cuda')
    top, ids = torch.topk(torch.softmax(logits, -1), top_k, dim=-1)
    return ids.contiguous(), (top / top.sum(-1, keepdim=True)).to(torch.bfloat16)


def _rows(gen, m, k, dtype):
    return torch.randn(m, k, generator=gen, device='cuda').to(DTYPES[dtype])


def _dense_inputs(case, seed):
    gen = _gen(case, seed)
    x = _rows(gen, case['m'], case['k'], case['dtype'])
    q, s = _bank(gen, 1, case['n'], case['k'])
    return x, q[0], s[0]


def _experts_inputs(case, seed):
    gen = _gen(case, seed)
    tokens = case.get('tokens', 1)
    x = _rows(gen, tokens, H, case['dtype'])
    e = case.get('experts', E)
    ids, w = _route(gen, tokens, case.get('skew', False), e, case.get('top', TOP))
    return (x, ids, w.to(DTYPES[case['dtype']])) + _bank(gen, e, 2 * I, H) + _bank(gen, e, H, I)


def _router_inputs(case, seed):
    gen = _gen(case, seed)
    x = _rows(gen, case['tokens'], H, 'bf16')
    w = (torch.randn(E, H, generator=gen, device='cuda') * 0.02).to(torch.bfloat16)
    bias = _bias(case)
    return x, w, None if bias is None else bias.to('cuda')


def _layers_of(case):
    return case.get('layers', 1)


def _tokens_of(case):
    return case.get('tokens', 1)


def _stack_weights(case, seed):
    """(x, list of per-layer dicts) of the fused layer: bank of E routed experts and the shared one."""
    gen = _gen(case, seed)
    x = _rows(gen, _tokens_of(case), H, 'bf16')
    layers = []
    for _ in range(_layers_of(case)):
        gu_q, gu_s = _bank(gen, E + 1, 2 * I, H)
        dn_q, dn_s = _bank(gen, E + 1, H, I)
        layers.append(dict(
            gu_q=gu_q, gu_s=gu_s, dn_q=dn_q, dn_s=dn_s,
            router_w=(torch.randn(E, H, generator=gen, device='cuda') * 0.02).to(torch.bfloat16),
            gate_w=(torch.randn(H, generator=gen, device='cuda') * 0.02).to(torch.bfloat16),
            norm_w=torch.randn(H, generator=gen, device='cuda') * 0.1))
    return x, layers


def _stack(case, seed):
    from localmoe35ba3b_amd.runtime.stack import MoEStack
    x, layers = _stack_weights(case, seed)
    # a program sizes the workspace for its chunk, and builds the tile copies
    # only where it prefills
    stack = MoEStack(len(layers), max_tokens=min(2048, x.shape[0]), router_bias=_bias(case),
                     norm=True)
    for l, w in enumerate(layers):
        for name in ('gu_q', 'gu_s', 'dn_q', 'dn_s', 'router_w', 'gate_w', 'norm_w'):
            getattr(stack, name)[l] = w[name]
        w.clear()
    if x.shape[0] > 1:
        stack.build_prefill_tiles()
    return stack, x


def prepare(case, seed):
    kind = case['kind']
    if kind == 'linear':
        from localmoe35ba3b_amd.operators.int8 import Int8Linear
        x, q, s = _dense_inputs(case, seed)
        return dict(kind=kind, x=x, module=Int8Linear(q, s))
    if kind == 'w8a8':
        x, q, s = _dense_inputs(case, seed)
        return dict(kind=kind, x=x, q=q, s=s, swiglu=case['swiglu'])
    if kind == 'experts':
        from localmoe35ba3b_amd.operators.int8 import Int8Experts
        x, ids, w, gq, gs, dq, ds = _experts_inputs(case, seed)
        module = Int8Experts(0, {'q': gq, 'scale': gs}, {'q': dq, 'scale': ds})
        return dict(kind=kind, x=x, ids=ids, w=w, module=module)
    if kind == 'routed':
        x, ids, w, gq, gs, dq, ds = _experts_inputs(case, seed)
        return dict(kind=kind, x=x, ids=ids, w=w, banks=[gq, gs, dq, ds])
    if kind == 'router':
        x, w, bias = _router_inputs(case, seed)
        return dict(kind=kind, x=x, w=w, bias=bias)
    stack, x = _stack(case, seed)
    state = dict(kind=kind, stack=stack, x=x)
    if kind == 'layer':
        state['ids'] = torch.empty((x.shape[0], TOP), dtype=torch.int32, device='cuda')
        state['weights'] = torch.empty((x.shape[0], TOP), dtype=torch.bfloat16, device='cuda')
    if kind == 'decode':
        # the decode step of a serving loop: captured once, replayed per token
        h = x.clone()
        stack.forward(h)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            stack.forward(h)
        state.update(h=h, graph=graph)
    return state


def run(state):
    kind = state['kind']
    if kind == 'linear':
        return state['module'](state['x'])
    if kind == 'w8a8':
        from localmoe35ba3b_amd.operators import w8a8
        return w8a8.linear(state['x'], state['q'], state['s'], state['swiglu'])
    if kind == 'experts':
        return state['module'](state['x'], state['ids'], state['w'])
    if kind == 'routed':
        from localmoe35ba3b_amd.runtime import gpu_routes
        return gpu_routes.routed_moe(state['x'], state['w'], state['ids'], state['banks'])
    if kind == 'router':
        from localmoe35ba3b_amd import router
        return router.router_topk(state['x'], state['w'], TOP, state['bias'])
    if kind == 'layer':
        h = state['x'].clone()
        state['stack'].layer_forward(h, 0, state['ids'], state['weights'])
        return h, state['ids'], state['weights']
    if kind == 'decode':
        state['h'].copy_(state['x'])
        state['graph'].replay()
        return state['h']
    return state['stack'].prefill(state['x'])


# ------------------------------------------------------------------ work
def _active(tokens, skew):
    """Experts that a chunk of this kind activates (a typical chunk's count)."""
    g = np.random.default_rng(11)
    logits = g.standard_normal((tokens, E)) * 0.9 + (_zipf() if skew else 0.0)
    return int(np.unique(np.argpartition(-logits, TOP - 1, axis=1)[:, :TOP]).size)


def _matrix_bytes(n, k):
    return n * k + n * (k // G) * 4


def work(case):
    kind = case['kind']
    if kind in ('linear', 'w8a8'):
        m, n, k = case['m'], case['n'], case['k']
        out = n // 2 if case.get('swiglu') else n
        return dict(bytes=_matrix_bytes(n, k) + 2 * m * (k + out), flops=2 * m * n * k)
    expert = _matrix_bytes(2 * I, H) + _matrix_bytes(H, I)
    expert_flops = 2 * (2 * I * H + H * I)
    t = _tokens_of(case)
    if kind == 'router':
        return dict(bytes=2 * (t + E) * H + t * (4 * E + 10 * TOP), flops=2 * t * E * H)
    if kind == 'experts':
        return dict(bytes=case['top'] * (expert + 10) + 4 * H, flops=case['top'] * expert_flops)
    if kind == 'routed':
        return dict(bytes=_active(t, case['skew']) * expert + 4 * t * H + 10 * t * TOP,
                    flops=t * TOP * expert_flops)
    layers = _layers_of(case)
    per_layer = (_active(t, case['skew']) + 1) * expert + 2 * (E + 1) * H + 4 * H
    return dict(bytes=layers * per_layer + 4 * t * H,
                flops=layers * t * ((TOP + 1) * expert_flops + 2 * E * H))


# ------------------------------------------------------------------ 64-bit results
def tolerance(case):
    """About four times the distance from the 64-bit result that the formats give."""
    kind = case['kind']
    # 16-bit results of 32-bit sums; the dequantized weights are rounded to 16 bits on the way
    if kind == 'linear':
        return dict(rel=1e-2, max=0.04) if case['dtype'] == 'bf16' else dict(rel=1.2e-3, max=6e-3)
    # 16-bit results of exact integer sums; SwiGLU rounds three times
    if kind == 'w8a8':
        return dict(rel=1.5e-2, max=0.06)
    # SwiGLU and down rows are rounded to 16 bits, and so is every step of the combine
    if kind in ('experts', 'routed'):
        return dict(rel=2.5e-2, max=0.15)
    # logits are bf16 values; ids may differ only at ties of the rounded logits
    if kind == 'router':
        return dict(rel=6.6e-3, max=0.016, differ=1e-3)
    if kind == 'layer':
        return dict(rel=8e-3, max=0.04, differ=1e-3)
    # a rounded residual moves a later layer's logits by a bf16 step, which can swap the last of
    # the selected experts of a token
    return dict(rel=0.03, max=0.8)


def _deq(q, s):
    return (q.double().view(*s.shape, G) * s.double()[..., None]).view(q.shape)


def _quant(x):
    """Per-row, per-128-group int8 quantization: the values the int8 product sees."""
    v = x.double().view(x.shape[0], -1, G)
    s = v.abs().amax(-1, keepdim=True).clamp_min(1e-10) / 127.0
    return (torch.round(v / s) * s).view(x.shape)


def _silu(v):
    return v * torch.sigmoid(v)


def _swiglu(gu):
    half = gu.shape[-1] // 2
    return _silu(gu[:, :half]) * gu[:, half:]


def _expert(x, gq, gs, dq, ds, quant=False):
    xin = _quant(x) if quant else x.double()
    h = _swiglu(xin @ _deq(gq, gs).t())
    return (_quant(h) if quant else h) @ _deq(dq, ds).t()


def _routed(x, ids, w, gq, gs, dq, ds, quant=False):
    y = torch.zeros(x.shape[0], H, dtype=torch.float64, device=x.device)
    for e in torch.unique(ids).tolist():
        tok, slot = torch.where(ids == e)
        y.index_add_(0, tok, _expert(x[tok], gq[e], gs[e], dq[e], ds[e], quant)
                     * w[tok, slot].double()[:, None])
    return y


def _router(x, w, bias):
    """The selection is defined on logits rounded to bf16 (then biased), ties to the smaller id."""
    logits = (x.double() @ w.double().t()).to(torch.float32).to(torch.bfloat16).float()
    if bias is not None:
        logits = logits + bias
    lg = logits.double()
    ids = torch.sort(lg, dim=-1, descending=True, stable=True).indices[:, :TOP]
    p = torch.softmax(lg, -1).gather(1, ids)
    return lg, p / p.sum(-1, keepdim=True), ids


def _layer(h, w, bias):
    """One block on h [T, H] in 64 bits.  The router sees the normalized row as the bf16 value it is
    defined on; one token runs its routed experts W8A8, several W8A16."""
    xn = h / torch.sqrt((h * h).mean(-1, keepdim=True) + EPS) * (1.0 + w['norm_w'].double())
    xr = xn.to(torch.float32).to(torch.bfloat16)
    _, p, ids = _router(xr, w['router_w'], bias)
    x = xr.double()
    one = h.shape[0] == 1
    bank = (w['gu_q'], w['gu_s'], w['dn_q'], w['dn_s'])
    y = _routed(x, ids, p, *bank, quant=one)
    shared = _expert(x, *(t[E] for t in bank))
    gate = torch.sigmoid(x @ w['gate_w'].double())[:, None]
    return h + y + gate * shared, ids, p


def exact(case, seed):
    kind = case['kind']
    if kind == 'linear':
        x, q, s = _dense_inputs(case, seed)
        return torch.cat([x.double() @ _deq(q[r:r + 8192], s[r:r + 8192]).t()
                          for r in range(0, q.shape[0], 8192)], dim=-1)
    if kind == 'w8a8':
        x, q, s = _dense_inputs(case, seed)
        y = _quant(x) @ _deq(q, s).t()
        return _swiglu(y) if case['swiglu'] else y
    if kind in ('experts', 'routed'):
        return _routed(*_experts_inputs(case, seed))
    if kind == 'router':
        return _router(*_router_inputs(case, seed))
    x, layers = _stack_weights(case, seed)
    bias = _bias(case)
    bias = None if bias is None else bias.to('cuda')
    h = x.double()
    for w in layers:
        h, ids, p = _layer(h, w, bias)
    return (h, ids.to(torch.int32), p) if kind == 'layer' else h
