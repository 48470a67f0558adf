"""The work whose speed this repository answers for, as a program that uses it calls it.

Four kinds of case:

  linear    one `QuantizedLinear` call (or `lowbit_hip.linear` where a rank-r correction goes with it): a
            module inside somebody's own model, called eagerly.
  block     the seven projections of a decoder block (q, k, v, o, gate, up, down) on prepared calls, with the
            output head where `vocab` is set.  Up to 32 rows they are one HIP graph, as a decode loop
            captures them; more rows (prefill) are launched one by one.  Every projection has its own
            activations: what lies between two of them is the program's.
  prefill   `FrozenSmolStack.prefill` of a prompt and the logits of its last position.
  decode    `FrozenSmolStack.decode` of a few tokens from a prefill snapshot, each followed by the
            logits.  Every pass goes on from the same snapshot, as several continuations of one prompt do.
  generate  `GraphDecoder`: a prefill snapshot is loaded, then whole tokens are replayed from a HIP graph.

Shapes: SmolLM-135M (576 / 192 / 1536, 30 layers, vocabulary 49152), SmolLM-360M's MLP (960 / 2560),
Llama-3-8B (4096 / 1024 / 14336), and generic ones between them.  Weights are N(0, 0.02) and quantized as
`quantize_weight` does it, activations N(0, 1).
"""
import sys
from pathlib import Path

import numpy as np
import torch

PACKAGE = str(Path(__file__).resolve().parents[1] / 'torch-intel-npu_amd')
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

import lowbit_hip  # noqa: E402
from torch_npu_lowbit import PackedWeight, QuantizedLinear  # noqa: E402
from torch_npu_lowbit_correction import LowRankCorrection  # noqa: E402
from torch_npu_smollm import FrozenSmolLayer, FrozenSmolStack, GraphDecoder  # noqa: E402
from torch_npu_smollm_io import FrozenSmolIO  # noqa: E402

CODEBOOK = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635,
            -0.18477343022823334, -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725,
            0.24611230194568634, 0.33791524171829224, 0.44070982933044434, 0.5626170039176941,
            0.7229568362236023, 1.0)
LIMIT = {'int4': 7, 'nf4': 1, 'int8': 127}
HIDDEN, KV, INTER, VOCAB, HEADS, KV_HEADS, HEAD_DIM = 576, 192, 1536, 49152, 9, 3, 64
SMOL = {'self_attn.q_proj.weight': (HIDDEN, HIDDEN), 'self_attn.k_proj.weight': (KV, HIDDEN),
        'self_attn.v_proj.weight': (KV, HIDDEN), 'self_attn.o_proj.weight': (HIDDEN, HIDDEN),
        'mlp.gate_proj.weight': (INTER, HIDDEN), 'mlp.up_proj.weight': (INTER, HIDDEN),
        'mlp.down_proj.weight': (HIDDEN, INTER)}
NORMS = ('input_layernorm.weight', 'post_attention_layernorm.weight')
MODE = {'int8': 'w8a16', 'int4': 'w4a16', 'nf4': 'nf4a16', 'fp16': 'fp16'}


# ---------------------------------------------------------------- cases
def _linear(name, format, m, n, k, group, bias=False, rank=0, grid=0.0, compact=False):
    return dict(name=name, kind='linear', format=format, m=m, n=n, k=k, group=group, bias=bias, rank=rank,
                grid=grid, compact=compact)


def _block(name, format, m, hidden, kv, inter, group, inter_group, blocks, vocab=0):
    return dict(name=name, kind='block', format=format, m=m, hidden=hidden, kv=kv, inter=inter, group=group,
                inter_group=inter_group, blocks=blocks, vocab=vocab)


def _smol(name, kind, format, rank, layers, batch, length, steps=0):
    return dict(name=name, kind=kind, format=format, rank=rank, layers=layers, batch=batch, length=length, steps=steps)


def listed():
    return [
        # The smallest call: one projection of a small model for one token, an ordinary module call.
        _linear('module int4 576x576 m1', 'int4', 1, 576, 576, 32),
        # W8A8, the option with an activation grid, at the size the reference times it at.
        _linear('module w8a8 1024x1024 m512', 'int8', 512, 1024, 1024, 1024, grid=2.0 ** -5),
        # An odd number of rows through a 360M model's up projection with a bias: a ragged prompt.
        _linear('module nf4 2560x960 m333', 'nf4', 333, 2560, 960, 64, bias=True),
        # Decoding one sequence with an 8B model: weights come from HBM once a token.
        _block('graph int4 8b m1', 'int4', 1, 4096, 1024, 14336, 128, 128, 2),
        # Four sequences decoded with a 135M model: launches of a few microseconds, and the head.
        _block('graph int4 135m m4', 'int4', 4, HIDDEN, KV, INTER, 64, 128, 30, VOCAB),
        # A small batch, NF4: the codebook's decode.
        _block('graph nf4 8b m8', 'nf4', 8, 4096, 1024, 14336, 128, 128, 2),
        # A larger batch, per-row INT8.
        _block('graph int8 8b m24', 'int8', 24, 4096, 1024, 14336, 4096, 14336, 1),
        # A long prompt through an 8B block: the matrix cores.
        _block('prefill int4 8b m1024', 'int4', 1024, 4096, 1024, 14336, 128, 128, 1),
        # A prompt of odd length through a 360M model's blocks.
        _block('prefill nf4 360m m500', 'nf4', 500, 960, 320, 2560, 64, 64, 4),
        # The whole SmolLM-135M with corrections: a prompt, eager tokens after it, replayed tokens.
        _smol('smol prefill int8 r32', 'prefill', 'int8', 32, 30, 1, 256),
        _smol('smol decode int8 r32', 'decode', 'int8', 32, 30, 1, 256, 4),
        _smol('smol generate int8 r32', 'generate', 'int8', 32, 30, 1, 256, 16),
    ]


def _between(rng, low, high):
    """A whole number of [low, high], spread over its logarithm."""
    return min(high, max(low, int(round(low * (high / low) ** rng.random()))))


def draw(rng):
    kind = rng.choice(('linear', 'linear', 'graph', 'graph', 'launched', 'smol'))
    format = rng.choice(('int4', 'int4', 'nf4', 'int8'))
    if kind == 'linear':
        group = rng.choice((32, 64, 128))
        k = group * _between(rng, max(1, 256 // group), 8192 // group)
        n = _between(rng, 64, 8192)
        m = 1 if rng.random() < 0.3 else _between(rng, 1, 1024)
        option = rng.random()
        if format == 'int8':
            return _drop(_linear('', 'int8', m, n, k, k, rank=rng.choice((8, 32)) if option < 0.3 else 0,
                                 grid=2.0 ** -5 if 0.3 <= option < 0.6 else 0.0, bias=option >= 0.8))
        return _drop(_linear('', format, m, n, k, group, bias=option < 0.3, compact=option > 0.9 and k // group <= 32))
    if kind in ('graph', 'launched'):
        hidden, kv, inter = rng.choice(((HIDDEN, KV, INTER), (960, 320, 2560), (2048, 512, 8192), (3072, 1024, 8192),
                                        (4096, 1024, 14336)))
        group = hidden if format == 'int8' else 32 if hidden == HIDDEN else rng.choice((32, 64))
        inter_group = inter if format == 'int8' else group
        if format != 'int8' and hidden >= 2048:
            group = inter_group = rng.choice((64, 128, 128))
        m = _between(rng, 1, 32) if kind == 'graph' else _between(rng, 33, 768)
        small = hidden < 2048
        blocks = rng.randint(4, 24) if small and kind == 'graph' else rng.randint(1, 4) if small else 1
        return _drop(_block('', format, m, hidden, kv, inter, group, inter_group, blocks))
    kind = rng.choice(('prefill', 'decode', 'generate'))
    format = rng.choice(('int8', 'int8', 'int4', 'nf4', 'fp16'))
    batch = 1 if kind == 'generate' else rng.choice((1, 1, 2, 3, 5, 8))
    rank = rng.choice((0, 8, 32)) if format == 'int8' else 0
    return _drop(_smol('', kind, format, rank, rng.randint(2, 16), batch, _between(rng, 5, 256 // batch),
                       0 if kind == 'prefill' else rng.randint(1, 4) if kind == 'decode' else rng.randint(2, 12)))


def _drop(case):
    del case['name']
    return case


# ---------------------------------------------------------------- inputs
def _randn(g, *shape):
    return torch.randn(shape, generator=g, device='cuda')


def _codes(w, format, group):
    """(code values int8 [N, K], fp16 scales [N, K/group]) of an fp32 weight: absmax scales."""
    n, k = w.shape
    w = w.view(n, k // group, group)
    scale = (w.abs().amax(-1, keepdim=True) / LIMIT[format]).clamp_min(2.0 ** -24).half()
    w = w / scale.float()
    if format == 'nf4':
        table = torch.tensor(CODEBOOK, device=w.device)
        q = torch.bucketize(w, (table[:-1] + table[1:]) / 2).to(torch.int8)
    else:
        q = w.round().clamp(-LIMIT[format], LIMIT[format]).to(torch.int8)
    return q.view(n, k), scale.view(n, -1)


def _packed(q, format):
    """The packed bytes of code values: int8 as they are, else pairs, the low nibble first."""
    if format == 'int8':
        return q.view(torch.uint8).reshape(-1)
    flat = (q.view(torch.uint8) & 15).view(-1)
    if flat.numel() % 2:
        flat = torch.cat((flat, flat.new_zeros(1)))
    return (flat[0::2] | (flat[1::2] << 4)).contiguous()


def _weight(g, format, n, k, group):
    return _codes(_randn(g, n, k) * 0.02, format, group)


def _packed_weight(q, scales, format, group):
    return PackedWeight(tuple(q.shape), format, group, _packed(q, format).cpu().numpy().tobytes(),
                        scales.cpu().numpy().tobytes())


def _value64(q, scales, format):
    """The weight that codes and scales stand for, in 64 bits (the codebook is stored in fp16)."""
    n, k = q.shape
    v = q.double()
    if format == 'nf4':
        v = torch.tensor(CODEBOOK, device=q.device).half().double()[q.long()]
    return (v.view(n, scales.shape[1], -1) * scales.double()[:, :, None]).view(n, k)


def _shapes(case):
    """(name, N, K, group) of a block's projections, and of the head."""
    h, kv, i, g, gi = (case[key] for key in ('hidden', 'kv', 'inter', 'group', 'inter_group'))
    rows = [(h, h, g), (kv, h, g), (kv, h, g), (h, h, g), (i, h, g), (i, h, g), (h, i, gi)] * case['blocks']
    return rows + ([(case['vocab'], h, g)] if case['vocab'] else [])


def _linear_inputs(case, seed):
    g = torch.Generator(device='cuda').manual_seed(seed)
    n, k, m = case['n'], case['k'], case['m']
    q, scales = _weight(g, case['format'], n, k, case['group'])
    x = _randn(g, m, k).half()
    bias = (_randn(g, n) * 0.1).half() if case['bias'] else None
    rank = case['rank']
    factors = ((_randn(g, rank, k) * 0.01).half(), (_randn(g, n, rank) * 0.01).half()) if rank else None
    return q, scales, x, bias, factors


def _block_inputs(case, seed):
    g = torch.Generator(device='cuda').manual_seed(seed)
    for n, k, group in _shapes(case):
        yield (*_weight(g, case['format'], n, k, group), _randn(g, case['m'], k).half())


def _smol_inputs(case, seed):
    """Per layer {projection: (codes, scales, fp16 weight, factors)}, the norms, embedding and token ids."""
    g = torch.Generator(device='cuda').manual_seed(seed)
    layers = []
    for _ in range(case['layers']):
        layer = {}
        for name, (n, k) in SMOL.items():
            w = (_randn(g, n, k) * 0.02).half()
            q, scales = (None, None) if case['format'] == 'fp16' else _codes(
                w.float(), case['format'], k if case['format'] == 'int8' else 32)
            factors = None
            if case['rank']:
                factors = (_randn(g, case['rank'], k) * 0.01).half(), (_randn(g, n, case['rank']) * 0.01).half()
            layer[name] = (q, scales, w, factors)
        for name in NORMS:
            layer[name] = (1 + 0.1 * _randn(g, HIDDEN)).half()
        layers.append(layer)
    embedding = (_randn(g, VOCAB, HIDDEN) * 0.02).half()
    norm = (1 + 0.1 * _randn(g, HIDDEN)).half()
    ids = torch.randint(0, VOCAB, (case['batch'], case['length'] + case['steps']), generator=g, device='cuda')
    return layers, embedding, norm, ids


def _config(layers):
    return dict(model_type='llama', hidden_size=HIDDEN, intermediate_size=INTER, num_attention_heads=HEADS,
                num_key_value_heads=KV_HEADS, hidden_act='silu', attention_bias=False, mlp_bias=False,
                rms_norm_eps=1e-5, rope_theta=10000.0, rope_scaling=None, pretraining_tp=1,
                num_hidden_layers=layers, tie_word_embeddings=True, vocab_size=VOCAB)


def _capacity(case):
    return case['length'] + case['steps'] + 8


def _smol_model(case, layers, embedding, norm):
    config, format, built = _config(case['layers']), case['format'], []
    for layer in layers:
        weights = {name: (layer[name][2] if name in SMOL else layer[name]).cpu() for name in layer}
        packed = corrections = None
        if format != 'fp16':
            packed = {name: _packed_weight(*layer[name][:2], format, k if format == 'int8' else 32)
                      for name, (_, k) in SMOL.items()}
        if case['rank']:
            corrections = {name: LowRankCorrection(shape, case['rank'], *(f.cpu().numpy().tobytes()
                                                                          for f in layer[name][3]))
                           for name, shape in SMOL.items()}
        built.append(FrozenSmolLayer(config, weights, mode=MODE[format], packed_weights=packed,
                                     corrections=corrections, capacity=_capacity(case)))
    return FrozenSmolStack.from_layers(built), FrozenSmolIO(config, embedding.cpu(), norm.cpu()).cuda()


# ---------------------------------------------------------------- what a program has in hand
@torch.no_grad()
def prepare(case, seed):
    kind = case['kind']
    if kind == 'linear':
        q, scales, x, bias, factors = _linear_inputs(case, seed)
        if factors is not None:  # corrections go through the functional entry point
            return dict(kind='corrected', x=x, args=(_packed(q, case['format']), scales), options=dict(
                format=case['format'], N=case['n'], K=case['k'], group_size=case['group'], down=factors[0],
                up=factors[1], rank=case['rank']))
        module = QuantizedLinear(_packed_weight(q, scales, case['format'], case['group']),
                                 bias=None if bias is None else bias.cpu(), compact_groups=case['compact'],
                                 activation_scale=case['grid'] or None)
        module(x[:1])  # the weight goes to the device with the first call
        return dict(kind='module', module=module, x=x)
    if kind == 'block':
        rows, calls, buffers = _shapes(case), [], []
        for at, ((n, k, group), (q, scales, x)) in enumerate(zip(rows, _block_inputs(case, seed))):
            if at % 7 == 0:  # one buffer for a block's outputs, one for the head's
                buffers.append(torch.empty(case['m'] * sum(r[0] for r in rows[at:at + 7]), dtype=torch.float16, device='cuda'))
                left = buffers[-1]
            y, left = left[:case['m'] * n].view(case['m'], n), left[case['m'] * n:]
            calls.append(lowbit_hip.PreparedLinear(x, _packed(q, case['format']), scales, format=case['format'], N=n,
                                                   K=k, group_size=group, out=y))
        if case['m'] > 32:
            return dict(kind='launched', calls=calls, outputs=buffers)
        for call in calls:
            call.run()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            for call in calls:
                call.run()
        return dict(kind='graph', graph=graph, calls=calls, outputs=buffers)
    layers, embedding, norm, ids = _smol_inputs(case, seed)
    stack, io = _smol_model(case, layers, embedding, norm)
    prompt, more = ids[:, :case['length']], ids[:, case['length']:]
    state = dict(kind=kind, stack=stack, io=io, prompt=prompt, more=more)
    h, caches = stack.prefill(io.embed_tokens(prompt))
    if kind == 'decode':
        state['caches'] = caches
    elif kind == 'generate':
        state['caches'], state['token'] = caches, int(io.logits(h[:, -1:])[0, 0].argmax())
        state['decoder'] = GraphDecoder(stack, io)
        state['decoder'].load(caches, state['token'])
        state['decoder'].capture()
        state['steps'] = case['steps']
    return state


# ---------------------------------------------------------------- one pass
@torch.no_grad()
def run(state):
    kind = state['kind']
    if kind == 'module':
        return state['module'](state['x'])
    if kind == 'corrected':
        return lowbit_hip.linear(state['x'], *state['args'], **state['options'])
    if kind == 'launched':
        for call in state['calls']:
            call.run()
        return state['outputs']
    if kind == 'graph':
        state['graph'].replay()
        return state['outputs']
    stack, io = state['stack'], state['io']
    if kind == 'prefill':
        h, caches = stack.prefill(io.embed_tokens(state['prompt']))
        return dict(h=h, logits=io.logits(h[:, -1:]), keys=[c.keys for c in caches], values=[c.values for c in caches])
    if kind == 'decode':
        caches, logits = state['caches'], []
        for token in state['more'].split(1, 1):
            h, caches = stack.decode(io.embed_tokens(token), caches)
            logits.append(io.logits(h))
        return dict(logits=logits, keys=[c.keys for c in caches], values=[c.values for c in caches])
    decoder = state['decoder']
    decoder.load(state['caches'], state['token'])
    decoder.generate(state['steps'])
    return dict(logits=decoder.logits, tokens=decoder.tokens, keys=decoder.keys, values=decoder.values)


# ---------------------------------------------------------------- what a pass cannot do without
def _weight_bytes(format, n, k, group):
    return 2 * n * k if format == 'fp16' else (n * k if format == 'int8' else n * k / 2) + 2 * n * (k // group)


def work(case):
    kind, format = case['kind'], case['format']
    if kind == 'linear':
        m, n, k, r = (case[key] for key in ('m', 'n', 'k', 'rank'))
        return dict(bytes=_weight_bytes(format, n, k, case['group']) + 2 * m * (n + k) + 2 * n * case['bias'] + 2 * r * (n + k),
                    flops=2 * m * n * k + 2 * m * r * (n + k))
    if kind == 'block':
        m = case['m']
        return dict(bytes=sum(_weight_bytes(format, n, k, g) + 2 * m * (n + k) for n, k, g in _shapes(case)),
                    flops=sum(2 * m * n * k for n, k, _ in _shapes(case)))
    layers, rank, batch, length, steps = (case[key] for key in ('layers', 'rank', 'batch', 'length', 'steps'))
    weights = layers * sum(_weight_bytes(format, n, k, k if format == 'int8' else 32) + 2 * rank * (n + k)
                           for n, k in SMOL.values())
    flops = layers * sum(2 * n * k + 2 * rank * (n + k) for n, k in SMOL.values())  # a token's
    head, slot = 2 * VOCAB * HIDDEN, layers * 2 * 2 * KV  # bytes of the head, and of one position's keys and values
    if kind == 'prefill':
        pairs = length * (length + 1) // 2
        return dict(bytes=weights + head + batch * length * (4 * HIDDEN + slot) + 2 * batch * VOCAB,
                    flops=batch * (length * flops + head + layers * 4 * HEADS * HEAD_DIM * pairs))
    seen = sum(length + t + 1 for t in range(steps))
    return dict(bytes=steps * (weights + head + 2 * batch * VOCAB) + batch * slot * seen,
                flops=batch * (steps * (flops + head) + layers * 4 * HEADS * HEAD_DIM * seen))


# ---------------------------------------------------------------- the same in 64 bits
def _norm64(x, gamma):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * gamma.double()


def _forward64(layers, x):
    """(output, keys, values per layer) of a causal pass over x [B, S, 576]."""
    b, s, _ = x.shape
    angles = torch.outer(torch.arange(s, device=x.device).double(),
                         10000.0 ** (-torch.arange(0, HEAD_DIM, 2, device=x.device).double() / HEAD_DIM)).repeat(1, 2)
    cos, sin = angles.cos(), angles.sin()
    mask = torch.triu(torch.full((s, s), float('-inf'), dtype=torch.float64, device=x.device), 1)
    heads = lambda t: t.view(b, s, -1, HEAD_DIM).transpose(1, 2)  # noqa: E731
    rotate = lambda t: t * cos + torch.cat((-t[..., 32:], t[..., :32]), -1) * sin  # noqa: E731
    keys, values = [], []
    for w, norms in layers:
        linear = lambda t, name: t @ w[name].T  # noqa: E731
        n1 = _norm64(x, norms[0])
        q, k, v = (heads(linear(n1, f'self_attn.{p}_proj.weight')) for p in 'qkv')
        q, k = rotate(q), rotate(k)
        keys.append(k)
        values.append(v)
        k, v = (t.repeat_interleave(HEADS // KV_HEADS, 1).contiguous() for t in (k, v))
        p = (q @ k.transpose(-1, -2).contiguous() * HEAD_DIM ** -0.5 + mask).softmax(-1)
        x = x + linear((p @ v).transpose(1, 2).reshape(b, s, HIDDEN), 'self_attn.o_proj.weight')
        n2 = _norm64(x, norms[1])
        gate, up = linear(n2, 'mlp.gate_proj.weight'), linear(n2, 'mlp.up_proj.weight')
        x = x + linear(gate * torch.sigmoid(gate) * up, 'mlp.down_proj.weight')
    return x, keys, values


@torch.no_grad()
def exact(case, seed):
    kind, format = case['kind'], case['format']
    if kind == 'linear':
        q, scales, x, bias, factors = _linear_inputs(case, seed)
        w, x64 = _value64(q, scales, format), x.double()
        if case['grid']:  # activations on their grid, the weight's steps as the FakeQuantize limits give them
            x64 = (x64 / case['grid']).round().clamp(-128, 127) * case['grid']
            s = scales.double()
            w = q.double() * (((127 * s).half().double() - (-128 * s).half().double()) / 255)
        y = x64 @ w.T
        if bias is not None:
            y = y + bias.double()
        return y if factors is None else y + x64 @ factors[0].double().T @ factors[1].double().T
    if kind == 'block':
        ys = [(x.double() @ _value64(q, scales, format).T).view(-1) for q, scales, x in _block_inputs(case, seed)]
        return [torch.cat(ys[at:at + 7]) for at in range(0, len(ys), 7)]
    raw, embedding, norm, ids = _smol_inputs(case, seed)
    layers = []
    for layer in raw:
        weights = {}
        for name in SMOL:
            q, scales, w, factors = layer[name]
            weights[name] = w.double() if q is None else _value64(q, scales, format)
            if factors is not None:
                weights[name] = weights[name] + factors[1].double() @ factors[0].double()
        layers.append((weights, [layer[name] for name in NORMS]))
    head = embedding.double()
    logits = lambda h: _norm64(h, norm) @ head.T  # noqa: E731
    length, steps = case['length'], case['steps']
    slots = lambda ts: [torch.cat((t, t.new_zeros(*t.shape[:2], _capacity(case) - t.shape[2], HEAD_DIM)), 2)  # noqa: E731
                        for t in ts]
    if kind == 'generate':
        ids = ids[:, :length]
        for _ in range(steps + 1):
            h, keys, values = _forward64(layers, head[ids])
            last = logits(h[:, -1])
            ids = torch.cat((ids, last.argmax(-1, keepdim=True)), 1)
        return dict(logits=last, tokens=None, keys=slots(keys), values=slots(values))
    h, keys, values = _forward64(layers, head[ids])
    if kind == 'prefill':
        return dict(h=h, logits=logits(h[:, -1:]), keys=slots(keys), values=slots(values))
    return dict(logits=[logits(h[:, length + t:length + t + 1]) for t in range(steps)], keys=slots(keys),
                values=slots(values))


def tolerance(case):
    # Seen against 64 bits: 2.0e-4 to 3.5e-4 for a linear (fp16 results, fp16(q s) weights, a bias added in
    # fp16), up to 1.6e-3 for the layers' outputs, keys and logits after 30 layers of fp16 rounding points.
    if case['kind'] in ('linear', 'block'):
        return {'rel': 1e-3}
    return {'rel': 6e-3}
