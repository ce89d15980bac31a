"""The work that users of this package have it do, as cases that can be timed.

A case is one pass through the public entry points: an ``Encoder`` layer forward, or forward and backward, at the
sizes people run such layers at; a stack of layers; the decoder layer; the softmax operators on their own.
``listed()`` names twelve, ``draw()`` gives others of the same ranges: batches of 1 to 96 samples, 16 to 2048 positions
(multiples of 128, multiples of 8 and neither), embeddings of 512 to 4096 with head sizes 64 and 128, ReLU and
GELU, with and without a causal mask, in this package's dimension orders and in those of the configurations that
the reference ships.  Everything is fp16, the only type the package computes in.
"""
import math

import torch

from substation_amd import DecoderLayer, Encoder, EncoderStack, causal_mask
from substation_amd import layouts as lay
from substation_amd.ops import Ops

#: heads and embedding: head size 64 at the usual widths, 128 at the wide ones
WIDTHS = [(8, 512), (12, 768), (16, 1024), (16, 2048), (32, 4096)]

REFERENCE = 'bert-b8-l512-h16-e1024'


def listed():
    def case(name, kind, B, L, H, E, act='gelu', p=0.1, **more):
        return dict(name=name, kind=kind, B=B, L=L, H=H, E=E, act=act, p=p, **more)
    return [
        # one short request to a served layer: latency, and nothing but launches and host work
        case('infer b1 l64 e768', 'infer', 1, 64, 12, 768, p=0.0),
        # a batch of requests padded to their longest, which is whatever it is
        case('infer b24 l77 e768', 'infer', 24, 77, 12, 768, p=0.0),
        # the smallest training step people write down: the configuration of the CPU baseline
        case('train b2 l128 e768', 'train', 2, 128, 12, 768, act='relu'),
        # the benchmark's layer, in this package's dimension orders
        case('train b8 l512 e1024', 'train', 8, 512, 16, 1024, act='relu'),
        # the same layer under the configuration that the reference ships (feature-major activations)
        case('train b8 l512 e1024 ref', 'train', 8, 512, 16, 1024, act='relu', layouts='reference'),
        # many short sequences
        case('train b96 l128 e1024', 'train', 96, 128, 16, 1024, act='relu', layouts='bert-b96-l128-h16-e1024'),
        # a wide layer on long sequences: the largest
        case('train b4 l2048 e4096', 'train', 4, 2048, 32, 4096),
        # sequences of a length that is a multiple of nothing: batch and length both odd
        case('train b13 l201 e768', 'train', 13, 201, 12, 768),
        # masked self-attention (a language model's layer) at a length that is a multiple of 8 only
        case('causal b4 l1000 e1024', 'train', 4, 1000, 16, 1024, causal=True),
        # several layers, with the workspaces that a stack keeps
        case('stack4 b4 l256 e768', 'stack', 4, 256, 12, 768, layers=4),
        # the decoder layer with attention over the encoder's output
        case('decoder b8 l256 e1024', 'decoder', 8, 256, 16, 1024, source=512),
        # softmax with dropout and its backward as single operators, at the size the benchmark gives them
        case('softmax b8 l512 h16', 'softmax', 8, 512, 16, 1024),
    ]


def _log_between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _length(rng, high):
    """16 .. high: a third multiples of 128, a third multiples of 8, a third any length."""
    step = rng.choice([128, 8, 1])
    return max(1, round(_log_between(rng, max(16, step), high) / step)) * step


def draw(rng):
    kind = rng.choice(['infer', 'infer', 'train', 'train', 'train', 'train', 'causal', 'reference', 'stack', 'decoder',
                       'softmax'])
    while True:
        H, E = rng.choice(WIDTHS)
        c = dict(kind=kind, B=_log_between(rng, 1, 96), L=_length(rng, 2048), H=H, E=E,
                 act=rng.choice(['relu', 'gelu']), p=0.0 if kind == 'infer' else 0.1)
        if kind in ('causal', 'reference'):
            c['kind'] = 'train'
            c['causal' if kind == 'causal' else 'layouts'] = True if kind == 'causal' else 'reference'
        elif kind == 'stack':
            c['layers'] = rng.randint(2, 4)
        elif kind == 'decoder':       # this layer takes multiples of 128 only
            c['L'] = 128 * rng.randint(1, 8)
            c['source'] = 128 * rng.randint(1, 8)
        # no drawn case costs more than the largest listed one: by its operations, and, for lengths that are
        # multiples of nothing, by its scores, which such a length makes dear
        scores = c['B'] * H * c['L'] * max(c['L'], c.get('source', 0))
        if work(c)['flops'] > 2.5e12 or scores > (2.2e7 if c['L'] % 8 else 2.7e8):
            continue
        return c


def _fill(module, generator, std):
    """Weights ~ N(0, std), biases ~ N(0, 0.02), LayerNorm scales 1 and biases 0."""
    with torch.no_grad():
        for name, t in module.named_parameters():
            name = name.split('.')[-1]
            if name in ('S1', 'S2') or name.endswith('_scale'):
                t.fill_(1.0)
            elif name in ('B1', 'B2') or name.startswith('norm'):
                t.fill_(0.0)
            else:
                small = t.dim() == 1 or name == 'BKQV' or name.endswith('_b')
                t.copy_(torch.randn(t.shape, generator=generator, device='cuda') * (0.02 if small else std))


def prepare(case, seed):
    B, L, H, E, act, p, kind = (case[k] for k in ('B', 'L', 'H', 'E', 'act', 'p', 'kind'))
    g = torch.Generator('cuda').manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, generator=g, device='cuda').half()

    if kind == 'softmax':
        ops = Ops(B, L, H, E, seed=seed)
        beta, d_drop = normal(H, B, L, L), normal(H, B, L, L)
        outs = [torch.empty_like(beta) for _ in range(4)]
        return dict(kind=kind, ops=ops, beta=beta, d_drop=d_drop, outs=outs, p=p, scale=1.0 / math.sqrt(E // H))

    std = 0.01 if E >= 4096 else 0.02
    if kind == 'decoder':
        with torch.device('cuda'):
            module = DecoderLayer(B, L, case['source'], H, E, p, p, p, p, activation=act, seed=seed)
        module = module.cuda()
        _fill(module, g, std)
        return dict(kind=kind, module=module, x=normal(B, L, E).requires_grad_(),
                    source=normal(B, case['source'], E).requires_grad_(), dy=normal(B, L, E))

    which = case.get('layouts')
    layouts = lay.reference_layouts(REFERENCE) if which == 'reference' else lay.mi355x_layouts(which)
    with torch.device('cuda'):
        if kind == 'stack':
            module = EncoderStack(case['layers'], B, L, H, E, layouts, torch.float16, p, p, p, p, activation=act, seed=seed)
        else:
            module = Encoder('unused', B, L, H, E, layouts, torch.float16, p, p, p, p, activation=act, seed=seed)
    _fill(module, g, std)
    if case.get('causal'):
        module.set_attention_mask(causal_mask(L))
    sizes = lay.sizes_map(B, L, H, E)
    x, dy = (normal(*lay.shape_of(layouts[k][1], sizes)) for k in ('input', 'output'))
    return dict(kind=kind, module=module, x=x if kind == 'infer' else x.requires_grad_(), dy=dy)


def run(state):
    kind = state['kind']
    if kind == 'infer':
        with torch.no_grad():
            return state['module'](state['x'])
    if kind == 'softmax':
        ops = state['ops']
        alpha, mask, drop, d_beta = state['outs']
        ops.softmax(state['beta'], 'HBJK', alpha, 'HBJK', mask, 'HBJK', drop, 'HBJK', scale=state['scale'], p=state['p'])
        ops.bs(alpha, 'HBJK', mask, 'HBJK', state['d_drop'], 'HBJK', d_beta, 'HBJK', scale=state['scale'])
        return [alpha, mask, drop, d_beta]
    # one training step's forward and backward: gradients cleared, then formed
    module = state['module']
    inputs = [state[k] for k in ('x', 'source') if k in state]
    module.zero_grad(set_to_none=True)
    for t in inputs:
        t.grad = None
    y = module(*inputs)
    y.backward(state['dy'])
    return [y.detach()] + [t.grad for t in inputs] + [t.grad for t in module.parameters()]


def work(case):
    """Inputs (weights among them) read once, outputs (gradients among them) written once; the multiplications and
    additions of the layer's products, twice as many again for the backward pass.  A causal mask leaves half of the
    attention products to do."""
    B, L, H, E, kind = (case[k] for k in ('B', 'L', 'H', 'E', 'kind'))
    if kind == 'softmax':
        return dict(bytes=6 * 2 * H * B * L * L, flops=20 * H * B * L * L)
    tokens, U = B * L, 4 * E
    weights = 4 * E * E + 2 * E * U + 9 * E + U
    acts = 2 * tokens * E
    products = 2 * tokens * (4 * E * E + 2 * E * U)
    attention = 4 * B * L * L * E / (2 if case.get('causal') else 1)
    if kind == 'decoder':
        S = case['source']
        weights += 4 * E * E + 6 * E
        acts += B * S * E
        products += 2 * (2 * tokens + 2 * B * S) * E * E
        attention = attention / 2 + 4 * B * L * S * E
    n = case.get('layers', 1)
    if kind == 'infer':
        return dict(bytes=2 * (weights + acts), flops=products + attention)
    return dict(bytes=2 * (2 * n * weights + 2 * acts), flops=3 * n * (products + attention))


def tolerance(case):
    """fp16 values rounded at every operator's boundary.  Training: where a pre-activation lies within rounding of zero,
    ReLU's gate may fall either way (about one in ten thousand does), which moves whole gradient elements."""
    if case['kind'] == 'softmax':
        return dict(rel=1e-3, max=4e-3)
    if case['kind'] == 'infer':
        return dict(rel=4e-3, max=4e-2)
    return dict(rel=1e-2, max=0.2)
