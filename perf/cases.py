"""What the speed of this framework is judged by: the calls a program that uses it makes, at the sizes it makes them.

    listed()              the named cases
    draw(rng)             one more case from the same ranges
    prepare(case, seed)   what the program holds before the call: the layer with its weights, the inputs
    run(state)            one pass through the public entry points and everything it computes
    work(case)            bytes and operations the pass cannot do without
    tolerance(case)       how far another correct implementation at the same precision may be off

Four kinds of case:

    serve      forward of a dropless layer without gradients: from a few tokens (decode) to a few thousand (prefill)
    train      forward and backward of a dropless layer, all gradients: grouped or block-sparse experts, MLP or GLU,
               16-bit or fp32 parameters, fp32 parameters under autocast, with or without the memory-optimised backward
               and the auxiliary losses; routing by the layer's own router or prescribed (skewed)
    capacity   forward and backward of the capacity-factor layer, which drops tokens
    permute    the routing and permutation operators called one by one, forward and backward
"""
import functools
import math

import torch
import torch.nn.functional as F

from megablocks_amd import ops
from megablocks_amd.layers import moe as moe_layers
from megablocks_amd.layers import router as router_layers
from megablocks_amd.layers.arguments import DEFAULT_ACTIVATION_FN, Arguments
from megablocks_amd.layers.dmoe import dMoE
from megablocks_amd.layers.moe import MoE

_DTYPES = {'bf16': torch.bfloat16, 'fp16': torch.float16, 'fp32': torch.float32}
_BLOCK = 128            # rows the block-sparse experts and the padded operators round an expert's rows up to
_LOSS_WEIGHT, _ZLOSS_WEIGHT = 0.01, 0.001

# the dearest listed case: no drawn one takes more
_MAX_FLOPS = 2.0e13
_MAX_WEIGHT_BYTES = 3 << 30


def _layer(kind, tokens, hidden, ffn, experts, top_k, mlp='mlp', impl='grouped', dtype='bf16', routing='router', amp=False,
           memopt=False, aux=False):
    return dict(kind=kind, tokens=tokens, hidden=hidden, ffn=ffn, experts=experts, top_k=top_k, mlp=mlp, impl=impl,
                dtype=dtype, routing=routing, amp=amp, memopt=memopt, aux=aux)


def listed():
    return [
        # Decoding a batch of 16 sequences with a few large experts: every expert is touched by a handful of rows, the
        # pass is the reading of 2.8 GB of weights.
        dict(_layer('serve', 16, 4096, 14336, 8, 2, mlp='glu'), name='decode_8e_top2'),
        # Decoding a few sequences with many small experts: the smallest call there is, latency and launches count.
        dict(_layer('serve', 5, 2048, 1408, 64, 6, mlp='glu'), name='decode_64e_top6'),
        # Prefill of one prompt of no particular length, one expert per token.
        dict(_layer('serve', 3001, 1024, 4096, 64, 1, dtype='fp16'), name='prefill_64e_top1'),
        # Training, a few large experts (the default workload of bench.py).
        dict(_layer('train', 8192, 4096, 14336, 8, 2, mlp='glu'), name='train_8e_top2'),
        # Training, many experts of a few hundred rows each.
        dict(_layer('train', 16384, 1024, 4096, 64, 1), name='train_64e_top1'),
        # Training, fine-grained experts with skewed popularity (some get no tokens at all).
        dict(_layer('train', 32768, 2048, 1408, 64, 6, mlp='glu', routing='zipf'), name='train_64e_top6_skewed'),
        # Training in the block-sparse mode: every expert's rows padded to blocks.
        dict(_layer('train', 24576, 2048, 8192, 16, 4, impl='sparse'), name='train_16e_top4_sparse'),
        # Training in fp32 (small models, and the runs others are checked against).
        dict(_layer('train', 4096, 1024, 4096, 8, 2, dtype='fp32'), name='train_fp32'),
        # A small model as it is usually trained: fp32 parameters under autocast, load-balancing loss and z-loss on.
        dict(_layer('train', 1024, 512, 1408, 8, 2, mlp='glu', dtype='fp32', amp=True, aux=True), name='train_small_autocast'),
        # Sizes that are no multiples of a tile in any direction, a number of experts that is no power of two, and the
        # backward that recomputes instead of keeping.
        dict(_layer('train', 3001, 1032, 2728, 12, 2, dtype='fp16', memopt=True), name='train_odd_memopt'),
        # Training with the capacity-factor layer.
        dict(kind='capacity', tokens=16384, hidden=768, ffn=3072, experts=32, top_k=1, dtype='fp16',
             name='train_capacity_32e'),
        # The routing and permutation operators by themselves.
        dict(kind='permute', tokens=16384, hidden=1024, experts=8, top_k=4, dtype='fp16', name='permute_8e_top4'),
    ]


def _log_uniform(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def _multiple(rng, low, high, of):
    return max(of, int(round(_log_uniform(rng, low, high) / of)) * of)


def _weight_bytes(c):
    return (3 if c.get('mlp') == 'glu' else 2) * c['experts'] * c['hidden'] * c['ffn'] * (4 if c['dtype'] == 'fp32' else 2)


def _draw_layer(rng, kind):
    mlp = rng.choice(['mlp', 'glu'])
    experts = rng.choice([4, 8, 12, 16, 32, 64, 128])
    top_k = rng.choice([k for k in (1, 2, 4, 6, 8) if 2 * k <= experts])
    if kind == 'serve':
        dtype = rng.choice(['bf16', 'fp16'])
        c = _layer('serve', int(_log_uniform(rng, 1, 4097)), _multiple(rng, 512, 4096, 64), _multiple(rng, 704, 14336, 64),
                   experts, top_k, mlp=mlp, dtype=dtype)
    else:
        shape = rng.choice(['plain', 'plain', 'plain', 'odd', 'fp32'])
        of = 8 if shape == 'odd' else 64
        c = _layer('train', int(_log_uniform(rng, 256, 32768)), _multiple(rng, 512, 4096, of), _multiple(rng, 704, 14336, of),
                   experts, top_k, mlp=mlp, dtype='fp32' if shape == 'fp32' else rng.choice(['bf16', 'bf16', 'fp16']),
                   routing=rng.choice(['router', 'router', 'zipf']), memopt=rng.random() < 0.25)
        if shape == 'plain':
            # block-sparse experts (no memory-optimised backward for GLU there), or autocast, or auxiliary losses
            option = rng.choice(['', '', 'sparse', 'amp', 'aux'])
            if option == 'sparse' and not (mlp == 'glu' and c['memopt']):
                c.update(impl='sparse', ffn=max(_BLOCK, c['ffn'] // _BLOCK * _BLOCK))
            elif option == 'amp':
                c.update(dtype='fp32', amp=True, aux=rng.random() < 0.5, routing='router')
            elif option == 'aux':
                c.update(aux=True, routing='router')
    return c


def draw(rng):
    kind = rng.choice(['serve', 'serve', 'serve', 'train', 'train', 'train', 'train', 'capacity', 'permute'])
    while True:
        if kind in ('serve', 'train'):
            c = _draw_layer(rng, kind)
        elif kind == 'capacity':
            experts = rng.choice([2, 4, 8, 16, 32, 64])
            c = dict(kind='capacity', tokens=int(_log_uniform(rng, 512, 32768)), hidden=_multiple(rng, 512, 2048, 64),
                     ffn=_multiple(rng, 1024, 8192, 64), experts=experts, top_k=rng.choice([1, 1, 2]),
                     dtype=rng.choice(['bf16', 'fp16']))
        else:
            experts = rng.choice([2, 4, 8, 16, 32, 64, 128])
            c = dict(kind='permute', tokens=int(_log_uniform(rng, 512, 131072)), hidden=_multiple(rng, 512, 4096, 8),
                     experts=experts, top_k=rng.choice([k for k in (1, 2, 4, 8) if k <= experts]),
                     dtype=rng.choice(['bf16', 'fp16', 'fp32']))
        # fp32 products run at a sixteenth of the 16-bit rate: they count that much more
        rate = 16 if c['dtype'] == 'fp32' and not c.get('amp') else 1
        if c.get('ffn') and _weight_bytes(c) > _MAX_WEIGHT_BYTES:
            continue
        if work(c)['flops'] * rate <= _MAX_FLOPS and c['tokens'] * c['top_k'] * c['hidden'] <= 32768 * 6 * 2048:
            return c


# ---------------------------------------------------------------------------------------------------------------- inputs
def _normal(gen, shape, dtype, std=1.0):
    return (torch.randn(shape, device='cuda', generator=gen) * std).to(dtype)


def _zipf_routing(c, gen, dtype):
    """Distinct experts per token by a popularity r^-1.2 over the ranks (the least popular sixteenth gets nothing, if top_k
    allows it), gate weights a softmax of N(0, 1)."""
    experts, top_k, tokens = c['experts'], c['top_k'], c['tokens']
    p = torch.arange(1, experts + 1, dtype=torch.float32, device='cuda') ** -1.2
    empty = min(experts // 16, experts - top_k)
    if empty:
        p[experts - empty:] = 0
    ids = torch.randperm(experts, generator=gen, device='cuda')
    # the k largest of log p + Gumbel noise: k draws without replacement
    noise = torch.empty(tokens, experts, device='cuda').exponential_(generator=gen).log_().neg_()
    top_experts = ids[(p.log() + noise).topk(top_k, dim=-1).indices].contiguous()
    weights = torch.randn(tokens, top_k, device='cuda', generator=gen).softmax(-1).to(dtype)
    scores = torch.zeros(tokens, experts, device='cuda', dtype=dtype).scatter_(1, top_experts, weights)
    return scores, weights, top_experts


def _build_layer(c, gen, cls):
    dtype = _DTYPES[c['dtype']]
    init = functools.partial(torch.nn.init.normal_, mean=0.0, std=0.02, generator=gen)
    aux = bool(c.get('aux'))
    args = Arguments(
        hidden_size=c['hidden'], ffn_hidden_size=c['ffn'], moe_num_experts=c['experts'], moe_top_k=c['top_k'], bias=False,
        mlp_type=c.get('mlp', 'mlp'), mlp_impl=c.get('impl', 'grouped'), moe_capacity_factor=1,
        activation_fn=F.silu if c.get('mlp') == 'glu' else DEFAULT_ACTIVATION_FN,
        moe_normalize_expert_weights=1 if c['top_k'] > 1 else None,
        moe_loss_weight=_LOSS_WEIGHT if aux else 0.0, moe_zloss_weight=_ZLOSS_WEIGHT if aux else 0.0,
        moe_lbl_in_fp32=aux, moe_zloss_in_fp32=aux,
        memory_optimized_mlp=bool(c.get('memopt')), fp16=dtype == torch.float16, bf16=dtype == torch.bfloat16,
        device=torch.device('cuda'), init_method=init, output_layer_init_method=init)
    return args, cls(args)


class _State:
    pass


def prepare(case, seed):
    gen = torch.Generator(device='cuda').manual_seed(seed)
    s = _State()
    s.kind, s.top_k = case['kind'], case['top_k']
    dtype = _DTYPES[case['dtype']]
    tokens, hidden, experts = case['tokens'], case['hidden'], case['experts']
    if s.kind == 'permute':
        s.experts = experts
        s.end_bit = max(int(math.ceil(math.log2(experts))), 1)
        logits = torch.randn(tokens, experts, device='cuda', generator=gen)
        weights, ids = logits.softmax(-1).topk(s.top_k, dim=-1)
        s.ids = ids.flatten().int()
        s.weights = weights.flatten().to(dtype).requires_grad_(True)
        s.x = _normal(gen, (tokens, hidden), dtype).requires_grad_(True)
        s.grad = _normal(gen, (tokens, hidden), dtype)
        return s
    s.args, s.layer = _build_layer(case, gen, MoE if s.kind == 'capacity' else dMoE)
    s.amp, s.aux = bool(case.get('amp')), bool(case.get('aux'))
    # [sequence, batch, hidden], as a transformer hands it over
    s.x = _normal(gen, (tokens, 1, hidden), dtype)
    s.routing = None
    if s.kind == 'serve':
        s.layer.eval()
        return s
    s.x.requires_grad_(True)
    s.grad = _normal(gen, (tokens, 1, hidden), torch.bfloat16 if s.amp else dtype)
    if case.get('routing') == 'zipf':
        scores, weights, top_experts = _zipf_routing(case, gen, dtype)
        s.routing = (scores, weights.requires_grad_(True), top_experts)
    return s


# ------------------------------------------------------------------------------------------------------------------ pass
def _permute(s):
    s.x.grad = s.weights.grad = None
    bin_ids, indices = ops.sort(s.ids, s.end_bit)
    tokens_per_expert = ops.histogram(s.ids, s.experts)
    padded_bins = ops.inclusive_cumsum(ops.round_up(tokens_per_expert, _BLOCK), 0)
    bins = ops.inclusive_cumsum(tokens_per_expert, 0)
    rows = ops.padded_gather(s.x, indices, bin_ids, bins, padded_bins, s.top_k)
    y = ops.padded_scatter(rows, indices, bin_ids, s.weights, bins, padded_bins, s.top_k)
    y.backward(s.grad)
    return dict(bin_ids=bin_ids, indices=indices, tokens_per_expert=tokens_per_expert, bins=bins, padded_bins=padded_bins,
                y=y, dx=s.x.grad, dweights=s.weights.grad)


def _train(s):
    s.layer.zero_grad(set_to_none=True)
    s.x.grad = None
    losses = []
    if s.aux:
        moe_layers.clear_load_balancing_loss()
        router_layers.clear_router_zloss()
    with torch.autocast('cuda', dtype=torch.bfloat16, enabled=s.amp):
        if s.routing is None:
            y = s.layer(s.x)
        else:
            s.routing[1].grad = None
            y = s.layer.experts(s.x, *s.routing)
        if s.aux:
            losses.append(moe_layers.batched_load_balancing_loss(s.args) + router_layers.batched_router_zloss(s.args))
    torch.autograd.backward([y] + losses, [s.grad] + [None] * len(losses))
    out = dict(y=y, losses=losses, dx=s.x.grad, grads={name: p.grad for name, p in s.layer.named_parameters() if p.grad is not None})
    if s.routing is not None:
        out['dweights'] = s.routing[1].grad
    return out


def run(state):
    if state.kind == 'serve':
        with torch.no_grad():
            return state.layer(state.x)
    if state.kind == 'permute':
        return _permute(state)
    return _train(state)


# ------------------------------------------------------------------------------------------------------------------ work
def _experts_touched(c):
    """Experts that get at least one token, for tokens that choose evenly."""
    return c['experts'] * (1.0 - (1.0 - c['top_k'] / c['experts']) ** c['tokens'])


def work(case):
    c = case
    size = 4 if c['dtype'] == 'fp32' else 2
    tokens, hidden, slots = c['tokens'], c['hidden'], c['tokens'] * c['top_k']
    if c['kind'] == 'permute':
        # each operator's tensors: gather x -> rows, scatter rows -> y, and backward (dy, rows) -> (drows, dweights), drows -> dx
        moved = (tokens + slots) + (slots + tokens) + (tokens + 2 * slots) + (slots + tokens)
        return {'bytes': moved * hidden * size + 5 * 4 * slots, 'flops': 6 * slots * hidden}
    products = 3 if c.get('mlp') == 'glu' else 2
    weights = products * c['experts'] * hidden * c['ffn'] * size
    router = c['experts'] * hidden * size
    forward = products * 2 * slots * hidden * c['ffn'] + 2 * tokens * hidden * c['experts']
    if c['kind'] == 'serve':
        return {'bytes': weights * _experts_touched(c) / c['experts'] + router + 2 * tokens * hidden * size, 'flops': forward}
    # x and the output's gradient in, the output and x's gradient out; weights in, their gradients out
    return {'bytes': 2 * (weights + router) + 4 * tokens * hidden * size, 'flops': 3 * forward}


def tolerance(case):
    return {'rel': {'bf16': 1.5e-2, 'fp16': 2e-3, 'fp32': 1e-5}['bf16' if case.get('amp') else case['dtype']]}
