"""Learned top-k router: megablocks/layers/router.py:10-114.  The linear layer is torch's (a small dense
GEMM), except for its gradients on large 16-bit batches, which go through the grouped kernels;
softmax, top-k and the renormalisation of the selected weights are one HIP kernel each way.  The outputs
feed the HIP routing kernels."""
import ctypes
from typing import Any

import torch

from megablocks_amd import _lib
from megablocks_amd.layers import common
from megablocks_amd.layers.arguments import Arguments

_ROUTER_LOGITS = []

# softmax / top-k / renormalisation as one HIP kernel each way (False: torch's operations, as the reference)
FUSED_SOFTMAX_TOPK = True


def _save_router_logits(logits: torch.Tensor, args: Arguments, lse=None):
    """router.py:17-22.  lse: logsumexp(logits, dim=1) in fp32 where the router kernel has written it (differentiable
    through that kernel's backward), else None."""
    if args.moe_zloss_weight == 0:
        return
    _ROUTER_LOGITS.append((logits, lse))


class LossSums(torch.autograd.Function):
    """[scales[l] * sum(values[l] * counts[l]) for l] with counts[l] a row for every row of values[l], or (counts None) * sum(values[l]^2): the
    sums of the auxiliary losses (moe.py:69-89, router.py:37-42), fp32, of all layers by one launch (two for long ones) forward and one backward.
    A single layer goes without the arrays of those for many, 2 us of the host's time a call."""

    @staticmethod
    def takes(values, counts) -> bool:
        """Plain contiguous tensors on the GPU, the values of one type, the counts int32, and nothing that acts on torch's operators at work (autocast
        does not cast these)."""
        device, dtype = values[0].device, values[0].dtype
        plain = lambda t, dtype: type(t) is torch.Tensor and t.dtype == dtype and t.device == device and t.is_contiguous()
        return values[0].is_cuda and dtype in _lib.DTYPE and all(plain(v, dtype) and v.numel() for v in values) and \
            (counts is None or all(plain(c, torch.int32) for c in counts)) and common.only_computed(autocast=True)

    @staticmethod
    def _arrays(sizes, scales):
        return (ctypes.c_int64 * len(sizes))(*sizes), (ctypes.c_float * len(scales))(*scales)

    @staticmethod
    def _pointers(tensors):
        return (ctypes.c_void_p * len(tensors))(*map(_lib.ptr, tensors))

    @staticmethod
    def forward(ctx: Any, scales, counts, *values):
        first, layers = values[0], len(values)
        period = 1 if counts is None else first.shape[1]
        sizes = [v.numel() for v in values]
        out = torch.empty(layers, dtype=torch.float32, device=first.device)
        nbytes = _lib.lib.mbx_loss_sums_scratch_bytes(max(sizes), layers)
        scratch = torch.empty(nbytes, dtype=torch.uint8, device=first.device) if nbytes else None
        with _lib.device_of(out):
            if layers == 1:
                rc = _lib.lib.mbx_loss_sum(_lib.ptr(first), _lib.dtype_of(first), None if counts is None else _lib.ptr(counts[0]), sizes[0], period,
                                           scales[0], _lib.ptr(out), _lib.ptr(scratch), _lib.stream())
            else:
                rc = _lib.lib.mbx_loss_sums(LossSums._pointers(values), _lib.dtype_of(first), None if counts is None else LossSums._pointers(counts),
                                            *LossSums._arrays(sizes, scales), layers, period, _lib.ptr(out), _lib.ptr(scratch), _lib.stream())
            _lib.check(rc, 'loss_sums')
        ctx.save_for_backward(*(values if counts is None else counts))
        ctx.scales, ctx.counted, ctx.period, ctx.shapes, ctx.dtype = scales, counts is not None, period, [v.shape for v in values], first.dtype
        return out

    @staticmethod
    def backward(ctx: Any, grad):
        saved, wanted, layers = ctx.saved_tensors, ctx.needs_input_grad[2:], len(ctx.shapes)
        grad = grad.float().contiguous()
        if torch.is_grad_enabled() or not _has_memory(grad):   # differentiated itself, or over a batch of gradients
            by = [scale if ctx.counted else 2 * scale for scale in ctx.scales]
            return (None, None, *((grad[l] * by[l] * saved[l].float()).to(ctx.dtype).expand(ctx.shapes[l]) if wanted[l] else None
                                  for l in range(layers)))
        saved = [t.contiguous() for t in saved]
        grads = [torch.empty(shape, dtype=ctx.dtype, device=grad.device) if want else None for shape, want in zip(ctx.shapes, wanted)]
        with _lib.device_of(grad):
            if layers == 1:
                values, counts = (None, _lib.ptr(saved[0])) if ctx.counted else (_lib.ptr(saved[0]), None)
                rc = _lib.lib.mbx_loss_gradient(_lib.ptr(grad), values, _lib.DTYPE[ctx.dtype], counts, ctx.shapes[0].numel(), ctx.period, ctx.scales[0],
                                                _lib.ptr(grads[0]), _lib.stream())
            else:
                pointers = LossSums._pointers(saved)
                values, counts = (None, pointers) if ctx.counted else (pointers, None)
                rc = _lib.lib.mbx_loss_gradients(_lib.ptr(grad), values, _lib.DTYPE[ctx.dtype], counts,
                                                 *LossSums._arrays([s.numel() for s in ctx.shapes], ctx.scales), layers, ctx.period,
                                                 LossSums._pointers(grads), _lib.stream())
            _lib.check(rc, 'loss_gradients')
        return (None, None, *grads)


def clear_router_zloss():
    _ROUTER_LOGITS.clear()


def batched_router_zloss(args: Arguments):
    """router.py:25-42: weight * mean(logsumexp(logits)^2) per router."""
    if args.moe_zloss_weight == 0:
        import warnings
        warnings.warn('Call to batched_router_zloss, but moe_zloss_weight=0')
        return 0
    if _ROUTER_LOGITS and all(lse is not None and (args.moe_zloss_in_fp32 or logits.dtype == torch.float32) for logits, lse in _ROUTER_LOGITS) and \
            LossSums.takes([lse for _, lse in _ROUTER_LOGITS], None):
        return LossSums.apply([args.moe_zloss_weight / lse.numel() for _, lse in _ROUTER_LOGITS], None, *(lse for _, lse in _ROUTER_LOGITS))
    terms = []
    for logits, lse in _ROUTER_LOGITS:
        if lse is None:
            lse = torch.logsumexp(logits.float() if args.moe_zloss_in_fp32 else logits, dim=1)
        elif not args.moe_zloss_in_fp32:
            lse = lse.to(logits.dtype)     # what torch.logsumexp returns for 16-bit logits: computed in fp32, rounded
        terms.append(lse.square().mean())
    return args.moe_zloss_weight * torch.stack(terms)


class _UniformExpertAssignment(torch.autograd.Function):

    @staticmethod
    def forward(ctx: Any, x: torch.Tensor, num_experts: int):
        out = torch.arange(x.numel(), dtype=x.dtype, device=x.device)
        return torch.remainder(out, num_experts).view(x.shape)


class _RouterLinear(torch.autograd.Function):
    """`x @ weight^T` of the router's `torch.nn.Linear` (router.py:96) with the gradients from the grouped kernels: the
    weight's, `[E, T] @ [T, h]` (a short, wide output over a reduction as long as the batch: a handful of tiles for the
    vendor GEMM), by the TN kernel over equal pieces of the token range, one group each, whose fp32 sums one kernel adds up
    and rounds; the input's, a reduction of E, by the NN kernel.  (GPU, 16384 tokens of 1024, 64 experts: weight 14 + 10 + 5 -> 14 + 5 us,
    input 18 -> 14; the backward's host time with the router kernel's 102 -> 81 us.  At 600 tokens, where the vendor's
    two products are as quick, a node of Python's in the forward is 5 us more than torch's own: from 1024 tokens.)"""

    PIECE_ROWS = 256   # tokens per piece (four K tiles of the TN kernel)
    MAX_PIECES = 64
    MAX_KEPT = 4096    # batch sizes; a captured graph may hold the bins of any of them, so none is given up for another

    _sizes = {}

    @staticmethod
    def piece_sizes(tokens: int) -> torch.Tensor:
        """Rows per piece (kept for the first MAX_KEPT batch sizes: the grouped GEMM caches the device-side bins on this tensor)."""
        sizes = _RouterLinear._sizes.get(tokens)
        if sizes is None:
            pieces = max(1, min(_RouterLinear.MAX_PIECES, tokens // _RouterLinear.PIECE_ROWS))
            sizes = torch.full((pieces,), tokens // pieces, dtype=torch.int64)
            sizes[:tokens % pieces] += 1
            if len(_RouterLinear._sizes) < _RouterLinear.MAX_KEPT:
                _RouterLinear._sizes[tokens] = sizes
        return sizes

    @staticmethod
    def whole_batch(sizes: torch.Tensor, tokens: int, device) -> torch.Tensor:
        """The pieces as one group, whose bin on the device is the last of theirs: a batch size met for the first time is
        copied there once (a copy waits for the queue to drain)."""
        whole = getattr(sizes, '_mbx_whole', None)
        if whole is None:
            from megablocks_amd import grouped_gemm_util as gg
            whole = sizes._mbx_whole = torch.tensor([tokens])
            gg._remember(whole, (gg._device_bins(sizes, device, tokens)[-1:], whole._version, tokens))
        return whole

    @staticmethod
    @torch.amp.custom_fwd(device_type='cuda')
    def forward(ctx: Any, x: torch.Tensor, weight: torch.Tensor):
        # Under autocast the product runs in x's 16-bit type, as torch's own linear would; the cast weight is
        # what the backward multiplies with, and the weight gradient goes back in the parameter's type (fp32
        # master weights).  Outside autocast mismatched types are an error, as for torch.nn.Linear.
        ctx.weight_dtype = weight.dtype
        if weight.dtype != x.dtype and torch.is_autocast_enabled():
            weight = weight.to(x.dtype)
        ctx.save_for_backward(x, weight)
        return torch.nn.functional.linear(x, weight)

    @staticmethod
    @torch.amp.custom_bwd(device_type='cuda')
    def backward(ctx: Any, grad: torch.Tensor):
        x, weight = ctx.saved_tensors
        return _linear_gradients(grad.to(x.dtype), x, weight, ctx.weight_dtype, *ctx.needs_input_grad[:2])


class _RouterLinearAndTokens(torch.autograd.Function):
    """_RouterLinear that hands out its input a second time, for the experts: their gradient of it comes back to this node, which adds the linear
    layer's where it forms it (`mbx_router_input_gradient`) instead of leaving two gradients of the input to be added up.  (16384 tokens of 1024, 64
    experts, GPU: product 17.5 and addition 17.5 -> 17 us; of 768, 32 experts: 18.3 and 12.5 -> 12.)"""

    @staticmethod
    @torch.amp.custom_fwd(device_type='cuda')
    def forward(ctx: Any, x: torch.Tensor, weight: torch.Tensor):
        logits = _RouterLinear.forward(ctx, x, weight)
        ctx.set_materialize_grads(False)
        return logits, x.detach()

    @staticmethod
    @torch.amp.custom_bwd(device_type='cuda')
    def backward(ctx: Any, grad: torch.Tensor, grad_tokens: torch.Tensor):
        x, weight = ctx.saved_tensors
        want_x, want_weight = ctx.needs_input_grad[:2]
        if grad is None:
            return grad_tokens, None
        grad = grad.to(x.dtype)
        tokens, experts = grad.shape
        padded = torch.empty((tokens, experts + -experts % 8), dtype=grad.dtype, device=grad.device) if want_weight and experts % 8 else None
        dx = _input_gradient_on(grad_tokens, grad, weight, padded) if want_x and grad_tokens is not None else None
        fused = dx is not None
        plain, dw = _linear_gradients(grad, x, weight, ctx.weight_dtype, want_x and not fused, want_weight, padded if fused else None)
        if not fused and want_x:
            dx = plain if grad_tokens is None else plain + grad_tokens
        return dx, dw


def _input_gradient_on(other, grad, weight, padded=None):
    """other + grad @ weight, in one pass over `other`, rounded once; None where the kernel does not take the call.  padded: gets `grad` with zeros up to
    a multiple of 8 columns."""
    if torch.is_grad_enabled() or not all(type(t) is torch.Tensor and _has_memory(t) for t in (other, grad)):
        return None
    tokens, experts = grad.shape
    if not (other.is_cuda and other.dtype == grad.dtype == weight.dtype and other.dtype in (torch.bfloat16, torch.float16) and experts <= 128 and
            other.shape == (tokens, weight.shape[1]) and _whole_pieces(other) and weight.is_contiguous()):
        return None
    grad, out = grad.contiguous(), torch.empty_like(other)
    with _lib.device_of(other):
        _lib.check(_lib.lib.mbx_router_input_gradient(_lib.ptr(grad), _lib.ptr(weight), _lib.ptr(other), _lib.dtype_of(other), tokens, other.shape[1],
                                                      experts, _lib.ptr(out), _lib.ptr(padded), _lib.stream()), 'router_input_gradient')
    return out


def _whole_pieces(t: torch.Tensor) -> bool:
    return t.shape[1] % 8 == 0 and t.is_contiguous() and t.data_ptr() % 16 == 0


def _has_memory(t: torch.Tensor) -> bool:
    try:
        t.data_ptr()
    except RuntimeError:
        return False
    return True


def _linear_gradients(grad, x, weight, weight_dtype, want_x, want_weight, padded=None):
    """(dx, dweight) of `x @ weight^T`, all 16-bit of one type on the GPU; dweight in `weight_dtype`.  padded: `grad` with zeros up to a multiple of
    8 experts, where the caller has it."""
    from megablocks_amd import grouped_gemm_util as gg
    if torch.is_grad_enabled() or not _has_memory(grad):
        # a backward that is differentiated itself (create_graph), or runs over a batch of gradients at once (is_grads_batched)
        return grad @ weight if want_x else None, (grad.t() @ x).to(weight_dtype) if want_weight else None
    tokens, experts = grad.shape
    grad = grad.contiguous()
    dx = dw = None
    sizes = _RouterLinear.piece_sizes(tokens) if want_weight else None
    if want_x:
        # the grouped kernels for whole 16-byte pieces of rows; the input's gradient alone is not worth the copy of a bin
        grouped = sizes is not None and tokens > 0 and _whole_pieces(grad) and _whole_pieces(weight)
        dx = gg.gmm(grad, weight.unsqueeze(0), _RouterLinear.whole_batch(sizes, tokens, x.device), _record_as='router_dgrad') \
            if grouped else grad @ weight
    if want_weight:
        pieces = sizes.shape[0]
        if experts % 8:
            grad = torch.nn.functional.pad(grad, (0, -experts % 8)) if padded is None else padded
        # [pieces, E, h]; a single piece's sums are rounded by the product itself
        parts = gg.weight_gradient(grad, x.contiguous(), sizes, torch.float32 if pieces > 1 else None, _record_as='router_wgrad')
        if pieces == 1 or parts.dtype != torch.float32:
            dw = (parts[0] if pieces == 1 else parts.sum(0, dtype=torch.float32))[:experts].to(weight_dtype)
        else:
            dw = torch.empty((experts, x.shape[1]), dtype=weight_dtype, device=x.device)
            with _lib.device_of(x):
                _lib.check(_lib.lib.mbx_sum_parts(_lib.ptr(parts), pieces, parts.stride(0), _lib.ptr(dw), _lib.dtype_of(dw),
                                                  dw.numel(), _lib.stream()), 'sum_parts')
    return dx, dw


class _SoftmaxTopK(torch.autograd.Function):
    """softmax -> top-k -> optional p-norm renormalisation (router.py:87-106) as one kernel each way.
    Returns (scores, expert_weights, expert_indices, expert_indices as int32, lse) with torch's shapes and dtypes (int64
    indices); the int32 copy, written by the same kernel, is what the layer's routing takes (moe.py:160 casts); lse
    (`want_lse`, else None) is logsumexp(logits, dim=1) in fp32, the term of the z-loss (router.py:37), which the
    backward kernel differentiates along with the rest."""

    @staticmethod
    def supported(logits: torch.Tensor, top_k: int) -> bool:
        return (logits.is_cuda and logits.ndim == 2 and logits.dtype in _lib.DTYPE and 0 < logits.shape[1] <= 512
                and 0 < top_k <= min(64, logits.shape[1]))

    @staticmethod
    def forward(ctx: Any, logits: torch.Tensor, top_k: int, norm_p: float, want_lse: bool = False):
        logits = logits.contiguous()
        tokens, experts = logits.shape
        scores = torch.empty_like(logits)
        weights = torch.empty((tokens, top_k), dtype=logits.dtype, device=logits.device)
        indices = torch.empty((tokens, top_k), dtype=torch.int64, device=logits.device)
        indices32 = torch.empty((tokens, top_k), dtype=torch.int32, device=logits.device)
        lse = torch.empty((tokens,), dtype=torch.float32, device=logits.device) if want_lse else None
        with _lib.device_of(logits):
            _lib.check(_lib.lib.mbx_router_forward(_lib.ptr(logits), _lib.dtype_of(logits), tokens, experts, top_k,
                                                   float(norm_p), _lib.ptr(scores), _lib.ptr(weights), _lib.ptr(indices),
                                                   _lib.ptr(indices32), _lib.ptr(lse), _lib.stream()), 'router_forward')
        ctx.save_for_backward(scores, indices)
        ctx.top_k, ctx.norm_p = top_k, float(norm_p)
        ctx.mark_non_differentiable(indices, indices32)
        # an output nobody differentiates (the scores without a load-balancing loss, lse without a z-loss, the indices)
        # arrives in backward as None instead of a zero-filled tensor: three fill launches less per step
        ctx.set_materialize_grads(False)
        return scores, weights, indices, indices32, lse

    @staticmethod
    def backward(ctx: Any, grad_scores, grad_weights, _grad_indices, _grad_indices32, grad_lse):
        scores, indices = ctx.saved_tensors
        return _logits_gradient(scores, indices, ctx.top_k, ctx.norm_p, grad_scores, grad_weights, grad_lse), None, None, None


def _logits_gradient(scores, indices, top_k, norm_p, grad_scores, grad_weights, grad_lse=None):
    """The gradient of the logits behind _SoftmaxTopK's outputs (`mbx_router_backward`); the outputs' may be None."""
    tokens, experts = scores.shape
    grad_logits = torch.empty_like(scores)
    gs = None if grad_scores is None else grad_scores.to(scores.dtype).contiguous()
    gw = None if grad_weights is None else grad_weights.to(scores.dtype).contiguous()
    gl = None if grad_lse is None else grad_lse.float().contiguous()
    with _lib.device_of(scores):
        _lib.check(_lib.lib.mbx_router_backward(_lib.ptr(gw), _lib.ptr(gs), _lib.ptr(scores), _lib.ptr(indices),
                                                _lib.dtype_of(scores), tokens, experts, top_k, norm_p,
                                                _lib.ptr(grad_logits), _lib.ptr(gl), _lib.stream()), 'router_backward')
    return grad_logits


class _LinearSoftmaxTopK(torch.autograd.Function):
    """The router's linear layer and _SoftmaxTopK's forward as one kernel, where no gradient is recorded: returns (scores,
    expert_weights, expert_indices, expert_indices as int32)."""

    MAX_TOKENS = 256           # one workgroup per token: all at once
    MAX_WEIGHTS = 1 << 18      # elements: every workgroup reads them all

    @staticmethod
    def supported(x: torch.Tensor, layer: torch.nn.Module, top_k: int) -> bool:
        return not torch.is_grad_enabled() and _LinearSoftmaxTopK.fits(x, layer, top_k)

    @staticmethod
    def fits(x: torch.Tensor, layer: torch.nn.Module, top_k: int) -> bool:
        """Few tokens and a small layer: one launch instead of two (64 experts of 2048, 5 tokens: 11.1 -> 9.1 us on the GPU, and
        the vendor library's call alone is 25 us of host time; 512 tokens: 11.5 against 14.5, 128 experts of 4096: 14.0
        against 16.1)."""
        if type(layer) is not torch.nn.Linear or not x.is_cuda or x.shape[0] > _LinearSoftmaxTopK.MAX_TOKENS:
            return False
        weight = layer.weight
        return (x.dtype in (torch.bfloat16, torch.float16) and type(weight) is torch.nn.Parameter and weight.dtype == x.dtype and
                weight.device == x.device and layer.bias is None and x.shape[0] > 0 and x.shape[1] == weight.shape[1] and
                x.shape[1] % 8 == 0 and weight.shape[0] <= 128 and weight.numel() <= _LinearSoftmaxTopK.MAX_WEIGHTS and 0 < top_k <= min(64, weight.shape[0]) and
                x.is_contiguous() and weight.is_contiguous() and (x.data_ptr() | weight.data_ptr()) % 16 == 0 and
                not torch.is_autocast_enabled() and not _has_hooks(layer))

    @staticmethod
    def forward(ctx: Any, x: torch.Tensor, weight: torch.Tensor, top_k: int, norm_p: float):
        tokens, experts = x.shape[0], weight.shape[0]
        scores = torch.empty((tokens, experts), dtype=x.dtype, device=x.device)
        weights = torch.empty((tokens, top_k), dtype=x.dtype, device=x.device)
        indices = torch.empty((tokens, top_k), dtype=torch.int64, device=x.device)
        indices32 = torch.empty((tokens, top_k), dtype=torch.int32, device=x.device)
        with _lib.device_of(x):
            _lib.check(_lib.lib.mbx_router_linear_forward(
                _lib.ptr(x), _lib.ptr(weight), _lib.dtype_of(x), tokens, x.shape[1], experts, top_k, float(norm_p), _lib.ptr(scores),
                _lib.ptr(weights), _lib.ptr(indices), _lib.ptr(indices32), _lib.stream()), 'router_linear_forward')
        ctx.mark_non_differentiable(indices, indices32)
        return scores, weights, indices, indices32


class _RecordedLinearSoftmaxTopK(torch.autograd.Function):
    """_LinearSoftmaxTopK where gradients are recorded.  The kernel sums a logit in another order than the vendor's product,
    so both modes have to take it: a step that is recomputed (activation checkpointing runs the forward without gradients
    first) must choose the experts, and weigh them, as the pass whose output it belongs to did."""

    @staticmethod
    def supported(x: torch.Tensor, layer: torch.nn.Module, top_k: int) -> bool:
        return torch.is_grad_enabled() and _LinearSoftmaxTopK.fits(x, layer, top_k)

    @staticmethod
    def forward(ctx: Any, x: torch.Tensor, weight: torch.Tensor, top_k: int, norm_p: float):
        scores, weights, indices, indices32 = _LinearSoftmaxTopK.forward(ctx, x, weight, top_k, norm_p)
        ctx.save_for_backward(x, weight, scores, indices)
        ctx.top_k, ctx.norm_p = top_k, float(norm_p)
        ctx.set_materialize_grads(False)
        return scores, weights, indices, indices32

    @staticmethod
    def backward(ctx: Any, grad_scores, grad_weights, _grad_indices, _grad_indices32):
        x, weight, scores, indices = ctx.saved_tensors
        grad = _logits_gradient(scores, indices, ctx.top_k, ctx.norm_p, grad_scores, grad_weights)
        # so few tokens: the vendor's two products, which need nothing from the host at a token count not met before (a capture
        # of such a step needs no eager one first) and are shorter on the GPU (out of a graph, 16 - 256 tokens: 8.3 - 10.2 us, the
        # grouped ones 10.3 - 12.6; their calls cost 39 us of host time and those 25)
        dx = grad @ weight if ctx.needs_input_grad[0] else None
        dw = grad.t() @ x if ctx.needs_input_grad[1] else None
        return dx, dw, None, None


def _has_hooks(module: torch.nn.Module) -> bool:
    """Whether calling `module` would run more than its forward (or its forward has been replaced on the object)."""
    glob = torch.nn.modules.module
    return bool(module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks or
                glob._global_forward_hooks or glob._global_forward_pre_hooks or glob._global_backward_hooks or
                glob._global_backward_pre_hooks or 'forward' in module.__dict__)


def int32_indices(expert_indices: torch.Tensor) -> torch.Tensor:
    """The int32 copy LearnedRouter.forward attached to its indices, if `expert_indices` still is that tensor with
    that content; else `expert_indices` itself (the routing then casts, as moe.py:160 does)."""
    attached = getattr(expert_indices, '_mbx_int32', None)
    if attached is not None and attached[1] == expert_indices._version and attached[0].shape == expert_indices.shape:
        return attached[0]
    return expert_indices


class LearnedRouter(torch.nn.Module):

    def __init__(self, args: Arguments):
        super().__init__()
        self.args = args
        self.layer = torch.nn.Linear(args.hidden_size, args.moe_num_experts, bias=False, dtype=common.dtype(args),
                                     device=args.device)
        args.init_method(self.layer.weight)

    def jitter(self, x: torch.Tensor):
        low = 1.0 - self.args.moe_jitter_eps
        high = 1.0 + self.args.moe_jitter_eps
        noise = torch.rand(x.size(), dtype=x.dtype, device=x.device)
        return low + noise * (high - low)

    def _top_k(self, scores: torch.Tensor):
        if self.args.moe_top_k == 1:
            return scores.max(dim=-1, keepdim=True)
        return torch.topk(scores, self.args.moe_top_k, dim=-1)

    def forward(self, x: torch.Tensor):
        scores, expert_weights, expert_indices, expert_indices32 = self.route(x)
        if expert_indices32 is not None:
            # out of band: the same indices as int32, valid while the int64 tensor is the one returned here, unmodified
            expert_indices._mbx_int32 = (expert_indices32, expert_indices._version)
        return scores, expert_weights, expert_indices

    def shares(self, x: torch.Tensor) -> bool:
        """Whether forward_and_tokens may stand for calling the module: forward would do nothing else, and both gradients of x are 16-bit rows on
        the GPU."""
        return (type(self) is LearnedRouter and torch.is_grad_enabled() and type(x) is torch.Tensor and x.requires_grad and self._takes_linear(x) and
                (not self.training or self.args.moe_jitter_eps is None) and not _has_hooks(self) and
                self.__dict__.keys().isdisjoint(('route', '_top_k', 'jitter')) and common.only_computed(autocast=True))

    def forward_and_tokens(self, x: torch.Tensor):
        """forward(x), and x again for the experts: their gradient of it comes back through the router's (_RouterLinearAndTokens)."""
        tokens = None

        def linear(x2d, weight):
            nonlocal tokens
            logits, tokens = _RouterLinearAndTokens.apply(x2d, weight)
            return logits

        scores, expert_weights, expert_indices, expert_indices32 = self.route(x, linear)
        if expert_indices32 is not None:   # as in forward
            expert_indices._mbx_int32 = (expert_indices32, expert_indices._version)
        return scores, expert_weights, expert_indices, x if tokens is None else tokens.view(x.shape)

    @staticmethod
    def _takes_linear(x: torch.Tensor) -> bool:
        return x.is_cuda and x.dtype in (torch.bfloat16, torch.float16) and x.numel() >= 4 * _RouterLinear.PIECE_ROWS * x.shape[-1]

    def route(self, x: torch.Tensor, linear=_RouterLinear.apply):
        """forward's (scores, expert_weights, expert_indices) and, where the router kernel wrote them, the indices as
        int32 (else None): the layer routes with those and skips the cast of moe.py:160.  linear: what forms the logits of more than a few
        16-bit rows on the GPU."""
        if self.training and self.args.moe_jitter_eps is not None:
            x = x * self.jitter(x)
        x2d = x.view(-1, x.shape[-1])
        args = self.args
        if FUSED_SOFTMAX_TOPK and args.moe_zloss_weight == 0 and not args.uniform_expert_assignment:
            for node in (_LinearSoftmaxTopK, _RecordedLinearSoftmaxTopK):   # without gradients, with
                if node.supported(x2d, self.layer, args.moe_top_k):
                    return node.apply(x2d, self.layer.weight, args.moe_top_k, args.moe_normalize_expert_weights or 0)
        if self._takes_linear(x2d):
            logits = linear(x2d, self.layer.weight)
        else:
            logits = self.layer(x2d)
        saved_logits, lse = logits, None
        if logits.is_cuda and logits.dtype != torch.float32 and torch.is_autocast_enabled():
            # autocast runs softmax in fp32 (router.py:98 under torch.autocast): scores and weights come out in fp32
            logits = logits.float()
        expert_indices32 = None
        if FUSED_SOFTMAX_TOPK and _SoftmaxTopK.supported(logits, self.args.moe_top_k):
            scores, expert_weights, expert_indices, expert_indices32, lse = _SoftmaxTopK.apply(
                logits, self.args.moe_top_k, self.args.moe_normalize_expert_weights or 0,
                self.args.moe_zloss_weight != 0)
        else:
            scores = logits.softmax(dim=-1)
            expert_weights, expert_indices = self._top_k(scores)
            if self.args.moe_normalize_expert_weights:
                expert_weights = expert_weights / torch.norm(
                    expert_weights, p=self.args.moe_normalize_expert_weights, dim=-1, keepdim=True)
        _save_router_logits(saved_logits, self.args, lse)
        if self.args.uniform_expert_assignment:
            expert_indices = _UniformExpertAssignment.apply(expert_indices, self.args.moe_num_experts)
            expert_indices32 = None
        return scores, expert_weights, expert_indices, expert_indices32
