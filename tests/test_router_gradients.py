"""Which products the gradients of the router's linear layer are formed by (megablocks/layers/router.py:96), without a GPU."""
import types

import pytest
import torch

from megablocks_amd import grouped_gemm_util as gg
from megablocks_amd.layers import router as r


@pytest.fixture
def no_grouped_products(monkeypatch):
    def refuse(*args, **kwargs):
        raise AssertionError('a grouped product')
    monkeypatch.setattr(gg, 'gmm', refuse)
    monkeypatch.setattr(gg, 'weight_gradient', refuse)


@pytest.fixture
def launched(monkeypatch):
    """The grouped products as plain ones: (layout, bins as they reach the kernel) of each."""
    calls = []

    def gmm(a, b, batch_sizes, trans_a=False, _record_as=None, **_):
        bins = gg._device_bins(batch_sizes, a.device, a.shape[0])
        calls.append(('tn' if trans_a else 'nn', bins.tolist()))
        if not trans_a:
            return (a.double() @ b[0].double()).to(a.dtype)
        cuts = bins[:-1].long()
        return torch.stack([(p.double().t() @ q.double()).to(a.dtype) for p, q in zip(a.tensor_split(cuts), b.tensor_split(cuts))])
    monkeypatch.setattr(gg, 'gmm', gmm)
    monkeypatch.setattr(gg, 'weight_gradient', lambda a, b, sizes, weight_dtype=None, **_: gmm(a, b, sizes, trans_a=True))
    monkeypatch.setattr(r._RouterLinear, '_sizes', {})
    return calls


@pytest.fixture
def copies(monkeypatch):
    """The batch sizes whose bins are copied to the device (`_device_bins` finds none kept)."""
    made = []
    cumsum = torch.cumsum
    monkeypatch.setattr(torch, 'cumsum', lambda t, *a, **k: made.append(t.tolist()) or cumsum(t, *a, **k))
    return made


def _operands(tokens, hidden, experts, dtype=torch.bfloat16):
    torch.manual_seed(tokens)
    return [torch.randn(*s).to(dtype) for s in ((tokens, hidden), (experts, hidden), (tokens, experts))]


@pytest.mark.parametrize('want', [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize('tokens', [1, 41, 256])
def test_gradients_of_a_few_tokens_are_the_two_plain_products(monkeypatch, no_grouped_products, tokens, want):
    """Up to 256 tokens, where the linear layer is part of the router kernel, a token count that comes up for the first time makes
    nothing on the host and copies nothing to the device (which a capture would refuse)."""
    x, weight, grad = _operands(tokens, 24, 8)
    monkeypatch.setattr(r, '_logits_gradient', lambda *a: grad)
    monkeypatch.setattr(r._RouterLinear, 'piece_sizes', None)
    ctx = types.SimpleNamespace(saved_tensors=(x, weight, None, None), top_k=1, norm_p=0.0, needs_input_grad=(*want, False, False))
    dx, dw, *rest = r._RecordedLinearSoftmaxTopK.backward(ctx, None, None, None, None)
    assert rest == [None, None] and (dx is not None, dw is not None) == want
    assert dx is None or torch.equal(dx, grad @ weight)
    assert dw is None or torch.equal(dw, grad.t() @ x)


@torch.no_grad()   # as a backward runs
def test_a_batch_size_is_copied_to_the_device_once(launched, copies):
    """One copy for both gradients at the first batch of a size, none for later ones, and none at all where only the input's
    gradient is wanted."""
    x, weight, grad = _operands(1100, 16, 8)
    dx, _ = r._linear_gradients(grad, x, weight, weight.dtype, True, False)
    assert not copies and torch.equal(dx, grad @ weight)
    for _ in range(2):
        r._linear_gradients(grad, x, weight, weight.dtype, True, True)
    assert copies == [[275] * 4]
    assert launched == 2 * [('nn', [1100]), ('tn', [275, 550, 825, 1100])]


@torch.no_grad()
def test_batch_sizes_are_kept_up_to_a_bound(monkeypatch, launched, copies):
    """Sizes past the bound are worked out anew each time; those kept stay, as graphs may hold them."""
    monkeypatch.setattr(r._RouterLinear, 'MAX_KEPT', 2, raising=False)
    for tokens in (1024, 1100, 1200, 1300, 1024, 1200):
        x, weight, grad = _operands(tokens, 16, 8)
        r._linear_gradients(grad, x, weight, weight.dtype, True, True)
    assert len(r._RouterLinear._sizes) == 2
    assert [sum(c) for c in copies] == [1024, 1100, 1200, 1300, 1200]


@pytest.mark.parametrize('form', ['hidden', 'experts', 'weight_offset', 'weight_strided', 'grad_offset'])
@torch.no_grad()
def test_rows_that_are_no_whole_pieces_leave_the_input_gradient_to_the_plain_product(launched, form):
    """The grouped product serves whole aligned 16-byte pieces of rows; others it would give to the element-wise kernel."""
    tokens, hidden, experts = 1100, 70 if form == 'hidden' else 72, 12 if form == 'experts' else 16
    x, weight, grad = _operands(tokens, hidden, experts)
    if form == 'weight_offset':
        weight = torch.cat([weight.new_zeros(1), weight.flatten()])[1:].view(experts, hidden)
    elif form == 'weight_strided':
        weight = weight.t().contiguous().t()
    elif form == 'grad_offset':
        grad = torch.cat([grad.new_zeros(1), grad.flatten()])[1:].view(tokens, experts)
    dx, dw = r._linear_gradients(grad, x, weight, weight.dtype, True, True)
    assert torch.equal(dx, grad @ weight) and [c[0] for c in launched] == ['tn']
    assert (dw.double() - grad.double().t() @ x.double()).norm() < 2.0 ** -7 * dw.double().norm()


def _linear(x, weight):
    return r._RouterLinear.apply(x, weight)


def test_gradients_of_the_linear_layer_can_be_differentiated(launched):
    """Under create_graph the backward is made of products autograd knows: second derivatives are those of torch's own linear."""
    x, weight, grad = (t.requires_grad_(True) for t in _operands(1100, 16, 8, torch.float64))

    def second(linear):
        launched.clear()
        dx, dw = torch.autograd.grad(linear(x, weight).tanh(), [x, weight], grad, create_graph=True)
        assert not launched
        return torch.autograd.grad([dx.square().sum(), dw.square().sum()], [x, weight, grad])
    for got, want in zip(second(_linear), second(torch.nn.functional.linear)):
        # the second pass adds four pieces' products in fp32
        torch.testing.assert_close(got, want, rtol=0, atol=4 * 2.0 ** -24 * float(want.abs().max()) * 4)


def test_gradients_of_the_linear_layer_over_a_batch_of_gradients(no_grouped_products):
    """is_grads_batched hands the backward a tensor without memory of its own."""
    x, weight, _ = (t.requires_grad_(True) for t in _operands(1100, 16, 8, torch.float64))
    grads = torch.randn(3, 1100, 8, dtype=torch.float64)
    for wanted in ([x], [weight], [x, weight]):
        for got, want in zip(*(torch.autograd.grad(linear(x, weight), wanted, grads, is_grads_batched=True)
                               for linear in (_linear, torch.nn.functional.linear))):
            torch.testing.assert_close(got, want)
