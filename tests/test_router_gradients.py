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
