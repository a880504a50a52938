"""When the dropless layer's forward without gradients is left to the separate calls (megablocks/layers/dmoe.py:239-280), without a
GPU: the call of the library is replaced by a mark."""
import contextlib

import pytest
import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from megablocks_amd import grouped_gemm_util as gg
from megablocks_amd.layers import dmoe
from megablocks_amd.layers.arguments import Arguments

TOKENS, HIDDEN, EXPERTS, TOP_K = 5, 16, 4, 2


class _Layer(dmoe.ParallelDroplessMLP):
    pass


def _layer(cls=dmoe.ParallelDroplessMLP, **kw):
    base = dict(hidden_size=HIDDEN, ffn_hidden_size=32, moe_num_experts=EXPERTS, moe_top_k=TOP_K, bias=False, fp16=False, bf16=True,
                device=torch.device('cpu'), mlp_impl='grouped')
    return cls(Arguments(**{**base, **kw}))


@pytest.fixture
def called(monkeypatch):
    calls = []

    def experts_forward(x, ids, weights, *args):
        calls.append(args)
        return x, ids
    monkeypatch.setattr(gg, 'experts_forward', experts_forward)
    return calls


def _inputs():
    return (torch.randn(TOKENS, 1, HIDDEN).bfloat16(), torch.rand(TOKENS * TOP_K).bfloat16(),
            torch.randint(EXPERTS, (TOKENS * TOP_K,)))


@pytest.mark.parametrize('kw', [dict(), dict(mlp_type='glu', activation_fn=F.silu), dict(memory_optimized_mlp=True)])
def test_the_built_in_layer_is_one_call(called, kw):
    with torch.no_grad():
        assert _layer(**kw)._one_call_forward(*_inputs()) is not None
    assert len(called) == 1


def _patched(name):
    def patch(layer):
        setattr(layer, name, getattr(layer, name))
    return patch


def _other_experts(layer):
    layer.mlp.__class__ = type('Experts', (type(layer.mlp),), {})


def _scaled(layer):
    layer.mlp.gradient_scale = 0.5


def _experts_patched(layer):
    layer.mlp.forward_tokens = layer.mlp.forward_tokens


@pytest.mark.parametrize('change', [_patched('indices_and_bins'), _patched('grouped_permute_and_compute'), _patched('permute_and_compute'),
                                    _other_experts, _scaled, _experts_patched])
def test_other_layers_and_experts_are_not(called, change):
    layer = _layer()
    change(layer)
    with torch.no_grad():
        assert layer._one_call_forward(*_inputs()) is None
    assert not called


@pytest.mark.parametrize('kw', [dict(cls=_Layer), dict(activation_fn=F.relu), dict(mlp_type='glu', activation_fn=F.relu)])
def test_layers_of_other_classes_and_activations_are_not(called, kw):
    with torch.no_grad():
        assert _layer(**kw)._one_call_forward(*_inputs()) is None
    assert not called


@contextlib.contextmanager
def _autocast():
    torch.set_autocast_enabled('cuda', True)
    try:
        yield
    finally:
        torch.set_autocast_enabled('cuda', False)


@pytest.mark.parametrize('context', [_autocast, forward_ad.dual_level])
def test_a_cast_or_dual_pass_is_not(called, context):
    layer = _layer()
    with torch.no_grad(), context():
        assert layer._one_call_forward(*_inputs()) is None
    assert not called


def test_a_compiled_pass_is_not(monkeypatch, called):
    monkeypatch.setattr(torch.compiler, 'is_compiling', lambda: True)
    with torch.no_grad():
        assert _layer()._one_call_forward(*_inputs()) is None
    assert not called


def _traced(f, x):
    torch.jit.trace(f, x, check_trace=False)


def _vmapped(f, x):
    torch.func.vmap(f)(x[None])


def _jvp(f, x):
    torch.func.jvp(f, (x,), (x,))


def _functional(f, x):
    torch.func.functionalize(f)(x)


@pytest.mark.parametrize('transform', [_traced, _vmapped, _jvp, _functional])
@pytest.mark.filterwarnings('ignore')
def test_a_traced_or_transformed_pass_is_not(called, transform):
    layer, (x, weights, ids) = _layer(), _inputs()
    results = []

    def f(t):
        results.append(layer._one_call_forward(t, weights, ids))
        return t * 2
    with torch.no_grad():
        transform(f, x)
    assert results and all(r is None for r in results) and not called


@pytest.mark.parametrize('owner,name', [(torch._C, '_are_functorch_transforms_active'), (forward_ad, '_current_level')])
def test_a_torch_that_does_not_say_takes_the_separate_calls(monkeypatch, called, owner, name):
    layer = _layer()
    with monkeypatch.context() as m:
        m.delattr(owner, name)
        assert not dmoe._only_computed()
        with torch.no_grad():
            assert layer._one_call_forward(*_inputs()) is None
    assert not called and dmoe._only_computed()


@pytest.fixture
def stepped(monkeypatch):
    calls = []

    def experts_step(x, ids, weights, *args):
        calls.append(args)
        return x, ids
    monkeypatch.setattr(gg, 'experts_step', experts_step)
    return calls


@pytest.mark.parametrize('kw', [dict(), dict(mlp_type='glu', activation_fn=F.silu)])
@pytest.mark.parametrize('context', [contextlib.nullcontext, _autocast])
def test_the_built_in_layers_step_is_one_call(stepped, kw, context):
    with context():
        assert _layer(**kw)._one_call_step(*_inputs()) is not None
    assert len(stepped) == 1


def _hooked(layer):
    layer.mlp.register_forward_hook(lambda *_: None)


def _frozen(layer):
    layer.requires_grad_(False)


@pytest.mark.parametrize('change', [_patched('indices_and_bins'), _patched('grouped_permute_and_compute'), _other_experts, _scaled, _experts_patched,
                                    _hooked, _frozen])
def test_other_layers_steps_are_not(stepped, change):
    layer = _layer()
    change(layer)
    assert layer._one_call_step(*_inputs()) is None
    assert not stepped


@pytest.mark.parametrize('kw', [dict(cls=_Layer), dict(activation_fn=F.relu), dict(memory_optimized_mlp=True)])
def test_steps_of_other_classes_and_activations_and_memory_optimized_ones_without_all_gradients_are_not(stepped, kw):
    assert _layer(**kw)._one_call_step(*_inputs()) is None
    assert not stepped


@pytest.mark.parametrize('transform', [_traced, _vmapped, _jvp, _functional])
@pytest.mark.filterwarnings('ignore')
def test_a_traced_or_transformed_step_is_not(stepped, transform):
    layer, (x, weights, ids) = _layer(), _inputs()
    results = []

    def f(t):
        results.append(layer._one_call_step(t, weights, ids))
        return t * 2
    transform(f, x)
    assert results and all(r is None for r in results) and not stepped
