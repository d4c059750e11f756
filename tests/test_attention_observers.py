"""Whoever looks at the modules of the attention keeps seeing what passes through them: hooks, subclasses and replaced methods of
the softmax module, hooks on ``CoreAttention`` in a layer with cached positions, dispatch modes,
tracers and compilers. On the CPU."""
import types

import pytest
import torch

from megatron.model import fused_attention
from megatron.model.attention_core import CoreAttention
from megatron.model.fused_softmax import FusedScaleMaskSoftmax
from megatron.model.fused_softmax import SoftmaxFusionTypes as T
from oracle import fallback_semantics as fb


class Quiet(FusedScaleMaskSoftmax):
    def forward(self, input, mask, bias=None, key_lengths=None):
        return super().forward(input, mask, bias, key_lengths) * 0.5


def core(**kw):
    return CoreAttention(64, 1, False, True, T.upper_triang, fb.fill_masked_with_dtype_min, attention_softmax_in_fp32=True, **kw)


def scale(c):
    """What the attention kernels would scale the scores by, None where ``c`` takes the products."""
    return c._plain_scale(fb.causal_mask(8), None)


def subclass(c):
    c.scale_mask_softmax.__class__ = Quiet


def another_module(c):
    c.scale_mask_softmax = torch.nn.Identity()


WATCHERS = {
    "forward hook": lambda c: c.scale_mask_softmax.register_forward_hook(lambda m, i, o: None),
    "forward pre-hook": lambda c: c.scale_mask_softmax.register_forward_pre_hook(lambda m, i: None),
    "backward hook": lambda c: c.scale_mask_softmax.register_full_backward_hook(lambda m, i, o: None),
    "backward pre-hook": lambda c: c.scale_mask_softmax.register_full_backward_pre_hook(lambda m, g: None),
    "hook on every module": lambda c: torch.nn.modules.module.register_module_forward_hook(lambda m, i, o: None),
    "subclass": subclass,
    "another module": another_module,
    "replaced forward": lambda c: setattr(c.scale_mask_softmax, "forward", lambda *a, **k: None),
    "replaced branch": lambda c: setattr(c.scale_mask_softmax, "forward_fused_softmax", lambda *a, **k: None),
    "replaced gate": lambda c: setattr(c.scale_mask_softmax, "is_kernel_available", lambda *a: False),
}


@pytest.mark.parametrize("who", WATCHERS)
def test_a_watched_softmax_is_called(who):
    c = core()
    assert scale(c) == pytest.approx(0.125)
    handle = WATCHERS[who](c)
    try:
        assert scale(c) is None
    finally:
        if hasattr(handle, "remove"):
            handle.remove()
            assert scale(c) == pytest.approx(0.125)


def test_the_switch_for_tools_that_inspect_the_tensors():
    assert scale(core(causal_gemm_blocks=False)) is None


def cpu_attention(use_cache, num_kv_heads=None):
    from megatron.model.transformer_layer import SelfAttention

    args = types.SimpleNamespace(hidden_size=128, num_attention_heads=2, num_kv_heads=num_kv_heads, seq_length=16, precision="fp32",
                                 pos_emb="rotary", rotary_pct=1.0, rope_fusion=False, attention_softmax_in_fp32=False, attention_dropout=0.0,
                                 scaled_upper_triang_masked_softmax_fusion=False, scaled_masked_softmax_fusion=False)
    return SelfAttention(args, lambda s, m: s.masked_fill(m, -10000.0), 1, rotary=True, use_cache=use_cache)


def test_a_hook_on_the_attention_of_a_layer_with_cached_positions():
    """It fires once a step, with the keys of all positions and the context."""
    attention = cpu_attention(use_cache=True)
    seen = []
    attention.core.register_forward_hook(lambda module, inputs, out: seen.append((inputs[1].size(0), tuple(out.shape))))
    x, mask = torch.randn(5, 1, 128), fb.causal_mask(5)
    with torch.no_grad():
        (_, present), _ = attention(x[:4], mask[..., :4, :4])
        attention(x[4:], mask[..., 4:, :], layer_past=present)
    assert seen == [(4, (4, 1, 128)), (5, (1, 1, 128))]


def test_a_watched_attention_takes_no_step_of_its_own():
    c = core(use_cache=True)
    assert fused_attention.untouched(c, CoreAttention)
    for watch in (lambda: c.register_forward_hook(lambda m, i, o: None), lambda: c.register_forward_pre_hook(lambda m, i: None)):
        handle = watch()
        assert not fused_attention.untouched(c, CoreAttention)
        handle.remove()
    assert fused_attention.untouched(c, CoreAttention)
    c.forward = lambda *a, **k: None
    assert not fused_attention.untouched(c, CoreAttention)
    assert not fused_attention.untouched(type("Own", (CoreAttention,), {})(64, 1, False, True, T.none, None), CoreAttention)


def test_a_dispatch_mode_follows_what_is_done():
    """Launches past torch would escape it: a count of operations, a trace over real tensors."""
    from torch.utils.flop_counter import FlopCounterMode

    from megatron.fused_kernels import _hotpath

    t, c = torch.zeros(2), core()
    assert not _hotpath.followed(t) and scale(c) is not None
    with FlopCounterMode(display=False):
        assert _hotpath.followed(t) and scale(c) is None


@pytest.mark.parametrize("skip_bias_add", [False, True])
def test_a_linear_layer_can_be_traced_scripted_and_exported(skip_bias_add):
    from megatron.model.transformer_layer import Linear

    layer, x = Linear(64, 32, skip_bias_add=skip_bias_add), torch.randn(5, 64)
    want = layer(x)
    exported = torch.export.export(layer, (x,), dynamic_shapes={"x": {0: torch.export.Dim("rows", min=2, max=4096)}}).module()
    for other in (torch.fx.symbolic_trace(layer), torch.jit.script(layer), exported):
        for got, expected in zip(other(x), want):
            assert got is expected or torch.equal(got, expected)


@pytest.mark.parametrize("past", [None, 3])
def test_a_layer_attention_compiles_whole(past):
    attention = cpu_attention(use_cache=True, num_kv_heads=1).eval()
    cached = None if past is None else torch.randn(2, past, 1, 1, 64)
    args = torch.randn(4, 1, 128), torch.zeros((1, 1, 4, 4 + (past or 0)), dtype=torch.bool), cached
    with torch.no_grad():
        (want, want_present), _ = attention(*args)
        (got, present), _ = torch.compile(attention, fullgraph=True, backend="eager")(*args)
    assert torch.allclose(got, want, atol=1e-6) and torch.equal(present, want_present)


class OnGpu(torch.Tensor):
    """Says that it is on a GPU, for what is asked before the first launch."""
    is_cuda = True


class Launches:
    """Stands for the extension module."""

    def linear_act(self, x, *args):
        return x

    def linear_add(self, *args):
        return "one launch"


def few_rows():
    from megatron.model.transformer_layer import MLP

    mlp = MLP(types.SimpleNamespace(activation="swiglu", hidden_size=512, use_bias_in_mlp=False))
    return mlp, torch.randn((1, 1, 512)).as_subclass(OnGpu)


def own_linear_layers(m, mlp):
    from megatron.model import transformer_layer as layers

    m.setattr(layers, "Linear", type("Own", (layers.Linear,), {}))
    mlp.linear1, mlp.linear2 = layers.Linear(512, 512, bias=False, skip_bias_add=True), layers.Linear(256, 512, bias=False, skip_bias_add=True)


REPLACED = {
    "forward of the class": lambda m, mlp: m.setattr(type(mlp), "forward", lambda self, x: None),
    "forward of the linear layers": lambda m, mlp: m.setattr(type(mlp.linear1), "forward", lambda self, x: None),
    "forward of the gate": lambda m, mlp: m.setattr(type(mlp.activation_func), "forward", lambda self, x: None),
    "call of the class": lambda m, mlp: m.setattr(type(mlp), "__call__", lambda self, x: None, raising=False),
    "call of every module": lambda m, mlp: m.setattr(torch.nn.Module, "__call__", lambda self, x: None),
    "compiled": lambda m, mlp: m.setattr(mlp.linear2, "_compiled_call_impl", lambda self, x: None, raising=False),
    "bias added in the layer": lambda m, mlp: m.setattr(mlp.linear2, "skip_bias_add", False),
    "another class of linear layers": lambda m, mlp: own_linear_layers(m, mlp),
    "another layer": lambda m, mlp: mlp.__setattr__("linear1", torch.nn.Linear(512, 512)),
}


@pytest.mark.parametrize("who", REPLACED)
def test_a_decoding_step_calls_what_was_replaced(who, monkeypatch):
    """The launches of few rows stand for the classes of this package as they are written."""
    from megatron.fused_kernels import _hotpath

    monkeypatch.setattr(_hotpath, "native", Launches)
    mlp, x = few_rows()
    with torch.no_grad():
        assert mlp.add_to(x, x) == "one launch"
        REPLACED[who](monkeypatch, mlp)
        assert mlp.add_to(x, x) is None


@pytest.mark.parametrize("who", ["softmax", "core"])
def test_attention_classes_that_were_replaced_are_called(who, monkeypatch):
    c = core()
    assert scale(c) is not None and fused_attention.untouched(c, CoreAttention)
    monkeypatch.setattr(FusedScaleMaskSoftmax if who == "softmax" else CoreAttention, "forward", lambda *a, **k: None)
    assert scale(c) is None if who == "softmax" else not fused_attention.untouched(c, CoreAttention)


@pytest.mark.parametrize("replaced", [False, True])
def test_a_replaced_addition_of_both_branches_is_called(replaced, monkeypatch):
    """In the parallel layout, where the attention's output is added in the launch of the feed forward block."""
    from megatron.model import transformer_layer as layers

    class Layer(layers.TransformerLayer):
        def _attend(self, x, attention_mask, layer_past):
            return x, None

        def _mlp_added(self, *args):
            return "one launch"

    args = types.SimpleNamespace(norm="layernorm", layernorm_epsilon=1e-5, hidden_size=128, num_attention_heads=2, seq_length=16, precision="fp32",
                                 pos_emb="none", activation="silu", intermediate_size=768, gpt_j_residual=True, gpt_j_tied=True, hidden_dropout=0.0,
                                 scaled_upper_triang_masked_softmax_fusion=False, scaled_masked_softmax_fusion=False)
    layer = Layer(args, lambda s, m: s, 1).eval()
    layer.mlp = torch.nn.Identity()
    layer.mlp.forward = lambda x: (x, None)
    if replaced:
        monkeypatch.setattr(layers, "bias_add_residual_pair", lambda *a: "the sum")
    with torch.no_grad():
        assert layer(torch.randn((2, 1, 128)), None) == ("the sum" if replaced else "one launch")
