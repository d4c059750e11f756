"""Whoever looks at the modules of the attention keeps seeing what passes through them: hooks, subclasses and replaced methods of
the softmax module, hooks on ``CoreAttention`` in a layer with cached positions. On the CPU; which route a call takes is asked
with the operand checks answered for a GPU."""
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


def scale(c, monkeypatch):
    monkeypatch.setattr(fused_attention, "supported", lambda q, k, v: True)
    t = torch.zeros((8, 1, 4, 64), dtype=torch.bfloat16)
    return c._plain_scale(t, t, t, fb.causal_mask(8), None)


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
def test_a_watched_softmax_is_called(who, monkeypatch):
    c = core()
    assert scale(c, monkeypatch) == pytest.approx(0.125)
    handle = WATCHERS[who](c)
    try:
        assert scale(c, monkeypatch) is None
    finally:
        if hasattr(handle, "remove"):
            handle.remove()
            assert scale(c, monkeypatch) == pytest.approx(0.125)


def test_the_switch_for_tools_that_inspect_the_tensors(monkeypatch):
    assert scale(core(causal_gemm_blocks=False), monkeypatch) is None
