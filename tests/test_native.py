"""What the host side in csrc/native.cpp leaves to Python, on the CPU: everything that is not a plain tensor on a GPU, and calls
of another form."""
import pytest
import torch

from megatron.fused_kernels import _hotpath as hp

X = torch.ones((4, 4))


class Sub(torch.Tensor):
    pass


OPERANDS = {"on the cpu": X, "subclass": X.as_subclass(Sub), "meta": torch.empty((4, 4), device="meta"), "none": None, "number": 3.0,
            "sparse": X.to_sparse(), "parameter": torch.nn.Parameter(X)}
CALLS = {"layer_norm": ("x", None, None, 1e-5), "layer_norm_pair": ("x", None, None, None, None, 1e-5), "rms_norm": ("x", None, None, 1e-5, 0, 4),
         "bias_gelu": ("x", None), "gated": ("x", 0), "causal_softmax": ("x", 1.0, -1), "masked_softmax": ("x", "x", 1.0),
         "rotary": ("x", "x", "x", "x", 0), "split_rotary": ("x", "x", "x", 0, 0, 0), "add_residual": ("x", None, None),
         "add_residual_pair": ("x", None, "x", None, "x"), "causal_attention": ("x", "x", "x", 1.0, -1, True),
         "masked_attention": ("x", "x", "x", "x", 1.0, -1e4, True), "decode_attention": ("x", "x", "x", "x", "x", 1.0, -1e4, True),
         "append_to_cache": ("x", "x", None), "linear": ("x", "x", None, 16, 32),
         "linear_act": ("x", "x", None, 0, 16, 32), "linear_add": ("x", "x", None, None, None, "x", 16, 32)}


@pytest.mark.parametrize("name", CALLS)
def test_left_to_python(name):
    call = getattr(hp.native(), name)
    for operand in OPERANDS.values():
        assert call(*(operand if a == "x" else a for a in CALLS[name])) is NotImplemented
    assert call() is NotImplemented and call(*CALLS[name]) is NotImplemented
    assert call(*(X if a == "x" else a for a in CALLS[name]), None) is NotImplemented
    assert call(*(X if a == "x" else 2 ** 80 for a in CALLS[name])) is NotImplemented
    with pytest.raises(TypeError):
        call(x=X)


def test_a_missing_module_is_an_error(monkeypatch):
    import sys

    monkeypatch.setattr(hp, "_native", None)
    monkeypatch.setitem(sys.modules, "megatron.fused_kernels._native", None)
    monkeypatch.delattr(sys.modules["megatron.fused_kernels"], "_native", raising=False)
    with pytest.raises(ImportError, match="_native.so"):
        hp.native()


@pytest.mark.parametrize("built", [("2.9.1+rocm6.4", None, None), (None, "3.11", None), (None, None, 0), None])
def test_a_module_built_for_something_else_is_an_error(built, monkeypatch):
    """Torch's C++ interface holds for one version: such a module is not called, neither by the layers nor after ``load``."""
    import sys
    import types

    import megatron.fused_kernels as fk

    fits = hp.native().BUILT_FOR
    assert fits == (torch.__version__, "%d.%d" % sys.version_info[:2], hp.lib().nhp_abi_version())
    other = types.SimpleNamespace() if built is None else types.SimpleNamespace(BUILT_FOR=tuple(b if b is not None else f for b, f in zip(built, fits)))
    monkeypatch.setattr(hp, "_native", None)
    monkeypatch.setattr(fk, "_native", other, raising=False)
    for call in (hp.native, fk.load):
        with pytest.raises(ImportError, match="rebuild"):
            call()
    assert hp._native is None


def test_the_build_is_for_the_running_python(monkeypatch):
    import sys

    seen = []
    monkeypatch.setattr(hp.subprocess, "run", lambda cmd, **kw: seen.append(cmd))
    hp.build()
    assert f"PYTHON={sys.executable}" in seen[0]


def test_what_works_without_a_gpu_needs_no_module(monkeypatch):
    """Linear layers, a feed forward block of torch's activations and the norms, on tensors that are not on a GPU."""
    import types

    from megatron.model.fused_linear import linear
    from megatron.model.norms import LayerNorm, RMSNorm
    from megatron.model.transformer_layer import MLP, Linear

    def missing():
        raise ImportError("not built")

    monkeypatch.setattr(hp, "native", missing)
    x = torch.randn((3, 512))
    mlp = MLP(types.SimpleNamespace(activation="silu", hidden_size=512, intermediate_size=1536))
    mlp.linear2 = Linear(1536, 512, skip_bias_add=True)
    for grad in (True, False):
        with torch.set_grad_enabled(grad):
            assert torch.equal(linear(x, mlp.linear1.weight), torch.nn.functional.linear(x, mlp.linear1.weight))
            assert Linear(512, 64)(x)[0].shape == (3, 64) and LayerNorm(512)(x).shape == RMSNorm(512)(x).shape == x.shape
            assert mlp(x)[0].shape == x.shape and mlp.add_to(x, x) is None


def test_what_could_be_scripted_still_can():
    """TorchScript takes the modules and functions around the native calls as it did, and leaves those out."""
    from megatron.model.activations import bias_gelu_impl
    from megatron.model.fused_bias_dropout import bias_add_residual_pair
    from megatron.model.norms import LayerNorm, RMSNorm

    x = torch.randn((3, 64), generator=torch.Generator().manual_seed(0))
    for module in (LayerNorm(64), RMSNorm(64)):
        for grad in (True, False):
            with torch.set_grad_enabled(grad):
                assert torch.equal(torch.jit.script(module)(x), module(x))

    def activation(x, b):
        return bias_gelu_impl(x, b)

    for f in (activation, bias_add_residual_pair):
        torch.jit.script(f)


@pytest.mark.parametrize("rows,n,k,taken", [(4096, 512, 512, True), (4097, 512, 512, False), (8192, 256, 768, False), (4096, 256, 768, True),
                                            (16384, 16, 768, True), (16385, 16, 768, False), (16384, 128, 1024, False), (2048, 1024, 1024, True)])
def test_many_rows_of_narrow_layers(rows, n, k, taken):
    """Where tiles share the CUs the rule of nhp_linear_tiles ends with the rows that were measured."""
    assert bool(hp.lib().nhp_linear_tiles_pay(rows, n, k)) == taken
