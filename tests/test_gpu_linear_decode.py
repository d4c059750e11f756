"""The few-row linear layer (csrc/linear_decode.hip) against fp64: one and two tiles of sixteen rows, weight tiles fewer and more than
workgroups, contractions that do not divide evenly among the waves, and the split ones.

Tolerance: one rounding of the result, at most u = 2^-8 (bf16) or 2^-11 (fp16), u / sqrt(3) in the mean square of a 2-norm;
the fp32 sums are three orders of magnitude below that."""
import math

import pytest
import torch

import util

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("n,k", [(16, 32), (48, 544), (4112, 96), (2304, 768), (6160, 4096), (80, 4128), (1040, 11008), (32, 16384)])
@pytest.mark.parametrize("rows", [1, 7, 16, 17, 32])
def test_against_fp64(dtype, n, k, rows):
    from megatron.model import fused_linear

    x, w = util.randn((rows, 1, k), dtype, seed=1).to(DEV), util.randn((n, k), dtype, seed=2).to(DEV)
    b = util.randn((n,), dtype, seed=3, std=math.sqrt(k)).to(DEV)
    assert fused_linear._few_rows(x, w, b) == (rows <= 16 or min(n, k) <= 2048)
    for bias in (None, b):
        got = fused_linear.linear(x, w, bias)
        want = x.double() @ w.double().t() + (0.0 if bias is None else bias.double())
        assert got.shape == (rows, 1, n)
        assert (got.double() - want).norm() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) / math.sqrt(3) * want.norm()
        assert torch.equal(got, fused_linear.linear(x, w, bias))


@pytest.mark.parametrize("n,k", [(20496, 96), (12304, 288), (8208, 2080), (4128, 4064), (272, 4192), (1040, 12320)])
@pytest.mark.parametrize("rows", [1, 16, 18])
def test_several_tiles_and_odd_steps(n, k, rows):
    """Up to six tiles for a workgroup, pieces of one step among those of two, waves with none; a bias that starts in the middle
    of a word."""
    from megatron.model import fused_linear

    x, w = util.randn((rows, k), torch.bfloat16, seed=1).to(DEV), util.randn((n, k), torch.bfloat16, seed=2).to(DEV)
    b = util.randn((n + 1,), torch.bfloat16, seed=3, std=math.sqrt(k)).to(DEV)
    for bias in (b[1:], b[:-1]):
        want = x.double() @ w.double().t() + bias.double()
        got = fused_linear.linear(x, w, bias)
        assert (got.double() - want).norm() <= 2.0 ** -8 / math.sqrt(3) * want.norm()


def test_an_infinite_weight_reaches_its_own_result_only():
    from megatron.model.fused_linear import linear

    x, w = util.randn((3, 800), torch.bfloat16, seed=1).to(DEV), util.randn((64, 800), torch.bfloat16, seed=2).to(DEV)
    w[37, 799] = float("inf")
    bad = ~torch.isfinite(linear(x, w))
    assert bad[:, 37].all() and int(bad.sum()) == 3


def test_everything_else_goes_to_the_library():
    from megatron.model import fused_linear
    from megatron.model.fused_linear import linear

    x, w = util.randn((4, 64), torch.bfloat16, seed=1).to(DEV), util.randn((32, 64), torch.bfloat16, seed=2).to(DEV)
    assert fused_linear._few_rows(x, w, None)
    g = w.clone().requires_grad_(True)
    assert not fused_linear._few_rows(x, g, None)
    linear(x, g).sum().backward()
    assert g.grad is not None
    with torch.no_grad():
        assert fused_linear._few_rows(x, g, None)
    for a, b in ((x.repeat(9, 1), w), (x.float(), w.float()), (x[:, :40], w[:, :40]), (x, w[:24]), (x[:0], w), (x.cpu(), w.cpu()),
                 (torch.cat((x, x), 1)[:, ::2], w)):
        assert not fused_linear._few_rows(a, b, None)
        assert linear(a, b).shape == (a.size(0), b.size(0))
    with torch.autocast("cuda", dtype=torch.float16):
        assert not fused_linear._few_rows(x, w, None)
    assert torch.func.vmap(lambda v: linear(v, w))(x).shape == (4, 32)


SHAPES = pytest.mark.parametrize("rows,n,k", [(1, 32, 32), (16, 64, 544), (5, 4160, 96), (17, 9248, 160), (3, 96, 4128), (32, 1056, 11008), (16, 12352, 800)])


@SHAPES
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_with_the_activation(rows, n, k, dtype):
    """The bits of the product and the activation called one after the other."""
    from megatron.fused_kernels import _hotpath as hp
    from megatron.model import fused_linear
    from megatron.model.activations import Gated_Activation, bias_gelu_impl

    x, w = util.randn((rows, k), dtype, seed=1).to(DEV), util.randn((n, k), dtype, seed=2, std=1.0 / math.sqrt(k)).to(DEV)
    b = util.randn((n + 1,), dtype, seed=3).to(DEV)
    native, most = hp.native(), (32, 32)
    product = native.linear(x, w, None, *most)
    for bias in (b[1:], b[:-1], None):
        # (an aligned bias: the activation's kernel for others rounds its product with the gate once, to fp16)
        want = bias_gelu_impl(product, torch.zeros_like(b[1:]) if bias is None else bias.clone())
        assert torch.equal(native.linear_act(x, w, bias, fused_linear.BIAS_GELU, *most), want)
    for kind in ("swiglu", "geglu", "reglu", "glu", "bilinear"):
        gate = Gated_Activation(kind)
        assert torch.equal(native.linear_act(x, w, None, gate._code, *most), gate(product))
    assert native.linear_act(x, w, b[1:], 0, *most) is NotImplemented and native.linear_act(x, w, None, 5, *most) is NotImplemented
    assert native.linear_act(x, w[:16], None, 0, *most) is NotImplemented


@SHAPES
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_with_the_residual_addition(rows, n, k, dtype):
    from megatron.fused_kernels import _hotpath as hp
    from megatron.model.fused_bias_dropout import bias_add_residual_pair, bias_dropout_add_fused_inference

    x, w = util.randn((rows, 1, k), dtype, seed=1).to(DEV), util.randn((n, k), dtype, seed=2, std=1.0 / math.sqrt(k)).to(DEV)
    r, x1 = util.randn((rows, 1, n), dtype, seed=3).to(DEV), util.randn((rows, 1, n), dtype, seed=4).to(DEV)
    b, b1 = util.randn((n + 1,), dtype, seed=5).to(DEV)[1:], util.randn((n,), dtype, seed=6).to(DEV)
    native, most = hp.native(), (32, 32)
    product = native.linear(x, w, None, *most)
    for bias in (b, None):
        assert torch.equal(native.linear_add(x, w, bias, None, None, r, *most), bias_dropout_add_fused_inference(product, bias, r, 0.0))
        for bias1 in (b1, None):
            assert torch.equal(native.linear_add(x, w, bias, x1, bias1, r, *most), bias_add_residual_pair(x1, bias1, product, bias, r))
    for bad in (r[:, :, 1:], r.float(), r.reshape(rows, n), r.transpose(0, 2)):
        assert native.linear_add(x, w, b, None, None, bad, *most) is NotImplemented or bad.shape == r.shape and bad.is_contiguous()
    assert native.linear_add(x, w, b, None, b1, r, *most) is NotImplemented


@pytest.mark.parametrize("style", ["gelu", "swiglu"])
def test_a_layer_takes_them_unless_somebody_looks(style):
    """One layer's step: the same bits by separate launches, which is what it makes while a module inside is watched."""
    import types

    from megatron.model.transformer_layer import TransformerLayer

    gelu = style == "gelu"
    args = types.SimpleNamespace(
        hidden_size=256, num_attention_heads=4, num_kv_heads=4, seq_length=64, precision="bfloat16", pos_emb="rotary", rotary_pct=1.0,
        rotary_emb_base=10000, rope_fusion=True, norm="layernorm" if gelu else "rmsnorm", layernorm_epsilon=1e-5, rms_norm_epsilon=1e-6,
        activation=style, bias_gelu_fusion=True, onnx_safe=False, scaled_upper_triang_masked_softmax_fusion=True,
        scaled_masked_softmax_fusion=False, attention_softmax_in_fp32=True, attention_dropout=0.0, hidden_dropout=0.0,
        bias_dropout_fusion=True, gpt_j_residual=gelu, use_bias_in_mlp=gelu, use_bias_in_attn_linear=gelu)
    torch.manual_seed(0)
    with torch.device(DEV):
        layer = TransformerLayer(args, lambda s, m: s.masked_fill_(m, -10000.0), 1, rotary=True, use_cache=True)
    layer = layer.bfloat16().eval()
    x, past = util.randn((1, 3, 256), torch.bfloat16, seed=1).to(DEV), util.randn((2, 9, 3, 4, 64), torch.bfloat16, seed=2).to(DEV)
    mask = torch.zeros((1, 1, 1, 10), dtype=torch.bool, device=DEV)
    seen = []

    def step(x=x):
        layer.layer_past = None
        with torch.no_grad():
            return layer(x, mask, layer_past=past)

    want = step()
    assert layer.mlp._activated(x) is None   # gradients are wanted here
    with torch.no_grad():
        assert layer.mlp._activated(x) is not None and layer.mlp.add_to(x, x) is not None
    for module in (layer.mlp, layer.mlp.linear1, layer.mlp.linear2):
        handle = module.register_forward_hook(lambda m, i, o: seen.append(m))
        assert torch.equal(step(), want) and seen[-1] is module
        handle.remove()
    layer.mlp.linear1.forward = lambda v: (torch.nn.functional.linear(v, layer.mlp.linear1.weight) * 0, layer.mlp.linear1.bias)
    assert not torch.equal(step(), want)
    del layer.mlp.linear1.forward
    assert torch.equal(step(), want)
    with torch.autocast("cuda", dtype=torch.float16):
        assert layer.mlp._activated(x) is None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def test_an_unaligned_bias_gives_the_bits_of_separate_launches(dtype):
    """The parameters of a layer may be slices of one buffer."""
    import types

    from megatron.model.transformer_layer import MLP

    mlp = MLP(types.SimpleNamespace(activation="gelu", bias_gelu_fusion=True, hidden_size=768)).to(DEV).to(dtype)
    x, buffer = util.randn((16, 1, 768), dtype, seed=1).to(DEV), util.randn((3073,), dtype, seed=2).to(DEV)
    mlp.linear1.bias = torch.nn.Parameter(buffer[1:])
    with torch.no_grad():
        mlp.linear1.weight.copy_(util.randn((3072, 768), dtype, seed=3, std=0.05))
        got = mlp(x)[0]
        mlp.linear1.register_forward_hook(lambda module, inputs, output: None)
        assert torch.equal(got, mlp(x)[0])


@pytest.mark.parametrize("rows", [1, 16, 20])
@pytest.mark.parametrize("splits", [1, 4])
def test_the_order_of_the_sums(rows, splits):
    """Sixteen sums of consecutive features each, added up one after the other, in each of the splits, and those. Whole numbers, whose
    products add up without rounding; the sixth sum takes the fifth, which is 2^18 times the size of the others, away again."""
    from megatron.fused_kernels import _hotpath as hp

    shares, each, n = 16 * splits, 128, 48
    g = torch.Generator().manual_seed(0)
    x, w = (torch.randint(-4, 5, (r, shares, each), generator=g).double() for r in (rows, n))
    w[:, 4] *= 2.0 ** 18
    w[:, 5], x[:, 5] = -w[:, 4], x[:, 4]
    sums = torch.einsum("rsk,nsk->srn", x, w).float().view(splits, 16, rows, n)
    want = torch.zeros((rows, n))
    for part in sums:
        v = torch.zeros_like(want)
        for s in part:
            v = v + s
        want = want + v if splits > 1 else v
    x, w = (t.reshape(t.size(0), -1).bfloat16().to(DEV) for t in (x, w))
    y, scratch = torch.empty((rows, n), dtype=torch.bfloat16, device=DEV), torch.empty((4 * splits * rows * n,), dtype=torch.uint8, device=DEV)
    hp.check(hp.lib().nhp_linear_decode(y.data_ptr(), x.data_ptr(), w.data_ptr(), None, scratch.data_ptr(), rows, n, shares * each, hp.BF16,
                                        hp.stream_of(x)), "linear")
    exact = torch.einsum("rk,nk->rn", x.double().cpu(), w.double().cpu())
    assert torch.equal(y.cpu(), want.bfloat16()) and not torch.equal(y.cpu(), exact.bfloat16())
