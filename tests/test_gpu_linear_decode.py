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
