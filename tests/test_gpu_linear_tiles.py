"""The linear layer of a short prompt (csrc/linear_tiles.hip) against fp64: one row, whole and broken tiles of 64 on both sides, fewer steps
of 64 features than the ring holds, as many and more.

Tolerance: one rounding of the result, at most u = 2^-8 (bf16) or 2^-11 (fp16), u / sqrt(3) in the mean square of a 2-norm;
the fp32 sums are three orders of magnitude below that."""
import math

import pytest
import torch

import util

pytestmark = pytest.mark.gpu
DEV = "cuda"


def tiles(x, w, bias):
    from megatron.fused_kernels import _hotpath as hp

    y = torch.full((x.size(0) + 1, w.size(0)), float("nan"), dtype=x.dtype, device=DEV)
    rc = hp.lib().nhp_linear_tiles(y.data_ptr(), x.data_ptr(), w.data_ptr(), None if bias is None else bias.data_ptr(), x.size(0), w.size(0),
                                   w.size(1), hp.dtype_code(x, "linear"), hp.stream_of(x))
    hp.check(rc, "linear")
    assert y[-1].isnan().all()   # nothing past the end
    return y[:-1]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("n,k", [(16, 64), (48, 128), (64, 192), (80, 256), (1040, 320), (2304, 768), (4112, 1024), (16400, 128), (192, 4096)])
@pytest.mark.parametrize("rows", [1, 33, 63, 64, 65, 129, 500])
def test_against_fp64(dtype, n, k, rows):
    x, w = util.randn((rows, k), dtype, seed=1).to(DEV), util.randn((n, k), dtype, seed=2).to(DEV)
    b = util.randn((n,), dtype, seed=3, std=math.sqrt(k)).to(DEV)
    for bias in (None, b):
        got = tiles(x, w, bias)
        want = x.double() @ w.double().t() + (0.0 if bias is None else bias.double())
        assert (got.double() - want).norm() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11) / math.sqrt(3) * want.norm()
        assert torch.equal(got, tiles(x, w, bias))


def test_an_infinite_weight_reaches_its_own_result_only():
    x, w = util.randn((70, 832), torch.bfloat16, seed=1).to(DEV), util.randn((80, 832), torch.bfloat16, seed=2).to(DEV)
    w[37, 831] = float("inf")
    x[69, 0] = float("nan")
    bad = ~torch.isfinite(tiles(x, w, None))
    assert bad[:, 37].all() and bad[69].all() and int(bad.sum()) == 70 + 80 - 1


@pytest.mark.parametrize("rows,n,k,taken", [(33, 2304, 768, True), (32, 2304, 768, False), (512, 4096, 1024, True), (513, 4096, 1024, False),
                                            (33, 8192, 2048, True), (33, 16400, 2048, False), (33, 8128, 2048, False), (65, 4096, 2112, True), (65, 4032, 2112, False),
                                            (64, 8192, 2112, False), (256, 4096, 4096, True), (257, 4096, 4096, False),
                                            (128, 4096, 4160, False), (100, 2304, 736, False)])
def test_who_is_called(rows, n, k, taken):
    """The rule on both sides of its lines, through the native and the Python path, and the calls that stay the library's."""
    from unittest import mock

    from megatron.fused_kernels import _hotpath as hp
    from megatron.model import fused_linear

    x, w = util.randn((rows, 1, k), torch.bfloat16, seed=1).to(DEV), util.randn((n, k), torch.bfloat16, seed=2).to(DEV)
    assert bool(fused_linear._some_rows(x, w, None)) == taken
    y = fused_linear.linear(x, w)
    want = x.double() @ w.double().t()
    assert y.shape == (rows, 1, n) and (y.double() - want).norm() <= 2.0 ** -8 / math.sqrt(3) * want.norm()
    if not taken:
        return
    assert torch.equal(y[:, 0], tiles(x[:, 0], w, None))
    with mock.patch.object(hp, "native", lambda: mock.Mock(linear=lambda *a: NotImplemented)):
        assert torch.equal(y, fused_linear.linear(x, w))
    b = util.randn((n + 1,), torch.bfloat16, seed=3).to(DEV)
    for other in ((x.transpose(0, 1).expand(2, rows, k).transpose(0, 1), w, None), (x.float(), w.float(), None),
                  (x, w.clone().requires_grad_(True), None), (x, w, b[1:])):
        assert not fused_linear._some_rows(*other)
        with mock.patch.object(fused_linear.F, "linear", wraps=fused_linear.F.linear) as library:
            fused_linear.linear(*other)
            assert library.call_count == 1
