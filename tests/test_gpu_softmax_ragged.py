"""Softmax rows of any length and alignment (csrc/softmax_ragged.hip) against the oracle: the edges of every geometry
(lanes per row, chunks per lane, waves per row), lengths around a chunk, views that start on odd elements, and what the
memory around the results holds afterwards."""
import math

import pytest
import torch

import oracle
import util

pytestmark = pytest.mark.gpu
DEV = "cuda"
DTYPES = pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
GUARD = 64


@pytest.fixture(scope="module")
def hotpath():
    from megatron.fused_kernels import _hotpath

    return _hotpath


class Guarded:
    """A tensor that starts ``offset`` elements into an allocation of NaNs."""

    def __init__(self, shape, dtype, offset, value=None):
        n = math.prod(shape)
        self.buf = torch.full((offset + n + GUARD,), float("nan"), dtype=dtype, device=DEV)
        self.t = self.buf[offset:offset + n].view(shape)
        if value is not None:
            self.t.copy_(value)

    def untouched(self):
        n = self.t.numel()
        start = (self.t.data_ptr() - self.buf.data_ptr()) // self.buf.element_size()
        return bool(self.buf[:start].isnan().all() and self.buf[start + n:].isnan().all())


# edges of the geometries: 64, 128, 256, 512, 1024, 1536, 2048, 4096, 6144, 8192, 12288, 16384 elements; offsets in elements
MASKED = [(2, 3, 5, 9, 0), (1, 2, 3, 63, 3), (2, 1, 7, 64, 1), (1, 4, 3, 65, 0), (2, 3, 4, 129, 5), (1, 2, 2, 257, 7), (1, 5, 6, 511, 0),
          (2, 2, 3, 513, 2), (1, 3, 3, 1021, 0), (1, 2, 2, 1025, 1), (1, 2, 2, 1537, 0), (1, 2, 3, 2047, 4), (1, 2, 2, 2049, 0),
          (1, 3, 2, 4099, 6), (1, 2, 2, 6145, 0), (1, 2, 2, 8191, 0), (1, 1, 2, 12289, 3), (1, 2, 2, 8200, 1), (1, 1, 2, 16383, 0)]


@DTYPES
@pytest.mark.parametrize("b,np_,sq,sk,offset", MASKED)
def test_padding_mask_forward_and_backward(hotpath, dtype, b, np_, sq, sk, offset):
    lib = hotpath.lib()
    x = util.randn((b, np_, sq, sk), dtype, seed=sk, std=2.0)
    dy = util.randn((b, np_, sq, sk), dtype, seed=sk + 1)
    mask = torch.rand((b, 1, sq, sk), generator=torch.Generator().manual_seed(sk)) < 0.3
    mask[..., sk // 2:] |= torch.rand((b, 1, sq, 1), generator=torch.Generator().manual_seed(3)) < 0.5
    mask[0, 0, -1] = True
    want = oracle.masked_softmax_fwd(x, mask, 0.3)
    y, xd, md = Guarded(x.shape, dtype, offset), Guarded(x.shape, dtype, offset, x), mask.to(DEV)
    code, st = hotpath.dtype_code(x, "test"), hotpath.stream_of(xd.t)
    assert lib.nhp_masked_softmax_fwd(y.t.data_ptr(), xd.t.data_ptr(), md.data_ptr(), 0.3, b, np_, sq, sk, b, code, st) == 0
    util.assert_ulp_close(y.t.cpu(), want, 2, "fwd")
    assert y.untouched()
    # in place, and with one mask row block for the whole batch
    want1 = oracle.masked_softmax_fwd(x, mask[:1], 0.3)
    m1 = mask[:1].to(DEV)
    assert lib.nhp_masked_softmax_fwd(xd.t.data_ptr(), xd.t.data_ptr(), m1.data_ptr(), 0.3, b, np_, sq, sk, 1, code, st) == 0
    util.assert_ulp_close(xd.t.cpu(), want1, 2, "fwd in place")
    assert xd.untouched()
    want_dx = oracle.softmax_bwd(dy, want, 0.3, causal=False)
    g, yd = Guarded(x.shape, dtype, offset, dy), Guarded(x.shape, dtype, (offset + 3) % 8, want)
    rows = b * np_ * sq
    assert lib.nhp_masked_softmax_bwd(g.t.data_ptr(), g.t.data_ptr(), yd.t.data_ptr(), 0.3, rows, sk, code, st) == 0
    util.assert_softmax_bwd_close(g.t.cpu(), want_dx, dy, want, 0.3, "bwd in place")
    assert g.untouched()


@DTYPES
@pytest.mark.parametrize("b,heads,s,window,lengths,offset", [
    (1, 3, 9, None, None, 0), (2, 2, 67, 5, None, 1), (2, 2, 129, None, [129, 0], 0), (1, 2, 255, 130, [77], 3), (1, 1, 513, None, None, 7),
    (1, 1, 1027, 700, None, 0), (1, 1, 2051, None, None, 0), (1, 1, 64, 9, None, 1), (1, 2, 264, None, [100], 5)])
def test_causal_forward_and_backward(hotpath, dtype, b, heads, s, window, lengths, offset):
    lib = hotpath.lib()
    x = util.randn((b * heads, s, s), dtype, seed=s, std=2.0)
    dy = util.randn(x.shape, dtype, seed=s + 1)
    kl = None if lengths is None else torch.tensor(lengths, dtype=torch.int32)
    want = oracle.causal_softmax_fwd(x, 0.3, window=window, key_lengths=kl)
    y, xd = Guarded(x.shape, dtype, offset), Guarded(x.shape, dtype, offset, x)
    kd = None if kl is None else kl.to(DEV)
    kp, w = None if kl is None else kd.data_ptr(), -1 if window is None else window
    code, st = hotpath.dtype_code(x, "test"), hotpath.stream_of(xd.t)
    assert lib.nhp_causal_softmax_ex_fwd(y.t.data_ptr(), xd.t.data_ptr(), 0.3, b * heads, s, w, None, None, kp, heads, code, st) == 0
    util.assert_ulp_close(y.t.cpu(), want, 2, "fwd")
    assert y.untouched()
    want_dx = oracle.softmax_bwd(dy, want, 0.3, causal=True, window=window, key_lengths=kl)
    g, yd = Guarded(x.shape, dtype, offset, dy), Guarded(x.shape, dtype, (offset + 3) % 8, want)
    assert lib.nhp_causal_softmax_ex_bwd(g.t.data_ptr(), g.t.data_ptr(), yd.t.data_ptr(), 0.3, b * heads, s, w, kp, heads, code, st) == 0
    util.assert_softmax_bwd_close(g.t.cpu(), want_dx, dy, want, 0.3, "bwd in place")
    assert g.untouched()


def test_scores_of_minus_infinity(hotpath):
    """They count for nothing, also where they are all that one wave of a row sees."""
    x = util.randn((1, 2, 2, 4099), torch.float32, seed=5)
    x[..., 512:] = float("-inf")
    mask = torch.zeros((1, 1, 2, 4099), dtype=torch.bool)
    got = util.abi_masked_fwd(hotpath, x.bfloat16().to(DEV), mask.to(DEV), 0.5).cpu()
    want = torch.softmax(x.bfloat16().double() * 0.5, dim=-1)
    assert (got.double() - want).norm() <= 2.0 ** -8 * want.norm()   # one rounding: 2^-9 at most
