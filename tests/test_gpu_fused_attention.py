"""The attention kernels (csrc/attention.hip) through ``megatron.model.fused_attention`` and ``CoreAttention``, against
textbook attention in fp32 torch ops: edges of the 64-key tiles and of the 128-query blocks, head sizes that fill a tile
row and ones that do not, grouped heads, sliding windows, and bit masks with rows that see nothing.

Tolerance: a rounding to the storage type is off by at most u = 2^-8 (bf16) or 2^-11 (fp16), u / sqrt(3) in the mean
square; n of them in a row by sqrt(n / 3) u relative to the 2-norm. A context goes through two (probability, result), a
gradient of v as well. A gradient of q or k goes through two (gradient of the score, result) and through that of the
context, which enters as dP - dO . context: a difference that is half as large as its members when a query sees only two
keys (window 1), so the rounding counts twice, in squares four times. Gradients of shared heads are summed in fp32."""
import math

import pytest
import torch

import util

pytestmark = pytest.mark.gpu
DEV = "cuda"
DTYPES = pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])


def limit(dtype, roundings):
    return math.sqrt(roundings / 3) * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)


def rel_err(a, b):
    return ((a.float() - b.float()).norm() / b.float().norm()).item()


def textbook(q, k, v, mask, fill=torch.finfo(torch.float32).min):
    """[sq, b, np, hn] in fp32; mask broadcastable to [b, np, sq, sk]."""
    group = q.size(2) // k.size(2)
    k, v = (torch.repeat_interleave(t.float(), group, dim=2).permute(1, 2, 0, 3) for t in (k, v))
    scores = torch.matmul(q.float().permute(1, 2, 0, 3).contiguous(), k.transpose(-1, -2).contiguous()) / math.sqrt(q.size(-1))
    probs = torch.softmax(scores.masked_fill(mask, fill), dim=-1)
    return torch.matmul(probs, v.contiguous()).permute(2, 0, 1, 3)


def hidden(sq, sk, window=None):
    q = torch.arange(sq, device=DEV).view(sq, 1) + sk - sq
    k = torch.arange(sk, device=DEV).view(1, sk)
    return (k > q) if window is None else (k > q) | (k < q - window)


def operands(dtype, sq, sk, b, np_, nkv, hn, seed):
    return [util.randn((s, b, n, hn), dtype, seed=seed + i).to(DEV) for i, (s, n) in enumerate(((sq, np_), (sk, nkv), (sk, nkv)))]


@DTYPES
@pytest.mark.parametrize("hn", [64, 80, 96, 128])
@pytest.mark.parametrize("s,b,np_,nkv,window", [(20, 1, 4, 4, None), (2113, 1, 2, 1, None), (1600, 1, 3, 3, 700), (64, 1, 4, 4, None), (65, 2, 4, 2, None), (128, 1, 8, 2, 1),
                                                (260, 3, 3, 3, None), (700, 1, 4, 1, 37), (513, 1, 9, 3, 128),
                                                # shared heads: two of four, all four, all three in one workgroup
                                                (65, 64, 16, 4, None), (65, 128, 16, 4, 7), (131, 64, 12, 4, None)])
def test_causal_forward_and_gradients(dtype, hn, s, b, np_, nkv, window):
    from megatron.model.fused_attention import causal_attention

    q, k, v = (t.requires_grad_(True) for t in operands(dtype, s, s, b, np_, nkv, hn, 1))
    out = causal_attention(q, k, v, 1 / math.sqrt(hn), window, merged=True)
    g = util.randn((s, b, np_ * hn), dtype, seed=9).to(DEV)
    out.backward(g)
    qr, kr, vr = (t.detach().float().requires_grad_(True) for t in (q, k, v))
    ref = textbook(qr, kr, vr, hidden(s, s, window))
    ref.backward(g.float().view(s, b, np_, hn))
    assert rel_err(out.view(s, b, np_, hn), ref) <= limit(dtype, 2)
    for got, want, n in ((q.grad, qr.grad, 6), (k.grad, kr.grad, 6), (v.grad, vr.grad, 2)):
        assert rel_err(got, want) <= limit(dtype, n)
    # the other layout, strided operands and a second run: the same bits
    wide = torch.stack((q.detach(), k.detach().expand_as(q) if nkv == np_ else q.detach()), dim=3).flatten(3)[..., :hn]
    again = causal_attention(wide, k.detach(), v.detach(), 1 / math.sqrt(hn), window).permute(2, 0, 1, 3)
    assert torch.equal(util.raw_bits(again.reshape(s, b, np_ * hn)), util.raw_bits(out.detach()))


@pytest.mark.parametrize("b,np_", [(1, 1), (1, 7), (1, 8), (2, 8), (3, 4), (1, 24)])
@pytest.mark.parametrize("s", [128, 129, 700])
def test_a_matrix_is_the_same_among_others(b, np_, s):
    """Matrices that divide among the XCDs and ones that do not, of one block and of several: the bits that each has alone."""
    from megatron.model.fused_attention import causal_attention

    leaves = [t.requires_grad_(True) for t in operands(torch.bfloat16, s, s, b, np_, np_, 64, 31)]
    g = util.randn((b, np_, s, 64), torch.bfloat16, seed=9).to(DEV)
    out = causal_attention(*leaves, 0.125)
    grads = torch.autograd.grad(out, leaves, g)
    for i in range(b):
        for h in range(np_):
            one = [t.detach()[:, i:i + 1, h:h + 1].requires_grad_(True) for t in leaves]
            alone = causal_attention(*one, 0.125)
            assert torch.equal(alone[0, 0], out[i, h])
            for got, want in zip(torch.autograd.grad(alone, one, g[i:i + 1, h:h + 1]), grads):
                assert torch.equal(got[:, 0, 0], want[:, i, h])


@DTYPES
@pytest.mark.parametrize("hn", [64, 96])
@pytest.mark.parametrize("sq,sk,b,np_,nkv,window", [(1, 2, 1, 4, 4, None), (1, 130, 2, 4, 2, 5), (63, 129, 1, 4, 4, None), (128, 192, 1, 8, 2, 64),
                                                    (200, 1301, 1, 3, 1, None), (129, 1000, 2, 4, 4, 300), (500, 501, 1, 2, 2, 3)])
def test_fewer_queries_than_keys(dtype, hn, sq, sk, b, np_, nkv, window):
    """The queries are the last ones: query i attends to keys up to ``i + sk - sq``, forward and gradients; keys before every
    window get none."""
    from megatron.model.fused_attention import causal_attention

    q, k, v = (t.requires_grad_(True) for t in operands(dtype, sq, sk, b, np_, nkv, hn, 61))
    g = util.randn((b, np_, sq, hn), dtype, seed=9).to(DEV)
    causal_attention(q, k, v, 1 / math.sqrt(hn), window).backward(g)
    qr, kr, vr = (t.detach().float().requires_grad_(True) for t in (q, k, v))
    ref = textbook(qr, kr, vr, hidden(sq, sk, window))
    ref.backward(g.float().permute(2, 0, 1, 3))
    out = causal_attention(q, k, v, 1 / math.sqrt(hn), window).permute(2, 0, 1, 3)
    # one query has one score gradient for each key and head, whose rounding all features share: the largest and not the mean
    # square of a rounding, a factor of sqrt(3)
    few = math.sqrt(3) if sq == 1 else 1.0
    assert rel_err(out, ref) <= limit(dtype, 2) * few
    for got, want, n in ((q.grad, qr.grad, 6), (k.grad, kr.grad, 6), (v.grad, vr.grad, 2)):
        assert rel_err(got, want) <= limit(dtype, n) * few
    if window is not None and sk - sq - window > 0:
        assert not k.grad[:sk - sq - window].any() and not v.grad[:sk - sq - window].any()


def test_values_that_are_not_finite_stay_with_what_sees_them():
    """In the causal kernels: a NaN in a query reaches that query, in a key the queries that see it, an infinite value one
    feature of theirs; a NaN in the gradient of one context reaches its query and the keys that it sees. (Positions at the
    edge of a tile: within one, a product with an exact zero spreads them, as the products over whole rows do.)"""
    from megatron.model.fused_attention import causal_attention

    def apart(value, *where):
        expected = torch.zeros(value.shape, dtype=torch.bool, device=DEV)
        for at in where:
            expected[at] = True
        assert torch.equal(~torch.isfinite(value), expected)

    q, k, v = operands(torch.bfloat16, 200, 200, 1, 4, 2, 64, 71)
    q2, k2, v2 = q.clone(), k.clone(), v.clone()
    q2[70, 0, 1, 3], k2[90, 0, 1, 5], v2[128, 0, 0, 7] = float("nan"), float("nan"), float("inf")
    out = causal_attention(q2, k2, v2, 1 / 8, merged=True).view(200, 1, 4, 64)
    apart(out, (70, 0, 1), (slice(90, None), 0, slice(2, 4)), (slice(128, None), 0, slice(0, 2), 7))
    # a score of -inf: that key counts for nothing
    q3, k3 = q.clone(), k.clone()
    q3[..., 0] = q3[..., 0].abs() + 0.125
    k3[50, 0, 1, 0] = float("-inf")
    out = causal_attention(q3, k3, v, 1 / 8, merged=True).view(200, 1, 4, 64)
    mask = hidden(200, 200).expand(1, 4, 200, 200).clone()
    mask[:, 2:, :, 50] = True
    k3[50, 0, 1, 0] = 0.0
    want = textbook(q3, k3, v, mask)
    assert rel_err(out, want) <= limit(torch.bfloat16, 2)
    leaves = [t.requires_grad_(True) for t in (q, k, v)]
    g = util.randn((200, 1, 4, 64), torch.bfloat16, seed=9).to(DEV)
    g[127, 0, 3, 9] = float("nan")
    causal_attention(*leaves, 1 / 8, merged=True).backward(g.view(200, 1, 256))
    apart(q.grad, (127, 0, 3))
    apart(k.grad, (slice(0, 128), 0, 1))
    apart(v.grad, (slice(0, 128), 0, 1, 9))


@pytest.mark.parametrize("b", [1, 64, 128], ids=["apart", "in pairs", "together"])
def test_gradients_of_shared_heads_are_summed_before_they_are_rounded(b):
    """A query head's part may lie beyond the range of fp16 where the sum does not. With q, k and v zero the probabilities are
    1 / (i + 1), and the gradients of four heads that share a key are c, -c, 1 and 1 times their column sums."""
    from megatron.model.fused_attention import causal_attention

    s, hn, c = 128, 64, 30000.0
    q, k, v = (torch.zeros((s, b, n, hn), dtype=torch.float16, device=DEV, requires_grad=True) for n in (16, 4, 4))
    g = torch.tensor([c, -c, 1.0, 1.0], dtype=torch.float16, device=DEV).repeat(4).view(1, 1, 16, 1).expand(s, b, 16, hn)
    causal_attention(q, k, v, 1 / 8, merged=True).backward(g.reshape(s, b, 16 * hn))
    probs = (1 / torch.arange(1, s + 1, device=DEV)).half().double()
    want = 2 * probs.flip(0).cumsum(0).flip(0).view(s, 1, 1, 1)
    # 256 additions to a sum of up to 5.4 c lose at most 2^-24 of it each; then one rounding of up to 10.9 to fp16
    assert (v.grad.double() - want).abs().max() <= 5.4 * c * 256 * 2.0 ** -24 + 10.9 * 2.0 ** -11
    assert not q.grad.any() and not k.grad.any()


@DTYPES
@pytest.mark.parametrize("hn", [64, 80, 128])
@pytest.mark.parametrize("sq,sk,b,np_,nkv", [(1, 1, 1, 4, 4), (1, 200, 2, 4, 2), (5, 64, 1, 4, 4), (130, 333, 2, 4, 4), (1531, 1531, 1, 2, 1),
                                             (300, 4100, 1, 2, 2)])
def test_masked_forward(dtype, hn, sq, sk, b, np_, nkv):
    """Random masks, a whole tile hidden from every query, and rows that see nothing: those are averages over all keys."""
    from megatron.model.fused_attention import masked_attention

    q, k, v = operands(dtype, sq, sk, b, np_, nkv, hn, 21)
    mask = torch.rand((b, 1, sq, sk), generator=torch.Generator().manual_seed(3)).to(DEV) < 0.6
    mask[:, :, :, 64:128] = True
    mask[0, :, -1] = True
    for m in (mask, mask[:1], hidden(sq, sk).view(1, 1, sq, sk)):
        for fill in (-10000.0, torch.finfo(torch.float32).min):
            out = masked_attention(q, k, v, m, 1 / math.sqrt(hn), fill, merged=True)
            assert rel_err(out.view(sq, b, np_, hn), textbook(q, k, v, m, fill)) <= limit(dtype, 2)


def test_masked_scores_as_low_as_the_fill_value_count():
    """With visible scores around -10000 the masked keys of the padding-mask kernel take part in the softmax."""
    from megatron.model.fused_attention import masked_attention

    q, k, v = operands(torch.bfloat16, 96, 192, 1, 4, 4, 64, 5)
    q[..., 0], k[..., 0] = 250.0, -320.0   # every score is near -80000 / 8
    mask = hidden(96, 192).view(1, 1, 96, 192)
    out = masked_attention(q, k, v, mask, 1 / 8, -10000.0, merged=True)
    want = textbook(q, k, v, mask, -10000.0)
    assert rel_err(want, textbook(q, k, v, mask)) > 0.1   # the masked keys matter
    # scores of 1e4 carry an fp32 rounding of up to 2^-11 here and in the reference: 1e-3 of a probability
    assert rel_err(out.view(96, 1, 4, 64), want) <= limit(torch.bfloat16, 2) + 2e-3


def test_the_caller_takes_the_kernels_and_the_mask_where_it_counts():
    """``CoreAttention``: a prompt of a length that the softmax gate rejects (forward only) attends by the mask it is
    given; with a gradient wanted, or a mask function that does not fill, the reference's torch branch stays."""
    from megatron.model import fused_attention
    from megatron.model.attention_core import CoreAttention
    from megatron.model.fused_softmax import SoftmaxFusionTypes as T

    def fills(scores, mask):
        return scores.masked_fill_(mask, torch.finfo(scores.dtype).min)

    def penalises(scores, mask):
        return scores - 2.0 * mask.to(scores.dtype)

    s, b, np_, hn = 77, 2, 4, 64
    q, k, v = operands(torch.bfloat16, s, s, b, np_, np_, hn, 31)
    mask = hidden(s, s).view(1, 1, s, s).repeat(b, 1, 1, 1)
    mask[1, :, :, :20] = True   # left padding: the first rows of the second entry see nothing
    want = textbook(q, k, v, mask)
    core = CoreAttention(hn, 1, False, True, T.upper_triang, fills, attention_softmax_in_fp32=True)
    soft = CoreAttention(hn, 1, False, True, T.upper_triang, penalises, attention_softmax_in_fp32=True)
    assert soft.scale_mask_softmax.mask_fill is None and core.scale_mask_softmax.mask_fill == torch.finfo(torch.float32).min
    assert core._one_kernel(q, k, v, mask, None, False) is not None
    assert soft._one_kernel(q, k, v, mask, None, False) is None
    assert core._one_kernel(q.clone().requires_grad_(True), k, v, mask, None, False) is None
    assert rel_err(core(q, k, v, mask).permute(2, 0, 1, 3), want) <= limit(torch.bfloat16, 2)
    # the torch branch rounds the scores to bf16 first: one more rounding, of a score of up to 4 instead of a value
    assert rel_err(core(q.clone().requires_grad_(True), k, v, mask).permute(2, 0, 1, 3), want) <= 2.0 ** -7
    assert not fused_attention.supported(q[..., :40], k[..., :40], v[..., :40])


def test_the_caller_refuses_operands_that_do_not_belong_together():
    """``CoreAttention`` leaves them to the products, which raise (the checks themselves: test_attention_operands.py)."""
    from megatron.model.attention_core import CoreAttention
    from megatron.model.fused_softmax import SoftmaxFusionTypes as T

    core = CoreAttention(64, 1, False, True, T.upper_triang, lambda s, m: s.masked_fill_(m, -1e4), attention_softmax_in_fp32=True)
    q, k, v = operands(torch.bfloat16, 128, 128, 4, 4, 4, 64, 1)
    mask = hidden(128, 128).view(1, 1, 128, 128)
    for grad in (False, True):
        for key, value in ((k[:, :2], v[:, :2]), (k[:, :1], v[:, :1]), (k.repeat(1, 2, 1, 1), v.repeat(1, 2, 1, 1)), (k.cpu(), v.cpu()),
                           (k, v.cpu()), (k[:, :, :3], v[:, :, :3])):
            with pytest.raises((RuntimeError, AssertionError)):
                core(q.clone().requires_grad_(grad), key, value, mask)
        with pytest.raises(RuntimeError):
            core(q.cpu().requires_grad_(grad), k, v, mask)


@pytest.mark.parametrize("merged", [True, False], ids=["merged", "bnsh"])
def test_the_context_may_be_changed_in_place(merged):
    """As the product's result may be: the gradients are those of the same change into new memory, bit for bit."""
    from megatron.model.attention_core import CoreAttention
    from megatron.model.fused_softmax import SoftmaxFusionTypes as T

    core = CoreAttention(64, 1, False, True, T.upper_triang, lambda s, m: s.masked_fill_(m, -1e4), attention_softmax_in_fp32=True)
    mask = hidden(128, 128).view(1, 1, 128, 128)
    results = []
    for change in (lambda t: t.mul_(0.5).add_(1.0), lambda t: t.mul(0.5).add(1.0)):
        leaves = [t.requires_grad_(True) for t in operands(torch.bfloat16, 128, 128, 2, 4, 2, 64, 1)]
        out = change(core(*leaves, mask, merged_heads=merged))
        out.square().sum().backward()
        results.append([util.raw_bits(t) for t in (out.detach(), *(leaf.grad for leaf in leaves))])
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("kind", ["subtracts 1e5", "-inf"])
def test_rows_that_see_nothing_follow_the_mask_function(kind):
    """A function that subtracts leaves the softmax of the scores in a row that sees nothing, -inf leaves NaN; a fill leaves
    the average. Left padding, without a gradient, a length that the softmax gate refuses."""
    from megatron.model.attention_core import CoreAttention
    from megatron.model.fused_softmax import SoftmaxFusionTypes as T

    func = {"subtracts 1e5": lambda s, m: s - 1e5 * m.to(s.dtype), "-inf": lambda s, m: s.masked_fill(m, float("-inf"))}[kind]
    q, k, v = operands(torch.bfloat16, 77, 77, 1, 4, 4, 64, 31)
    mask = hidden(77, 77).view(1, 1, 77, 77).clone()
    mask[:, :, :, :20] = True
    core = CoreAttention(64, 1, False, True, T.upper_triang, func, attention_softmax_in_fp32=True)
    got = core(q, k, v, mask).float()
    scores = torch.matmul(q.float().permute(1, 2, 0, 3).contiguous(), k.float().permute(1, 2, 3, 0).contiguous()) / 8
    want = torch.matmul(torch.softmax(func(scores, mask), -1), v.float().permute(1, 2, 0, 3).contiguous())
    assert torch.equal(got.isnan(), want.isnan()) and bool(want[:, :, :20].isnan().all()) == (kind == "-inf")
    # scores of up to 4 are rounded to bf16 first; beside 1e5 an fp32 score keeps 2^-7
    assert rel_err(got[~want.isnan()], want[~want.isnan()]) <= 2.0 ** -6


def test_a_hook_on_the_softmax_module_sees_the_probabilities():
    """While it is there the probabilities are formed; the result agrees with the kernel's."""
    from megatron.model.attention_core import CoreAttention
    from megatron.model.fused_softmax import SoftmaxFusionTypes as T

    core = CoreAttention(64, 1, False, True, T.upper_triang, lambda s, m: s.masked_fill_(m, -1e4), attention_softmax_in_fp32=True)
    q, k, v = operands(torch.bfloat16, 128, 128, 2, 4, 4, 64, 1)
    mask, seen = hidden(128, 128).view(1, 1, 128, 128), []
    handle = core.scale_mask_softmax.register_forward_hook(lambda module, args, out: seen.append(out))
    with_hook = core(q, k, v, mask)
    handle.remove()
    without = core(q, k, v, mask)
    assert len(seen) == 1 and seen[0].shape == (2, 4, 128, 128) and core._one_kernel(q, k, v, mask, None, False) is not None
    # the products round the scores (up to 4, instead of a value of 1) once more
    assert rel_err(with_hook, without) <= 2.0 ** -7


@pytest.mark.parametrize("s", [128, 77], ids=["causal", "by mask"])
def test_autocast_to_another_type_keeps_its_result(s, monkeypatch):
    """The products take the type that autocast gives them, and so does the result; to their own type it changes nothing."""
    from megatron.model import fused_attention
    from megatron.model.attention_core import CoreAttention
    from megatron.model.fused_softmax import SoftmaxFusionTypes as T

    core = CoreAttention(64, 1, True, False, T.upper_triang, lambda s, m: s.masked_fill_(m, -1e4), attention_softmax_in_fp32=True)
    q, k, v = operands(torch.bfloat16, s, s, 1, 4, 4, 64, 1)
    mask = hidden(s, s).view(1, 1, s, s)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert core._one_kernel(q, k, v, mask, None, False) is not None
    with torch.autocast("cuda", dtype=torch.float16):
        assert core._one_kernel(q, k, v, mask, None, False) is None
        got = core(q, k, v, mask)
        monkeypatch.setattr(fused_attention, "supported", lambda *a: False)
        want = core(q, k, v, mask)
    assert got.dtype == want.dtype == torch.float16 and torch.equal(got, want)


@pytest.mark.parametrize("merged", [True, False], ids=["merged", "bnsh"])
def test_hooks_on_saved_tensors(merged):
    """They may keep them anywhere and hand them back in another layout: the same gradients, bit for bit."""
    from megatron.model.fused_attention import causal_attention

    def elsewhere(t):
        return t.cpu().transpose(0, -1).contiguous()   # the last dimension outermost

    g = None
    results = []
    for hooks in (None, (elsewhere, lambda t: t.to(DEV).transpose(0, -1))):
        leaves = [t.requires_grad_(True) for t in operands(torch.bfloat16, 136, 136, 2, 8, 2, 64, 1)]
        if hooks is None:
            out = causal_attention(*leaves, 1 / 8, merged=merged)
            g = util.randn(tuple(out.shape), torch.bfloat16, seed=9).to(DEV)
        else:
            with torch.autograd.graph.saved_tensors_hooks(*hooks):
                out = causal_attention(*leaves, 1 / 8, merged=merged)
        out.backward(g)
        results.append([util.raw_bits(leaf.grad) for leaf in leaves])
    assert all(torch.equal(a, b) for a, b in zip(*results))
