"""The decoding kernel (csrc/attention_decode.hip) and the cache append, against textbook attention in fp32 and torch's
concatenation: edges of the 16-key tiles, of the 32 keys of a wave and the 128 of a workgroup, positions cut into several
workgroups, one and two tiles of queries, grouped heads, strided operands, and rows that see nothing."""
import math

import pytest
import torch

from test_gpu_fused_attention import DTYPES, hidden, limit, operands, rel_err, textbook

pytestmark = pytest.mark.gpu
DEV = "cuda"


def cached(dtype, past, sq, b, np_, nkv, hn):
    q, k, v = operands(dtype, sq, past + sq, b, np_, nkv, hn, 41)
    return q, k, v, torch.stack((k[:past], v[:past]))


@DTYPES
@pytest.mark.parametrize("hn", [64, 80, 96, 128])
@pytest.mark.parametrize("past,sq,b,np_,nkv", [(3, 1, 1, 2, 2), (15, 1, 2, 3, 3), (31, 2, 1, 4, 2), (127, 1, 1, 4, 1), (126, 5, 2, 8, 2), (200, 1, 3, 4, 4),
                                               (257, 4, 1, 8, 1), (1000, 1, 1, 4, 2), (700, 16, 1, 2, 2)])
def test_decode(dtype, hn, past, sq, b, np_, nkv):
    from megatron.model.fused_attention import append_to_cache, decode_attention, decode_supported

    q, k, v, layer_past = cached(dtype, past, sq, b, np_, nkv, hn)
    sk = past + sq
    causal = hidden(sq, sk).view(1, 1, sq, sk)
    some = torch.rand((b, 1, sq, sk), generator=torch.Generator().manual_seed(3)).to(DEV) < 0.6
    some[0, 0, -1] = True   # sees nothing: an average over all keys
    kn, vn = k[past:], v[past:]
    assert decode_supported(q, kn, vn, layer_past)
    # a slice of a wider projection and a cache written heads first: the same operands with other strides
    wide = torch.cat((q, q), dim=3)[..., :hn]
    other = layer_past.permute(0, 2, 3, 1, 4).contiguous().permute(0, 3, 1, 2, 4)
    for mask, fill in ((causal, -10000.0), (causal.expand(b, 1, sq, sk), -10000.0), (some, torch.finfo(torch.float32).min), (some, -10000.0)):
        out, present = decode_attention(q, kn, vn, layer_past, mask, 1 / math.sqrt(hn), fill, merged=True)
        assert torch.equal(present, torch.stack((k, v)))
        assert rel_err(out.view(sq, b, np_, hn), textbook(q, k, v, mask, fill)) <= limit(dtype, 2)
        again, present = decode_attention(wide, kn, vn, other, mask, 1 / math.sqrt(hn), fill)
        assert torch.equal(again.permute(2, 0, 1, 3).reshape(out.shape), out) and torch.equal(present, torch.stack((k, v)))
    assert torch.equal(append_to_cache(kn, vn, layer_past), torch.stack((k, v)))
    assert torch.equal(append_to_cache(k.transpose(0, 1).contiguous().transpose(0, 1), v, None), torch.stack((k, v)))


@pytest.mark.parametrize("hn", [64, 80, 96, 128])
@pytest.mark.parametrize("past", [3, 31, 32, 63, 64, 65, 97, 128, 161, 300])
@pytest.mark.parametrize("sq,b,np_,nkv", [(1, 160, 4, 4), (1, 128, 4, 4), (2, 97, 8, 4), (1, 192, 2, 2), (9, 192, 4, 2), (1, 131, 3, 3)])
def test_many_sequences(hn, past, sq, b, np_, nkv):
    """One and two heads of keys per workgroup; rounds of 32 keys that a wave has one, two or several of."""
    from megatron.model.fused_attention import decode_attention

    q, k, v, layer_past = cached(torch.bfloat16, past, sq, b, np_, nkv, hn)
    mask = hidden(sq, past + sq).view(1, 1, sq, past + sq)
    out, present = decode_attention(q, k[past:], v[past:], layer_past, mask, 1 / math.sqrt(hn), -10000.0, merged=True)
    assert torch.equal(present, torch.stack((k, v)))
    assert rel_err(out.view(sq, b, np_, hn), textbook(q, k, v, mask, -10000.0)) <= limit(torch.bfloat16, 2)


@pytest.mark.parametrize("hn", [64, 80, 96, 128])
@pytest.mark.parametrize("past,sq,b,np_,nkv", [(767, 1, 160, 4, 4), (768, 1, 176, 4, 4), (800, 2, 100, 8, 4), (830, 1, 192, 2, 2), (911, 9, 192, 4, 2)])
def test_many_long_sequences(hn, past, sq, b, np_, nkv):
    """Two and four heads of keys per workgroup, whole and with their keys cut into parts, the last of them down to one key."""
    from megatron.model.fused_attention import decode_attention

    q, k, v, layer_past = cached(torch.bfloat16, past, sq, b, np_, nkv, hn)
    mask = hidden(sq, past + sq).view(1, 1, sq, past + sq)
    out, present = decode_attention(q, k[past:], v[past:], layer_past, mask, 1 / math.sqrt(hn), -10000.0, merged=True)
    assert torch.equal(present, torch.stack((k, v)))
    assert rel_err(out.view(sq, b, np_, hn), textbook(q, k, v, mask, -10000.0)) <= limit(torch.bfloat16, 2)


@pytest.mark.parametrize("hn,heads,b", [(64, 32, 32), (96, 32, 32), (128, 32, 16)])
def test_sums_do_not_depend_on_the_heads_of_a_workgroup(hn, heads, b):
    """With two or four heads per workgroup the same bits as with one, which is what 256 pairs get (8 sequences of 32 heads): the
    fewer sums a head's keys go into, the further off is the result."""
    from megatron.model.fused_attention import decode_attention

    q, k, v, layer_past = cached(torch.bfloat16, 800, 1, b, heads, heads, hn)
    mask = torch.zeros((1, 1, 1, 801), dtype=torch.bool, device=DEV)
    out, _ = decode_attention(q, k[800:], v[800:], layer_past, mask, 1 / math.sqrt(hn), -10000.0, merged=True)
    few, _ = decode_attention(q[:, :8], k[800:, :8], v[800:, :8], layer_past[:, :, :8], mask, 1 / math.sqrt(hn), -10000.0, merged=True)
    assert torch.equal(out[:, :8], few)


def test_nan_and_infinite_keys_stay_where_they_are():
    """A value that is not finite reaches the queries that see it and no others; the cache keeps it."""
    from megatron.model.fused_attention import decode_attention

    q, k, v, layer_past = cached(torch.bfloat16, 150, 2, 1, 4, 4, 80)
    layer_past[1, 151 - 2, 0, 1, 7] = float("nan")
    k[:150], v[:150] = layer_past
    mask = torch.zeros((1, 1, 2, 152), dtype=torch.bool, device=DEV)
    out, present = decode_attention(q, k[150:], v[150:], layer_past, mask, 0.1, -10000.0)
    want = torch.zeros((1, 4, 2, 80), dtype=torch.bool, device=DEV)
    want[:, 1, :, 7] = True
    assert torch.equal(out.isnan(), want) and present[1, 149, 0, 1, 7].isnan()


def test_what_the_kernel_does_not_take():
    """Such calls are concatenated, as before: gradients, other types, dropout, too many queries."""
    from megatron.model.attention_core import CoreAttention
    from megatron.model.fused_attention import cache_supported, decode_supported
    from megatron.model.fused_softmax import SoftmaxFusionTypes as T

    q, k, v, layer_past = cached(torch.bfloat16, 100, 2, 1, 4, 4, 64)
    k, v = k[100:], v[100:]
    core = CoreAttention(64, 1, False, True, T.upper_triang, lambda s, m: s.masked_fill_(m, torch.finfo(s.dtype).min),
                         attention_softmax_in_fp32=True, attention_dropout=0.5)
    mask = hidden(2, 102).view(1, 1, 2, 102)
    assert core.train()(q, k, v, mask, layer_past=layer_past) is None
    assert core.eval()(q, k, v, mask, layer_past=layer_past) is not None
    assert core(q, k, v, mask[..., :101], layer_past=layer_past) is None
    assert core(q.clone().requires_grad_(True), k, v, mask, layer_past=layer_past) is None
    assert not cache_supported(k, v, layer_past.float()) and not cache_supported(k, v.clone().requires_grad_(True), layer_past)
    assert not decode_supported(q, k, v, layer_past[:, :0]) and not decode_supported(q.float(), k.float(), v.float(), layer_past.float())
    many = operands(torch.bfloat16, 33, 33, 1, 4, 4, 64, 1)
    assert not decode_supported(*many, layer_past) and cache_supported(many[1], many[2], layer_past)
