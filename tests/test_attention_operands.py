"""Operands that do not belong together never reach the attention kernels, which are handed addresses and the sizes of q: the
checks of ``megatron.model.fused_attention`` on stand-ins that have a GPU tensor's type, shape and device but no memory.
Nothing is launched (the library is out of reach)."""
import pytest
import torch

from megatron.model import fused_attention as fa

BF16 = torch.bfloat16


class Standin(torch.Tensor):
    @staticmethod
    def __new__(cls, *shape, dtype=BF16, device="cuda:0"):
        return torch.Tensor._make_wrapper_subclass(cls, shape, dtype=dtype, device=device)

    __torch_function__ = torch._C._disabled_torch_function_impl

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        if func is torch.ops.aten.unbind.int:   # layer_past -> cached keys, cached values
            t = args[0]
            return [Standin(*t.shape[1:], dtype=t.dtype, device=t.device) for _ in range(t.shape[0])]
        raise AssertionError(f"{func} on a stand-in: an operand was used before it was refused")


@pytest.fixture(autouse=True)
def out_of_reach(monkeypatch):
    def no_library():
        raise AssertionError("the kernels were reached")

    monkeypatch.setattr(fa._hp, "lib", no_library)
    monkeypatch.setattr(fa, "plain", lambda *tensors: True)   # stand-ins are followed by torch, real tensors are not


def operands(sq=8, sk=8, b=4, np_=8, nkv=4, hn=64, **kw):
    return Standin(sq, b, np_, hn, **kw), Standin(sk, b, nkv, hn, **kw), Standin(sk, b, nkv, hn, **kw)


def mask(sq=8, sk=8, b=1, dtype=torch.bool, device="cuda:0"):
    return Standin(b, 1, sq, sk, dtype=dtype, device=device)


Q, K, V = operands()
STRANGERS = {
    "fewer batch entries in k and v": (Q, Standin(8, 2, 4, 64), Standin(8, 2, 4, 64)),
    "one batch entry in k and v": (Q, Standin(8, 1, 4, 64), Standin(8, 1, 4, 64)),
    "more batch entries in k and v": (Q, Standin(8, 5, 4, 64), Standin(8, 5, 4, 64)),
    "k on the CPU": (Q, Standin(8, 4, 4, 64, device="cpu"), V),
    "v on the CPU": (Q, K, Standin(8, 4, 4, 64, device="cpu")),
    "k and v on another GPU": (Q, Standin(8, 4, 4, 64, device="cuda:1"), Standin(8, 4, 4, 64, device="cuda:1")),
    "q on the CPU": (Standin(8, 4, 8, 64, device="cpu"), K, V),
    "heads that do not divide": (Q, Standin(8, 4, 3, 64), Standin(8, 4, 3, 64)),
    "more key heads than query heads": (Q, Standin(8, 4, 16, 64), Standin(8, 4, 16, 64)),
    "another head size in k and v": (Q, Standin(8, 4, 4, 128), Standin(8, 4, 4, 128)),
    "another head size in v": (Q, K, Standin(8, 4, 4, 128)),
    "another length in v": (Q, K, Standin(9, 4, 4, 64)),
    "another type in v": (Q, K, Standin(8, 4, 4, 64, dtype=torch.float16)),
    "three dimensions in q": (Standin(8, 4, 64), K, V),
    "a head size without a kernel": operands(hn=72),
    "more queries than keys": operands(sq=9),
    "rows of 2^24 elements": operands(sq=2, sk=2, b=2048, np_=64, nkv=64, hn=128),
    "rows of 2^24 elements in k and v alone": operands(sq=1, sk=2, b=2048, np_=64, nkv=64, hn=128),
    "2^24 workgroups": operands(sq=128, sk=128, b=1 << 24, np_=1, nkv=1),
}


def test_what_belongs_together_is_taken():
    for kw in ({}, {"dtype": torch.float16}, {"sq": 1}, {"nkv": 8}, {"nkv": 1}, {"hn": 80}, {"hn": 128, "sq": 4096, "sk": 4096},
               {"sq": 1, "sk": 1, "b": 2048, "np_": 64, "nkv": 64, "hn": 128}):
        assert fa.supported(*operands(**kw)), kw
    assert fa.decode_supported(*operands(sq=2, sk=2), Standin(2, 100, 4, 4, 64))
    for b in (1, 4):
        assert fa.mask_supported(mask(2, 102, b), 4, 2, 102, Q.device)


@pytest.mark.parametrize("why", STRANGERS)
def test_strangers_are_refused_before_any_launch(why):
    q, k, v = STRANGERS[why]
    assert not fa.supported(q, k, v)
    past = Standin(2, 100, *k.shape[1:])
    assert not fa.decode_supported(q, k, v, past)
    for call in (lambda: fa.causal_attention(q, k, v, 0.1), lambda: fa.masked_attention(q, k, v, mask(q.size(0), k.size(0)), 0.1, -1e4),
                 lambda: fa.decode_attention(q, k, v, past, mask(q.size(0), 100 + k.size(0)), 0.1, -1e4)):
        with pytest.raises(RuntimeError, match="do not take these operands"):
            call()


def test_masks_that_do_not_fit():
    for m in (mask(8, 7), mask(7, 8), mask(8, 8, 2), mask(dtype=torch.uint8), mask(device="cpu"), mask(device="cuda:1"),
              Standin(8, 8, dtype=torch.bool), Standin(1, 2, 8, 8, dtype=torch.bool)):
        assert not fa.mask_supported(m, 4, 8, 8, Q.device)
        with pytest.raises(RuntimeError, match="do not take these operands"):
            fa.masked_attention(Q, K, V, m, 0.1, -1e4)
    assert not fa.mask_supported(mask(4, 65537), 1, 4, 65537, Q.device)
    assert not fa.mask_supported(mask(512, 512, 1 << 17), 1 << 17, 512, 512, Q.device)


def test_caches_that_do_not_fit():
    q, k, v = operands(sq=2, sk=2)
    more, short = operands(sq=3, sk=3), operands(sq=1, sk=2)
    for query, key, value, past in ((q, k, v, Standin(2, 100, 2, 4, 64)), (q, k, v, Standin(2, 100, 4, 2, 64)), (q, k, v, Standin(2, 0, 4, 4, 64)),
                                    (q, k, v, Standin(2, 100, 4, 4, 64, device="cpu")), (q, k, v, Standin(2, 100, 4, 4, 64, dtype=torch.float16)),
                                    (q, k, v, Standin(2, 1, 4, 4, 64)), (short[0], short[1], short[2], Standin(2, 100, 4, 4, 64)),
                                    (q, more[1], more[2], Standin(2, 100, 4, 4, 64))):
        assert not fa.decode_supported(query, key, value, past)
        with pytest.raises(RuntimeError, match="do not take these operands"):
            fa.decode_attention(query, key, value, past, mask(2, 102), 0.1, -1e4)
    for past in (Standin(2, 100, 2, 4, 64), Standin(2, 100, 4, 4, 64, device="cpu"), Standin(2, 100, 4, 4, 64, dtype=torch.float16)):
        with pytest.raises(RuntimeError, match="do not take these operands"):
            fa.append_to_cache(k, v, past)
    with pytest.raises(RuntimeError, match="do not take these operands"):
        fa.append_to_cache(k, Standin(2, 4, 4, 64, device="cpu"), None)
