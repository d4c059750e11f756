"""The host side in csrc/native.cpp against the Python functions that take what it leaves: the same kernels with the same
arguments, so the same bits, layouts and refusals, over layouts, types, partial gradients, hooks on saved tensors, modes and
repeated backward passes."""

import pytest
import torch

import util

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF16, FP16, FP32 = torch.bfloat16, torch.float16, torch.float32


class Leaves:
    """Stands for the extension module: leaves every call to Python."""

    def __getattr__(self, name):
        return lambda *a: NotImplemented


def randn(shape, dtype, seed):
    return util.randn(shape, dtype, seed=seed).to(DEV)


def wide(t):
    """The same values as a slice of something wider."""
    return torch.cat((t, t), dim=-1)[..., :t.size(-1)]


def turned(t):
    """The same values with the first two dimensions swapped in memory."""
    return t.transpose(0, 1).contiguous().transpose(0, 1)


def norm_call(kind, dtype, pdtype, layout, bias=True):
    from megatron.model.norms import LayerNorm, RMSNorm, layer_norm_pair

    x = layout(randn((5, 3, 96), dtype, 1))
    if kind == "pair":
        a, b = (LayerNorm(96, bias=bias).to(DEV).to(pdtype) for _ in range(2))
        return lambda x, *p: layer_norm_pair(x, a, b), [x] + list(a.parameters()) + list(b.parameters())
    m = (LayerNorm(96, bias=bias) if kind == "layer" else RMSNorm(96, p=0.5 if kind == "partial" else -1.0, bias=bias)).to(DEV).to(pdtype)
    return lambda x, *p: m(x), [x] + list(m.parameters())


def softmax_call(kind, layout, window=None):
    from megatron.model.fused_softmax import FusedScaleMaskSoftmax, SoftmaxFusionTypes as T

    m = FusedScaleMaskSoftmax(False, True, T.upper_triang if kind == "causal" else T.general,
                              lambda s, k: s.masked_fill_(k, -10000.0), True, 0.125, sliding_window_width=window)
    x = layout(randn((2, 4, 64, 64), BF16, 2))
    mask = torch.ones((1, 1, 64, 64), dtype=torch.bool, device=DEV).triu(1)
    return lambda x: m(x, mask if kind == "causal" else turned(mask)), [x]


def rope_call(dtype, layout, offset=0):
    from megatron.model.fused_rope import fused_apply_rotary_pos_emb_qk_cached as f
    from megatron.model.positional_embeddings import RotaryEmbedding

    cos, sin = RotaryEmbedding(32, 40, precision=dtype)(torch.empty(1, device=DEV), seq_len=40)
    return lambda q, k: f(q, k, cos, sin, offset), [layout(randn((33, 2, 4, 64), dtype, 3)), layout(randn((33, 2, 2, 64), dtype, 4))]


def split_call(grouped, layout):
    from megatron.model.attention_core import split_gqa_and_rotate, split_qkv_and_rotate
    from megatron.model.positional_embeddings import RotaryEmbedding

    rotary = RotaryEmbedding(64, 50, precision=BF16)
    past = torch.empty((2, 7, 1, 1, 1), device=DEV)
    if grouped:
        return lambda x: split_gqa_and_rotate(x, rotary, 4, 2, layer_past=past), [layout(randn((20, 2, 8 * 64), BF16, 5))]
    return lambda x: split_qkv_and_rotate(x, rotary), [layout(randn((20, 2, 4, 192), BF16, 5))]


def act_call(kind, dtype, layout):
    from megatron.model.activations import Gated_Activation, bias_gelu_impl

    x = layout(randn((7, 2, 64), dtype, 6))
    if kind == "gelu":
        return bias_gelu_impl, [x, randn((64,), dtype, 7)]
    return Gated_Activation(kind), [x]


def attention_call(layout, merged, np_=4, nkv=2, window=None):
    from megatron.model.fused_attention import causal_attention

    shapes = ((70, 2, np_, 64), (70, 2, nkv, 64), (70, 2, nkv, 64))
    return (lambda q, k, v: causal_attention(q, k, v, 0.125, window, merged)), [layout(randn(s, BF16, 8 + i)) for i, s in enumerate(shapes)]


def add_call(kind, dtype, layout):
    from megatron.model.fused_bias_dropout import bias_add_residual_pair, bias_dropout_add_fused_inference

    x, y, r = (layout(randn((6, 2, 64), dtype, 20 + i)) for i in range(3))
    b, c = randn((64,), dtype, 24), randn((64,), dtype, 25)
    if kind == "pair":
        return bias_add_residual_pair, [x, b, y, c, r]
    if kind == "plain":
        return lambda x, r: bias_dropout_add_fused_inference(x, None, r, 0.0), [x, r]
    return lambda x, b, r: bias_dropout_add_fused_inference(x, b, r, 0.0), [x, b, r]


def same(t):
    return t


CALLS = {
    **{f"{kind}-{name}": (lambda kind=kind, args=args: norm_call(kind, *args)) for kind in ("layer", "pair", "rms", "partial")
       for name, args in {"bf16": (BF16, BF16, same), "fp16 turned": (FP16, FP16, turned), "fp32 parameters": (BF16, FP32, wide),
                          "fp32": (FP32, FP32, same), "no bias": (BF16, BF16, same, False)}.items()},
    "softmax causal": lambda: softmax_call("causal", same), "softmax window": lambda: softmax_call("causal", same, 5),
    "softmax general": lambda: softmax_call("general", same), "softmax general strided": lambda: softmax_call("general", turned),
    "rope": lambda: rope_call(BF16, same), "rope wide": lambda: rope_call(FP16, wide), "rope offset": lambda: rope_call(FP32, turned, 7),
    "split": lambda: split_call(False, same), "split turned": lambda: split_call(False, turned), "split grouped": lambda: split_call(True, same),
    "gelu": lambda: act_call("gelu", BF16, same), "gelu fp32": lambda: act_call("gelu", FP32, wide), "swiglu": lambda: act_call("swiglu", BF16, same),
    "geglu": lambda: act_call("geglu", FP16, turned),
    "attention": lambda: attention_call(same, True), "attention wide": lambda: attention_call(wide, False),
    "attention turned": lambda: attention_call(turned, True, 3, 3, 9),
    "attention odd": lambda: attention_call(lambda t: torch.cat((t, t[..., :4]), dim=-1)[..., :64], True),
    "add pair": lambda: add_call("pair", BF16, same), "add": lambda: add_call("bias", FP16, turned), "add plain": lambda: add_call("plain", BF16, same),
}


def outputs(y):
    return list(y) if isinstance(y, (tuple, list)) else [y]


def described(t):
    return None if t is None else (tuple(t.shape), t.dtype, t.stride(), t.requires_grad)


def attempt(call, *args):
    try:
        return call(*args)
    except Exception as e:   # noqa: BLE001  (the kind of refusal is what is compared)
        return e


def both(monkeypatch, call):
    """What ``call`` gives natively and in Python."""
    from megatron.fused_kernels import _hotpath as hp

    here = call()
    with monkeypatch.context() as m:
        m.setattr(hp, "native", Leaves)
        there = call()
    assert len(here) == len(there)
    for x, y in zip(here, there):
        if isinstance(y, Exception) or isinstance(x, Exception):
            assert type(x) is type(y), (x, y)
        elif isinstance(y, torch.Tensor) and isinstance(x, torch.Tensor):
            assert described(x) == described(y)
            assert torch.equal(util.raw_bits(x.detach().contiguous()), util.raw_bits(y.detach().contiguous()))
        else:
            assert x == y or (x is None and y is None)


def prepared(make, wanted=None):
    call, inputs = make()
    leaves = [t.detach().requires_grad_(wanted is None or i in wanted) for i, t in enumerate(inputs)]
    # (parameters of a module are its own; they are what the call uses)
    return call, [own if isinstance(own, torch.nn.Parameter) else leaf for own, leaf in zip(inputs, leaves)]


def backward(y, inputs, **kw):
    grads = [util.randn(tuple(t.shape), t.dtype, seed=50 + i).to(DEV) for i, t in enumerate(y)]
    return torch.autograd.grad(y, [t for t in inputs if t.requires_grad], grads, allow_unused=True, **kw)


@pytest.mark.parametrize("name", CALLS)
def test_results_and_gradients(name, monkeypatch):
    def whole():
        torch.manual_seed(0)
        call, inputs = prepared(CALLS[name])
        y = outputs(call(*inputs))
        return y + list(backward(y, inputs))

    both(monkeypatch, whole)


@pytest.mark.parametrize("name", CALLS)
def test_some_gradients_no_gradients_and_one_output(name, monkeypatch):
    def some():
        result = []
        for i in range(3):
            call, inputs = prepared(CALLS[name], {i})
            if any(t.requires_grad for t in inputs):
                y = outputs(call(*inputs))
                result += [t for t in y] + list(backward(y, inputs))
        return result

    def none():
        call, inputs = prepared(CALLS[name])
        with torch.no_grad():
            result = outputs(call(*inputs))
        with torch.inference_mode():
            return result + [t.is_inference() for t in outputs(call(*inputs))]

    def one():
        call, inputs = prepared(CALLS[name])
        y = outputs(call(*inputs))
        return list(torch.autograd.grad(y[-1].float().sum(), [t for t in inputs if t.requires_grad], allow_unused=True))

    for run in (some, none, one):
        both(monkeypatch, run)


@pytest.mark.parametrize("name", CALLS)
def test_hooks_on_saved_tensors(name, monkeypatch):
    """Hooks that hand tensors back from another place; their copies are what the backward uses."""
    def away():
        call, inputs = prepared(CALLS[name])
        with torch.autograd.graph.save_on_cpu():
            y = outputs(call(*inputs))
        return y + list(backward(y, inputs))

    def checkpointed():
        call, inputs = prepared(CALLS[name])
        y = outputs(torch.utils.checkpoint.checkpoint(call, *inputs, use_reentrant=False))
        return y + list(backward(y, inputs))

    both(monkeypatch, away)
    both(monkeypatch, checkpointed)


@pytest.mark.parametrize("name", CALLS)
def test_second_backward_and_changes_in_place(name, monkeypatch):
    def twice():
        call, inputs = prepared(CALLS[name])
        y = outputs(call(*inputs))
        first = list(backward(y, inputs, retain_graph=True))
        second = list(backward(y, inputs))
        third = attempt(backward, y, inputs)
        return first + second + ([third] if isinstance(third, Exception) else list(third))

    def changed():
        call, inputs = prepared(CALLS[name])
        y = outputs(call(*inputs))
        with torch.no_grad():
            inputs[0].mul_(1.5)
        got = attempt(backward, y, inputs)
        return [got] if isinstance(got, Exception) else list(got)

    def result_changed():
        call, inputs = prepared(CALLS[name])
        y = outputs(call(*inputs))
        got = [attempt(lambda t=t: t.mul_(2.0)) for t in y]
        got = [g for g in got if isinstance(g, Exception)]
        grads = attempt(backward, y, inputs)
        return got + ([grads] if isinstance(grads, Exception) else list(grads))

    def of_gradients():
        call, inputs = prepared(CALLS[name])
        y = outputs(call(*inputs))
        seeds = [util.randn(tuple(t.shape), t.dtype, seed=50 + i).to(DEV).requires_grad_() for i, t in enumerate(y)]
        grads = torch.autograd.grad(y, [t for t in inputs if t.requires_grad], [s * 1 for s in seeds], create_graph=True, allow_unused=True)
        return list(grads)

    for run in (twice, changed, result_changed, of_gradients):
        both(monkeypatch, run)


@pytest.mark.parametrize("name", CALLS)
def test_what_torch_follows_stays_in_python(name, monkeypatch):
    """Forward mode, function transforms and modes see what they always saw."""
    class Count(torch.utils._python_dispatch.TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.seen = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen.append(str(func))
            return func(*args, **(kwargs or {}))

    def dual():
        call, inputs = prepared(CALLS[name])
        with torch.autograd.forward_ad.dual_level():
            first = torch.autograd.forward_ad.make_dual(inputs[0].detach(), torch.ones_like(inputs[0]))
            got = attempt(call, first, *inputs[1:])
        return [got] if isinstance(got, Exception) else [described(t) for t in outputs(got)]

    def mapped():
        call, inputs = prepared(CALLS[name])
        got = attempt(lambda: torch.func.vmap(lambda x: outputs(call(x, *inputs[1:]))[0])(torch.stack([inputs[0].detach()] * 2)))
        return [type(got).__name__ if isinstance(got, Exception) else described(got)]

    def counted():
        call, inputs = prepared(CALLS[name])
        with Count() as mode:
            call(*inputs)
        return list(mode.seen)

    for run in (dual, mapped, counted):
        both(monkeypatch, run)


def test_operands_that_do_not_fit_are_refused_as_before(monkeypatch):
    from megatron.model.activations import bias_gelu_impl
    from megatron.model.fused_attention import causal_attention
    from megatron.model.fused_bias_dropout import bias_add_residual_pair
    from megatron.model.fused_rope import fused_apply_rotary_pos_emb_qk_cached
    from megatron.model.norms import LayerNorm, RMSNorm

    x, y = randn((4, 2, 64), BF16, 1), randn((4, 2, 64), FP16, 1)
    q = randn((8, 1, 4, 64), BF16, 2)
    cos = randn((8, 1, 1, 32), BF16, 3)
    calls = [lambda: LayerNorm(64).to(DEV).half()(x), lambda: LayerNorm(64)(x), lambda: RMSNorm(64).to(DEV).half()(x), lambda: LayerNorm(64).to(DEV)(x.double()),
             lambda: bias_gelu_impl(x, randn((32,), BF16, 1)), lambda: bias_gelu_impl(x, y[0, 0]), lambda: bias_gelu_impl(x.cpu(), x[0, 0].cpu()),
             lambda: bias_add_residual_pair(x, None, y, None, x), lambda: bias_add_residual_pair(x, None, x, None, x[:2]),
             lambda: fused_apply_rotary_pos_emb_qk_cached(q, q, cos, cos, offset=1), lambda: fused_apply_rotary_pos_emb_qk_cached(q, q.half(), cos, cos),
             lambda: fused_apply_rotary_pos_emb_qk_cached(q, q, cos.half(), cos.half()), lambda: causal_attention(q, q[:4], q[:4], 0.1),
             lambda: causal_attention(q, q.half(), q.half(), 0.1), lambda: LayerNorm(64).to(DEV).bfloat16()(x[:0])]

    def all_of_them():
        return [str(got) if isinstance(got, Exception) else described(got) for got in map(attempt, calls)]

    both(monkeypatch, all_of_them)


def test_inference_calls(monkeypatch):
    """Few-row layers, decoding, the cache and attention by a mask, which have no gradient."""
    from megatron.model.fused_attention import append_to_cache, checked_decode_attention, masked_attention
    from megatron.model.fused_linear import linear

    w, b = randn((48, 64), BF16, 1), randn((48,), BF16, 2)
    q, k, v = (randn((3, 2, n, 64), BF16, 3 + n) for n in (4, 2, 2))
    past = randn((2, 37, 2, 2, 64), BF16, 9)
    mask = torch.rand((2, 1, 3, 40), generator=torch.Generator().manual_seed(1)).to(DEV) < 0.4
    keys = randn((40, 2, 2, 64), BF16, 11)

    def calls():
        result = [linear(randn((r, 64), BF16, 5), w, bias) for r in (1, 16, 33) for bias in (None, b)]
        result += [linear(wide(randn((4, 64), BF16, 5)), w, None), linear(randn((0, 64), BF16, 5), w, None)]
        with torch.autocast("cuda", dtype=FP16):
            result.append(linear(randn((4, 64), BF16, 5), w, b))
        for cached in (past, turned(past.transpose(0, 1)).transpose(0, 1), past.permute(0, 2, 3, 1, 4).contiguous().permute(0, 3, 1, 2, 4)):
            result += list(checked_decode_attention(wide(q), k, turned(v), cached, mask, 0.125, -10000.0, True))
            result += list(checked_decode_attention(q, k, v, cached, mask[:1], 0.125, -10000.0, False))
            result.append(append_to_cache(k, wide(v), cached, checked=True))
        result.append(append_to_cache(k, v, None, checked=True))
        return result + [masked_attention(wide(q), keys, keys, m, 0.125, -10000.0, merged) for m in (mask, mask[:1]) for merged in (True, False)]

    with torch.no_grad():
        both(monkeypatch, calls)


def test_another_stream_and_thread():
    """The backward runs where autograd puts it: on the forward's stream, from a thread of its own."""
    import threading

    call, inputs = prepared(CALLS["layer-bf16"])
    want = backward(outputs(call(*inputs)), inputs)
    torch.cuda.synchronize()
    got, failed = [None] * 4, []

    def work(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                got[i] = backward(outputs(call(*inputs)), inputs)
            stream.synchronize()
        except Exception as e:   # noqa: BLE001
            failed.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not failed
    assert all(torch.equal(a, b) for result in got for a, b in zip(result, want))


def test_other_threads_run_during_a_call():
    """Allocations and launches leave the interpreter's lock to others. The calls follow each other without any of this thread's
    own bytecode in between, where it would hand over the lock anyway (one that is left to a busy thread comes back after 5 ms)."""
    import collections
    import itertools
    import threading
    import time

    from megatron.fused_kernels import _hotpath as hp

    x, w, rows = randn((8, 64), BF16, 1), randn((64, 64), BF16, 2), randn((64,), BF16, 3)
    with torch.no_grad():
        for call, args in ((hp.native().layer_norm, (x, rows, rows, 1e-5)), (hp.native().linear, (x, w, None, 16, 32))):
            ticks, stop = [], threading.Event()

            def tick():
                while not stop.is_set():
                    ticks.append(time.perf_counter())

            other = threading.Thread(target=tick)
            other.start()
            start = time.perf_counter()
            collections.deque(itertools.starmap(call, itertools.repeat(args, 100)), maxlen=0)
            end = time.perf_counter()
            stop.set()
            other.join()
            quarters = {int(4 * (t - start) / (end - start)) for t in ticks if start <= t < end}
            assert {1, 2} <= quarters, (quarters, end - start)
