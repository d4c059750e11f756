"""Scores -> probabilities -> context in one kernel on MI355X.

What ``ParallelSelfAttention.attention`` (megatron/model/transformer.py:526-625) computes with two batched GEMMs and
the fused softmax between them, for the cases in which nothing is added to the scores and nothing is dropped: the
kernels of ``csrc/attention.hip`` form scores, row statistics and context on the matrix cores tile by tile, so the
``[b, np, sq, sk]`` tensors (scores, probabilities and their gradients) do not exist. Scores, statistics and sums are
fp32; the probabilities are rounded to the storage type before the second product, as they are between the GEMMs.

Layouts as in ``CoreAttention``: q ``[sq, b, np, hn]``, k and v ``[sk, b, nkv, hn]`` with ``nkv`` dividing ``np``, any
strides with contiguous features.
"""
import ctypes

import torch
from torch.nn.modules.module import _has_any_global_hook

from ..fused_kernels import _hotpath as _hp

HEAD_DIMS = (64, 80, 96, 128)
_I64x3 = ctypes.c_int64 * 3


def _strides(t):
    """Element strides of the first three dimensions; that of a dimension of one entry means nothing and is 0."""
    return tuple(st if n > 1 else 0 for st, n in zip(t.stride()[:3], t.shape))


def _readable(t):
    """``t``, or a copy where the kernels cannot read it: they want contiguous features and 16-byte aligned rows."""
    return _operand(t)[0]


def _strides3(t):
    return _I64x3(*_strides(t))


def _operand(t):
    """``_readable`` and the strides that the entry points take."""
    s = _strides(t)
    if t.stride(3) == 1 and (s[0] | s[1] | s[2]) % 8 == 0 and t.data_ptr() % 16 == 0 and s[0] < 1 << 24:
        return t, _I64x3(*s)
    t = t.clone(memory_format=torch.contiguous_format)
    return t, _strides3(t)


def supported(q, k, v):
    """Whether the kernels take these operands. They get addresses and the sizes of q alone, so everything that makes q, k
    and v belong together is checked here: one device and type, one batch, heads that divide, a head size there is a kernel
    for, no more queries than keys, and sizes that the kernels can address."""
    device, dtype, shape, kv_shape = q.device, q.dtype, q.shape, k.shape
    if not (q.is_cuda and (dtype is torch.bfloat16 or dtype is torch.float16) and k.dtype is dtype and v.dtype is dtype
            and k.device == device and v.device == device and len(shape) == 4 and len(kv_shape) == 4 and v.shape == kv_shape):
        return False
    sq, b, np_, hn = shape
    sk, kv_b, nkv, kv_hn = kv_shape
    return (hn in HEAD_DIMS and kv_hn == hn and kv_b == b > 0 and nkv > 0 < np_ and np_ % nkv == 0 and 0 < sq <= sk
            and _addressable(sq, sk, b, np_, nkv, hn))


def _addressable(sq, sk, b, np_, nkv, hn):
    """The limits of the entry points (fill_operand and the grids in csrc/attention.hip): a row of a contiguous copy, of
    the result or of a gradient is below 2^24 elements, and a grid of 256 work-items a workgroup below 2^32."""
    return (sk < 1 << 24 and (sq == 1 or b * np_ * hn < 1 << 24) and (sk == 1 or b * nkv * hn < 1 << 24)
            and (b * np_ + 7) // 8 * 8 * ((sk + 127) // 128) < 1 << 24 and sk * b * nkv * hn < 1 << 35)


def mask_supported(mask, b, sq, sk, device):
    """Whether the kernels take ``mask`` for ``sq`` queries over ``sk`` keys of ``b`` batch entries."""
    return (mask.dtype == torch.bool and mask.device == device and mask.shape in ((1, 1, sq, sk), (b, 1, sq, sk))
            and sk <= 65536 and mask.size(0) * sq < 1 << 26)


def _refuse_unless(taken, who, *tensors):
    if not taken:
        raise RuntimeError(f"{who}: the kernels do not take these operands: "
                           + ", ".join(f"{tuple(t.shape)} {t.dtype} on {t.device}" for t in tensors))


def _new_context(q, merged):
    """Memory for the context in the layout that the caller of ``CoreAttention`` gets, ``[sq, b, np * hn]`` with ``merged`` and
    ``[b, np, sq, hn]`` without, and its strides over position, batch entry and head. (Made in that shape, not as a view of
    another: a view inside an autograd function is closed to changes in place, one outside costs a node of the graph.)"""
    sq, b, np_, hn = q.shape
    if merged:
        return torch.empty((sq, b, np_ * hn), dtype=q.dtype, device=q.device), _I64x3(b * np_ * hn if sq > 1 else 0, np_ * hn, hn)
    return torch.empty((b, np_, sq, hn), dtype=q.dtype, device=q.device), _I64x3(hn, np_ * sq * hn, sq * hn)


def _launch(out, out_strides, kept, lse, q, k, v, strides, bits, mask_batches, fill, scale, window, who):
    """``out`` and ``out_strides`` from ``_new_context``, ``kept`` laid out like ``out``, or None; q, k, v and ``strides`` from
    ``_operand``."""
    sq, b, np_, hn = q.shape
    with _hp.device_guard(q):
        rc = _hp.lib().nhp_attention_fwd_keep(
            out.data_ptr(), None if kept is None else kept.data_ptr(), None if lse is None else lse.data_ptr(), q.data_ptr(),
            k.data_ptr(), v.data_ptr(), None if bits is None else bits.data_ptr(), mask_batches, fill, scale,
            -1 if window is None else window, b, np_, k.size(2), sq, k.size(0), hn, *strides, out_strides, _hp.dtype_code(q, who), _hp.stream_of(q))
    _hp.check(rc, who)


class CausalAttention(torch.autograd.Function):
    """``softmax(scale * q k^T) v`` under the causal mask (by index, with an optional sliding window).

    The backward needs the context. The caller may change it in place (the products would not mind: their backward does not
    use it), so the kernel stores it a second time for the backward."""

    @staticmethod
    def forward(ctx, q, k, v, scale, window, merged, checked=False):
        """``checked``: the caller has asked ``supported`` already (twice would cost a short call 8 of 155 us)."""
        _refuse_unless(checked or supported(q, k, v), "CausalAttention", q, k, v)
        (q, q_strides), (k, k_strides), (v, v_strides) = _operand(q), _operand(k), _operand(v)
        out, out_strides = _new_context(q, merged)
        need = any(ctx.needs_input_grad[:3])
        kept = torch.empty_like(out) if need else None
        lse = torch.empty((q.size(1) * q.size(2), q.size(0)), dtype=torch.float32, device=q.device) if need else None
        _launch(out, out_strides, kept, lse, q, k, v, (q_strides, k_strides, v_strides), None, 1, 0.0, scale, window, "CausalAttention")
        if need:
            ctx.save_for_backward(q, k, v, kept, lse)
            ctx.conf = (scale, window, merged, out_strides)
        return out

    @staticmethod
    def backward(ctx, grad):
        who = "CausalAttention backward"
        # (a hook on saved tensors may hand them back laid out otherwise)
        q, k, v, out, lse = ctx.saved_tensors
        (q, q_strides), (k, k_strides), (v, v_strides) = _operand(q), _operand(k), _operand(v)
        out, lse = out.contiguous(), lse.contiguous()
        scale, window, merged, out_strides = ctx.conf
        sq, b, np_, hn = q.shape
        sk, nkv = k.size(0), k.size(2)
        g, g_strides = _operand(grad.reshape(sq, b, np_, hn) if merged else grad.permute(2, 0, 1, 3))
        dq, dk, dv = torch.empty_like(q, memory_format=torch.contiguous_format), torch.empty_like(
            k, memory_format=torch.contiguous_format), torch.empty_like(v, memory_format=torch.contiguous_format)
        lib = _hp.lib()
        workspace = torch.empty(lib.nhp_attention_bwd_workspace_bytes(b, np_, nkv, sq, sk, hn), dtype=torch.uint8, device=q.device)
        with _hp.device_guard(q):
            rc = lib.nhp_attention_bwd(
                dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), g.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                out.data_ptr(), lse.data_ptr(), workspace.data_ptr(), scale, -1 if window is None else window, b, np_, nkv,
                sq, sk, hn, _strides3(dq), _strides3(dk), _strides3(dv), g_strides, q_strides, k_strides, v_strides, out_strides,
                _hp.dtype_code(q, who), _hp.stream_of(q))
        _hp.check(rc, who)
        needs = ctx.needs_input_grad
        return dq if needs[0] else None, dk if needs[1] else None, dv if needs[2] else None, None, None, None, None


def causal_attention(q, k, v, scale, window=None, merged=False, checked=False):
    """Context of q ``[s, b, np, hn]`` over k, v ``[s, b, nkv, hn]``: ``[b, np, s, hn]``, or with ``merged``
    ``[s, b, np * hn]``. Query i attends to keys ``i - window .. i``. ``checked``: the caller has asked
    ``supported`` already."""
    if not _hp._is_compiling():
        out = _hp.native().causal_attention(q, k, v, float(scale), -1 if window is None else window, merged)
        if out is not NotImplemented:
            return out
    return CausalAttention.apply(q, k, v, float(scale), window, merged, checked)


def masked_attention(q, k, v, mask, scale, fill, merged=False, checked=False):
    """Inference only: the context under a boolean mask ``[1 or b, 1, sq, sk]`` (True = masked), whose scores are
    replaced by ``fill`` after scaling. ``checked``: the caller has asked ``supported`` and ``mask_supported`` already."""
    _refuse_unless(checked or supported(q, k, v) and mask_supported(mask, q.size(1), q.size(0), k.size(0), q.device),
                   "masked_attention", q, k, v, mask)
    if not _hp._is_compiling():
        out = _hp.native().masked_attention(q, k, v, mask, float(scale), float(fill), merged)
        if out is not NotImplemented:
            return out
    (q, q_strides), (k, k_strides), (v, v_strides) = _operand(q), _operand(k), _operand(v)
    sq, sk = q.size(0), k.size(0)
    mask = mask.contiguous()
    bits = torch.empty((mask.size(0), sq, (sk + 63) // 64), dtype=torch.int64, device=q.device)
    out, out_strides = _new_context(q, merged)
    with _hp.device_guard(q):
        rc = _hp.lib().nhp_attention_mask_bits(bits.data_ptr(), mask.data_ptr(), mask.size(0), sq, sk, _hp.stream_of(q))
    _hp.check(rc, "masked_attention")
    _launch(out, out_strides, None, None, q, k, v, (q_strides, k_strides, v_strides), bits, mask.size(0), fill, float(scale), None, "masked_attention")
    return out


MAX_DECODE_ROWS = 32   # queries that share a key/value head, in nhp_attention_decode


def plain(*tensors):
    """Whether nobody differentiates these or otherwise follows what is done with them."""
    return not (torch.is_grad_enabled() and any(t.requires_grad for t in tensors)) and not _hp.followed(*tensors)


_AS_WRITTEN = {}
_Module = torch.nn.Module
_CALL = _Module.__call__


def as_written(cls):
    """Class decorator: remembers what the class consists of, for ``untouched``."""
    cls.__annotations__   # torch.jit would make it later
    members = dict(vars(cls))
    methods = (name for name, member in members.items() if callable(member) or isinstance(member, (property, staticmethod)))
    _AS_WRITTEN[cls] = vars(cls), members, frozenset(methods) | {"_call_impl", "_compiled_call_impl"}
    return cls


def untouched(module, cls):
    """Whether ``module`` is a ``cls`` as it stands in its file (the class is marked ``as_written``): no subclass, nothing of the
    class replaced or added, none of its methods replaced in the module, no hooks, not compiled. Whoever put such a thing there
    wants the tensors that pass through the module, so it has to be called, with those tensors; so does torch while it compiles."""
    return not _hp._is_compiling() and as_it_stands(module, cls)


def as_it_stands(module, cls):
    """``untouched`` for a caller that knows that torch is not compiling."""
    if cls not in _AS_WRITTEN:   # somebody's own in the place of a class of this package
        return False
    own = module.__dict__
    now, members, methods = _AS_WRITTEN[cls]
    return (type(module) is cls and own.keys().isdisjoint(methods) and now == members
            and _Module.__call__ is _CALL
            and not (own["_forward_hooks"] or own["_forward_pre_hooks"] or own["_backward_hooks"] or own["_backward_pre_hooks"]
                     or _has_any_global_hook()))


def recast(t):
    """Whether autocast would hand the products another type than that of ``t``."""
    return torch.is_autocast_enabled("cuda") and torch.get_autocast_dtype("cuda") is not t.dtype


def _cache_fits(key, value, past):
    """Whether these are 16-bit keys and values on one GPU, of one shape and a size that the kernels can address after ``past``
    cached positions."""
    dtype, shape = key.dtype, key.shape
    if not (key.is_cuda and (dtype is torch.bfloat16 or dtype is torch.float16) and len(shape) == 4 and value.shape == shape
            and value.dtype is dtype and value.device == key.device):
        return False
    sq, b, nkv, hn = shape
    sk, heads = past + sq, b * nkv
    return sq > 0 < heads and hn > 0 and hn % 8 == 0 and heads * hn < 1 << 24 and sk < 1 << 24 and sk * heads < 1 << 31


def _continues(cached, key):
    """Whether cached keys or values, ``[.., past, b, nkv, hn]``, are followed by ``key``."""
    return cached.shape[-3:] == key.shape[1:] and cached.dtype == key.dtype and cached.device == key.device


def cache_supported(key, value, layer_past):
    """Whether a layer can use ``append_to_cache`` for these: what the kernel takes, and nobody differentiates; ``layer_past``
    (None: no cached positions) ``[2, past, b, nkv, hn]``."""
    if layer_past is None:
        return _cache_fits(key, value, 0) and plain(key, value)
    return (isinstance(layer_past, torch.Tensor) and layer_past.dim() == 5 and layer_past.size(0) == 2
            and _cache_fits(key, value, layer_past.size(1)) and _continues(layer_past, key) and plain(key, value, layer_past))


def _past_fits(key, value, past_key, past_value):
    """``cache_supported`` for a direct call, whoever differentiates."""
    return (past_key.dim() == 4 and past_value.shape == past_key.shape and _cache_fits(key, value, past_key.size(0))
            and _continues(past_key, key) and _continues(past_value, key))


def append_to_cache(key, value, layer_past, checked=False):
    """``torch.stack((cat(past keys, key), cat(past values, value)))`` in one launch: ``[2, past + sq, b, nkv, hn]``.
    ``checked``: the caller has asked ``cache_supported`` already."""
    if checked and not _hp._is_compiling():
        present = _hp.native().append_to_cache(key, value, layer_past)
        if present is not NotImplemented:
            return present
    past_k, past_v = (None, None) if layer_past is None else layer_past
    if layer_past is None:
        _refuse_unless(checked or _cache_fits(key, value, 0), "append_to_cache", key, value)
    else:
        _refuse_unless(checked or _past_fits(key, value, past_k, past_v), "append_to_cache", key, value, past_k, past_v)
        past_k, past_v = _readable(past_k), _readable(past_v)
    key, value = _readable(key), _readable(value)
    past = 0 if past_k is None else past_k.size(0)
    sq, b, nkv, hn = key.shape
    present = torch.empty((2, past + sq, b, nkv, hn), dtype=key.dtype, device=key.device)
    with _hp.device_guard(key):
        rc = _hp.lib().nhp_kv_cache_append(
            present.data_ptr(), key.data_ptr(), value.data_ptr(), past_k.data_ptr() if past else None,
            past_v.data_ptr() if past else None, b, nkv, sq, past, hn, _strides3(key), _strides3(value),
            _strides3(past_k) if past else None, _strides3(past_v) if past else None, _hp.dtype_code(key, "append_to_cache"),
            _hp.stream_of(key))
    _hp.check(rc, "append_to_cache")
    return present


def _decode_fits(query, key, value, past):
    """A key for every query, some cached positions, and few enough queries for each key/value head."""
    return (supported(query, key, value) and query.size(0) == key.size(0) and past > 0 and past + key.size(0) >= 4
            and query.size(0) * (query.size(2) // key.size(2)) <= MAX_DECODE_ROWS)


def decode_supported(query, key, value, layer_past):
    """Whether ``decode_attention`` takes these, and nobody differentiates."""
    return (isinstance(layer_past, torch.Tensor) and layer_past.dim() == 5 and layer_past.size(0) == 2
            and _cache_fits(key, value, layer_past.size(1)) and _continues(layer_past, key)
            and _decode_fits(query, key, value, layer_past.size(1)) and plain(query, key, value, layer_past))


def _cached_rows(layer_past):
    """Address and strides of the cached keys and of the values, their number, and what has to live until the launch. Of one
    tensor without making two of it, which takes the host 5 us."""
    if isinstance(layer_past, torch.Tensor):
        pair, past, b, nkv, hn = layer_past.stride()
        if hn == 1 and (pair | past | b | nkv) % 8 == 0 and past < 1 << 24 and layer_past.data_ptr() % 16 == 0:
            n = layer_past.shape
            strides = _I64x3(past if n[1] > 1 else 0, b if n[2] > 1 else 0, nkv if n[3] > 1 else 0)
            keys = layer_past.data_ptr()
            return (keys, strides), (keys + 2 * pair, strides), n[1], layer_past
    keys, values = (_readable(t) for t in layer_past)
    return (keys.data_ptr(), _strides3(keys)), (values.data_ptr(), _strides3(values)), keys.size(0), (keys, values)


def decode_attention(query, key, value, layer_past, mask, scale, fill, merged=False):
    """``masked_attention`` of new positions over the cached ones and themselves, and ``append_to_cache``, in one pass
    over the cache: ``(context, present)``. ``mask`` ``[1 or b, 1, sq, past + sq]``, True = masked."""
    past_k, past_v = layer_past
    fits = (_past_fits(key, value, past_k, past_v) and _decode_fits(query, key, value, past_k.size(0))
            and mask_supported(mask, query.size(1), query.size(0), past_k.size(0) + key.size(0), query.device))
    _refuse_unless(fits, "decode_attention", query, key, value, past_k, past_v, mask)
    return checked_decode_attention(query, key, value, layer_past, mask, scale, fill, merged)


def checked_decode_attention(query, key, value, layer_past, mask, scale, fill, merged):
    """``decode_attention`` for a caller that has asked ``decode_supported`` and ``mask_supported`` already: a step of a small
    model waits for the host, and the checks cost it several microseconds a layer."""
    if not _hp._is_compiling():
        both = _hp.native().decode_attention(query, key, value, layer_past, mask, float(scale), float(fill), merged)
        if both is not NotImplemented:
            return both
    query, key, value = _readable(query), _readable(key), _readable(value)
    (keys, key_strides), (values, value_strides), past, _alive = _cached_rows(layer_past)
    sq, b, np_, hn = query.shape
    nkv = key.size(2)
    if mask.stride(3) != 1:
        mask = mask.contiguous()
    out, out_strides = _new_context(query, merged)
    present = torch.empty((2, past + sq, b, nkv, hn), dtype=key.dtype, device=key.device)
    lib = _hp.lib()
    scratch = lib.nhp_attention_decode_workspace_bytes(b, np_, nkv, sq, past, hn)
    workspace = torch.empty(scratch, dtype=torch.uint8, device=query.device) if scratch else None
    with _hp.device_guard(query):
        rc = lib.nhp_attention_decode(
            out.data_ptr(), present.data_ptr(), query.data_ptr(), key.data_ptr(), value.data_ptr(), keys,
            values, mask.data_ptr(), mask.stride(0) if mask.size(0) > 1 else 0, mask.stride(2), fill,
            None if workspace is None else workspace.data_ptr(), scale, b, np_, nkv, sq, past, hn,
            out_strides, _strides3(query), _strides3(key), _strides3(value), key_strides, value_strides,
            _hp.dtype_code(query, "decode_attention"), _hp.stream_of(query))
    _hp.check(rc, "decode_attention")
    return out, present
