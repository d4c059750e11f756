"""``y = x W^T (+ b)`` for the few rows of a decoding step, on the kernel of csrc/linear_decode.hip.

The reference's Column / RowParallelLinear (megatron/mpu/layers.py) call the library GEMM whatever the number of rows. With
few of them the product is a single read of the weights, and the library's call alone takes the host 25 us (this one 4).

Where the line lies. On the GPU, weights not in any cache, us here / library:
    rows           1            4            16           24           32
    [2304, 768]    3.8 / 6.3    3.9 / 6.4    3.9 / 6.4    4.7 / 9.3    4.8 / 9.2
    [2048, 2048]   5.1 / 10.9   5.1 / 11.0   6.0 / 11.0   7.4 / 11.0   8.3 / 11.3
    [1024, 4096]   6.4 / 14.4   6.8 / 14.5   8.6 / 14.4   11.5 / 14.2  12.9 / 11.9
    [4096, 4096]   9.8 / 15.8   9.9 / 15.9   11.7 / 15.9  14.6 / 14.1  15.7 / 14.0
    [12288, 4096]  20.4 / 27.5  20.8 / 28.9  22.6 / 28.7  25.1 / 24.6  26.9 / 24.7
    [22016, 4096]  34.0 / 51.8  34.8 / 52.0  37.6 / 52.5  40.4 / 44.8  42.3 / 45.2
    [6144, 4096]   13.4 / 15.8  13.5 / 16.1  15.5 / 15.9  17.9 / 16.3  19.4 / 17.0
    [7680, 2560]   10.4 / 12.4  10.5 / 12.3  11.6 / 12.7  13.5 / 13.2  15.0 / 13.3
    [5120, 5120]   14.5 / 14.8  14.8 / 15.2  15.5 / 17.9  17.3 / 20.5  17.8 / 20.9
    [2560, 10240]  14.6 / 19.7  15.0 / 19.5  16.2 / 20.1  18.3 / 22.5  19.6 / 22.6
    [4096, 11008]  20.9 / 38.5  21.2 / 38.9  22.8 / 38.8  25.0 / 32.5  26.2 / 31.9
    [4096, 14336]  24.9 / 26.8  25.5 / 26.7  27.3 / 27.3  29.6 / 32.0  31.0 / 34.0
Up to 16 rows the kernel is ahead everywhere, up to 28 where a side has at most 2048 features and up to 32 where four workgroups
share the contraction (more than 4096 features; [8192, 8192] 33.1 / 31.3); in between the library catches up. At 29 to 32 rows with a
side of at most 2048 features and more than 2048 in the library is up to 14 % ahead on the GPU ([2048, 4096] 13.8 / 12.1, [1536, 3072]
10.7 / 10.1); these are taken for the 20 us that its call costs the host.

More rows than that (a short prompt, many sequences) go to csrc/linear_tiles.hip where it is ahead; its table and rule stand there."""
from typing import Optional

import torch
import torch.nn.functional as F

from ..fused_kernels import _hotpath as _hp
from .fused_attention import plain

MAX_ROWS = 16          # of any layer
MAX_ROWS_NARROW = 32   # where one of its sides has at most 2048 features, or more than 4096 come in
MAX_FEATURES = 16384
BIAS_GELU = 16   # NHP_LINEAR_BIAS_GELU; gates go by their codes


def _are_few(x, weight):
    n, k = weight.shape
    return x.numel() <= (MAX_ROWS_NARROW if min(n, k) <= 2048 or k > 4096 else MAX_ROWS) * k


def _few_rows(x, weight, bias):
    return _are_few(x, weight) and _rows_ready(x, weight, bias)


def _some_rows(x, weight, bias):
    """More rows that csrc/linear_tiles.hip takes (its rule stands there)."""
    n, k = weight.shape
    return (not _are_few(x, weight) and _rows_ready(x, weight, bias) and _hp.lib().nhp_linear_tiles_pay(x.numel() // k, n, k)
            and (bias is None or bias.data_ptr() % 16 == 0))


def _rows_ready(x, weight, bias):
    n, k = weight.shape
    dtype = x.dtype
    return (x.is_cuda and x.dim() > 0 and x.size(-1) == k and x.numel() > 0
            and (dtype is torch.bfloat16 or dtype is torch.float16) and weight.dtype is dtype and weight.device == x.device
            and k % 32 == 0 and k <= MAX_FEATURES and n % 16 == 0 and 0 < n <= 1 << 24 and weight.is_contiguous()
            and x.is_contiguous()
            and (bias is None or (bias.dtype is dtype and bias.device == x.device and bias.shape == (n,) and bias.is_contiguous()))
            and (plain(x, weight) if bias is None else plain(x, weight, bias)) and not torch.is_autocast_enabled("cuda")
            and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0)


def linear(x, weight, bias: Optional[torch.Tensor] = None):
    """``torch.nn.functional.linear``; in inference with up to some hundred rows of a 16-bit type by one kernel (two with few rows
    and more than 4096 features). Scripted, compiled, exported or traced over proxies it is torch's: the sizes below would become conditions."""
    if torch.jit.is_scripting():
        return F.linear(x, weight, bias)
    else:
        return _linear(x, weight, bias)


@torch.jit.unused
def _linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
    if isinstance(x, torch.Tensor) and x.is_cuda and not _hp._is_compiling():
        y = _hp.native().linear(x, weight, bias, MAX_ROWS, MAX_ROWS_NARROW)
        if y is not NotImplemented:
            return y
    if (_hp._is_compiling() or _hp._tracing_state() is not None or not isinstance(x, torch.Tensor) or not isinstance(weight, torch.Tensor)
            or weight.dim() != 2 or not (_few_rows(x, weight, bias) or _some_rows(x, weight, bias))):
        return F.linear(x, weight, bias)
    n, k = weight.shape
    rows = x.numel() // k
    y = torch.empty(x.shape[:-1] + (n,), dtype=x.dtype, device=x.device)
    lib = _hp.lib()
    if not _are_few(x, weight):
        with _hp.device_guard(x):
            rc = lib.nhp_linear_tiles(y.data_ptr(), x.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(), rows, n,
                                      k, _hp.dtype_code(x, "linear"), _hp.stream_of(x))
        _hp.check(rc, "linear")
        return y
    scratch = lib.nhp_linear_decode_workspace_bytes(rows, n, k)
    workspace = torch.empty(scratch, dtype=torch.uint8, device=x.device) if scratch else None
    with _hp.device_guard(x):
        rc = lib.nhp_linear_decode(y.data_ptr(), x.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(),
                                   None if workspace is None else workspace.data_ptr(), rows, n, k, _hp.dtype_code(x, "linear"),
                                   _hp.stream_of(x))
    _hp.check(rc, "linear")
    return y
