"""``y = x W^T (+ b)`` for the few rows of a decoding step, on the kernel of csrc/linear_decode.hip.

The reference's Column / RowParallelLinear (megatron/mpu/layers.py) call the library GEMM whatever the number of rows. With
few of them the product is a single read of the weights, and the library's call alone takes the host 25 us (this one 8).

Where the line lies. On the GPU, weights not in any cache, us here / library:
    rows           1            4            16            32
    [2304, 768]    3.7 / 8.6    3.8 / 6.7    4.1 / 6.7     5.0 / 9.5
    [2048, 2048]   5.1 / 13.0   5.5 / 11.3   6.4 / 11.3    8.3 / 11.5
    [1024, 4096]   7.3 / 16.5   7.9 / 14.7   10.0 / 14.7   13.7 / 12.1
    [4096, 4096]   9.7 / 17.6   9.7 / 15.8   11.8 / 15.7   15.4 / 13.3
    [22016, 4096]  39.5 / 51.5  39.7 / 50.0  40.9 / 50.8   45.3 / 41.5
    [4096, 11008]  25.4 / 40.1  24.4 / 37.6  26.2 / 37.6   29.1 / 29.8
    [6144, 4096]   14.4 / 16.3  14.9 / 14.5  16.9 / 14.4   20.8 / 15.3
    [5120, 5120]   14.8 / 15.6  15.1 / 14.0  16.0 / 15.4   18.3 / 18.2
    [4096, 14336]  31.2 / 28.2  30.1 / 25.2  32.1 / 25.8   35.6 / 30.9
    [7680, 2560]   12.8 / 13.3  13.1 / 11.4  14.4 / 11.5   16.9 / 12.1
    [2560, 10240]  19.4 / 21.5  18.9 / 16.8  20.6 / 17.2   23.3 / 21.5
Where a side has at most 2048 features the kernel is ahead up to about 24 rows. Larger ones are mixed: with 2560 features a
wave has five of its eight steps to do and the tiles do not divide among the workgroups (160 for 64, 480 for 256). They are
taken all the same up to 16 rows, because it is the host that a step waits for until its cache is long: a layer of 2560
features called step by step takes 222 us here and 272 to 282 with those products in the library, with 1 to 8 sequences of up
to 2000 positions, and 16 of 200. Where the GPU is what is waited for the library is ahead there: 16 sequences of 2000 positions
336 / 320 us, and in a captured graph 71 / 76 us with one sequence, 90 / 91 with four, 195 / 176 with eight of 2000, 336 / 314
with 16. With 4096 features, 8 heads of keys: 247 / 274 us step by step, 178 / 175 in a graph (16 of 2000)."""
from typing import Optional

import torch
import torch.nn.functional as F

from ..fused_kernels import _hotpath as _hp
from .fused_attention import plain

MAX_ROWS = 16          # of any layer
MAX_ROWS_NARROW = 32   # where one of its sides has at most 2048 features
MAX_FEATURES = 16384


def _few_rows(x, weight, bias):
    n, k = weight.shape
    dtype = x.dtype
    return (x.numel() <= (MAX_ROWS_NARROW if min(n, k) <= 2048 else MAX_ROWS) * k and x.is_cuda and x.dim() > 0 and x.size(-1) == k and x.numel() > 0
            and (dtype is torch.bfloat16 or dtype is torch.float16) and weight.dtype is dtype and weight.device == x.device
            and k % 32 == 0 and k <= MAX_FEATURES and n % 16 == 0 and 0 < n <= 1 << 24 and weight.is_contiguous()
            and x.is_contiguous()
            and (bias is None or (bias.dtype is dtype and bias.device == x.device and bias.shape == (n,) and bias.is_contiguous()))
            and (plain(x, weight) if bias is None else plain(x, weight, bias)) and not torch.is_autocast_enabled("cuda")
            and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0)


def linear(x, weight, bias: Optional[torch.Tensor] = None):
    """``torch.nn.functional.linear``; in inference with few rows of a 16-bit type by one kernel (two with more than 4096
    features). Scripted, compiled, exported or traced over proxies it is torch's: the sizes below would become conditions."""
    if torch.jit.is_scripting():
        return F.linear(x, weight, bias)
    else:
        return _linear(x, weight, bias)


@torch.jit.unused
def _linear(x: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor]) -> torch.Tensor:
    if not _hp._is_compiling():
        y = _hp.native().linear(x, weight, bias, MAX_ROWS, MAX_ROWS_NARROW)
        if y is not NotImplemented:
            return y
    if (_hp._is_compiling() or _hp._tracing_state() is not None or not isinstance(x, torch.Tensor) or not isinstance(weight, torch.Tensor)
            or weight.dim() != 2 or not _few_rows(x, weight, bias)):
        return F.linear(x, weight, bias)
    n, k = weight.shape
    rows = x.numel() // k
    y = torch.empty(x.shape[:-1] + (n,), dtype=x.dtype, device=x.device)
    lib = _hp.lib()
    scratch = lib.nhp_linear_decode_workspace_bytes(rows, n, k)
    workspace = torch.empty(scratch, dtype=torch.uint8, device=x.device) if scratch else None
    with _hp.device_guard(x):
        rc = lib.nhp_linear_decode(y.data_ptr(), x.data_ptr(), weight.data_ptr(), None if bias is None else bias.data_ptr(),
                                   None if workspace is None else workspace.data_ptr(), rows, n, k, _hp.dtype_code(x, "linear"),
                                   _hp.stream_of(x))
    _hp.check(rc, "linear")
    return y
