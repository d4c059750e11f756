"""``y = x W^T (+ b)`` for the few rows of a decoding step, on the kernel of csrc/linear_decode.hip.

The reference's Column / RowParallelLinear (megatron/mpu/layers.py) call the library GEMM whatever the number of rows. With
few of them the product is a single read of the weights, and the library's call alone takes the host 25 us (this one 8).

Where the line lies, library -> here on the GPU: 16 rows [4096, 4096] 14.9 -> 11.5 us, [22016, 4096] 51.7 -> 43.5,
[4096, 11008] 38.2 -> 27.6, [2048, 8192] 12.6 -> 13.2, [2560, 10240] 16.9 -> 22.1; one row [2304, 768] 7.2 -> 3.6. 32 rows
[2304, 768] 6.9 -> 4.9, [8192, 2048] 12.9 -> 13.4, [2048, 2048] 11.3 -> 8.3, [1024, 4096] 11.8 -> 14.3, but [4096, 4096]
12.6 -> 15.4, [7680, 2560] 12.0 -> 18.5. Layers up to 2048 features wait for the host in either case."""
import torch
import torch.nn.functional as F

from ..fused_kernels import _hotpath as _hp
from .fused_attention import plain

MAX_ROWS = 16          # of any layer
MAX_ROWS_NARROW = 32   # where one of its sides has at most 2048 features
MAX_FEATURES = 16384


def _few_rows(x, weight, bias):
    n, k = weight.shape
    return (x.numel() <= (MAX_ROWS_NARROW if min(n, k) <= 2048 else MAX_ROWS) * k and x.is_cuda and x.dim() > 0 and x.size(-1) == k and x.numel() > 0
            and x.dtype in (torch.bfloat16, torch.float16) and weight.dtype == x.dtype and weight.device == x.device
            and k % 32 == 0 and k <= MAX_FEATURES and n % 16 == 0 and 0 < n <= 1 << 24 and weight.is_contiguous()
            and x.is_contiguous()
            and (bias is None or (bias.dtype == x.dtype and bias.device == x.device and bias.shape == (n,) and bias.is_contiguous()
                                  and plain(bias)))
            and plain(x, weight) and not torch.is_autocast_enabled("cuda")
            and x.data_ptr() % 16 == 0 and weight.data_ptr() % 16 == 0)


def linear(x, weight, bias=None):
    """``torch.nn.functional.linear``; in inference with few rows of a 16-bit type by one kernel (two with more than 4096
    features)."""
    if weight.dim() != 2 or not _few_rows(x, weight, bias):
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
