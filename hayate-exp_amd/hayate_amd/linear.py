"""The products of a tick's rows with the model's weights (csrc/skinny.hip for
a decode tick's few rows, csrc/tiles.hip for a prompt's many), and the rule that
says when a module's forward may take them in place of its submodules' own calls.

For few rows ``norm_linear`` is RMSNorm then a projection (optionally the gated
pair with silu) and ``linear_add`` a projection plus the residual; for many,
``row_norm`` is the norm and ``tile_linear`` the gated pair or the projection
plus the residual. They compute what the torch modules do with
fp32 sums and fewer bf16 roundings, and know nothing of autograd, hooks or
tracing: ``takes`` and ``plain`` hold every condition under which a caller must
leave the modules in charge.
"""

from __future__ import annotations

import sys
from typing import Optional

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad as _forward_ad
from torch.nn.modules import module as _module
from torch.utils._device import DeviceContext as _DeviceContext

from . import _native

MAX_ROWS = 32
_MAX_STRIDE = 1 << 22
_BF16 = torch.bfloat16
_C, _peek_functorch = torch._C, torch._C._functorch.peek_interpreter_stack
_Parameter, _Module, _Linear, _RMSNorm = nn.Parameter, nn.Module, nn.Linear, nn.RMSNorm


def _as_shipped(f, home) -> object:
    """`f` if it is the function that module `home` defines, else an object that
    nothing compares equal to: patched before this import, it stays in charge."""
    code = getattr(f, "__code__", None)
    return f if code is not None and code.co_filename == home.__file__ else object()


# What calling a module and the functions in it runs, unless somebody has put
# something else in their place.
_CALL = _as_shipped(nn.Module.__call__, _module)
_LINEAR = _as_shipped(nn.Linear.forward, sys.modules["torch.nn.modules.linear"])
_NORM = _as_shipped(nn.RMSNorm.forward, sys.modules["torch.nn.modules.normalization"])
_F_LINEAR = _C._nn.linear
_RMS_NORM, _SILU = _as_shipped(F.rms_norm, F), _as_shipped(F.silu, F)


def unwatched() -> bool:
    """True when nothing watches the operators a call runs: tracing, dispatch or
    function modes, functorch, forward-mode gradients. A default device is held
    in a function mode too, but watches nothing: it names the device of factory
    calls that leave theirs open, which the callers of this do not."""
    n = _C._len_torch_function_stack()
    return (_C._len_torch_dispatch_stack() == 0
            and (n == 0 or all(type(_C._get_function_stack_at(i)) is _DeviceContext
                               for i in range(n)))
            and _C._get_tracing_state() is None and not torch.compiler.is_compiling()
            and _forward_ad._current_level < 0
            and _peek_functorch() is None)


def takes(x: torch.Tensor) -> bool:
    """True when `x` (..., d) is a plain bf16 tensor on the current HIP device and
    nothing watches the operators run on it, nor gradients or autocast change
    them."""
    return (type(x) is torch.Tensor and x.dtype is torch.bfloat16 and x.is_cuda
            and x.numel() > 0
            and not torch.is_grad_enabled() and not torch.is_autocast_enabled()
            and unwatched() and x.device.index == torch.cuda.current_device())


def few_rows(x: torch.Tensor) -> bool:
    """`takes`, and at most MAX_ROWS rows."""
    return takes(x) and x.numel() <= MAX_ROWS * x.shape[-1]


def _unpatched() -> bool:
    """True when calling the modules of a block runs torch's own code."""
    return (_Linear.__call__ is _CALL and _RMSNorm.__call__ is _CALL and _Module.__call__ is _CALL
            and _Linear.forward is _LINEAR and _RMSNorm.forward is _NORM
            and F.linear is _F_LINEAR and F.rms_norm is _RMS_NORM and F.silu is _SILU)


def _bare(m: nn.Module) -> bool:
    """No hooks and no forward of its own, compiled or not."""
    d = m.__dict__
    return not (d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"]
                or d["_backward_pre_hooks"] or "forward" in d or "_compiled_call_impl" in d)


def _plain_weight(w, device_index: int, dim: int) -> bool:
    if (type(w) is not _Parameter or w.dtype is not _BF16 or w.data_ptr() & 15
            or w.get_device() != device_index):
        return False
    st = w.stride()
    if dim == 1:
        return st == (1,)
    return len(st) == 2 and st[1] == 1 and st[0] & 7 == 0 and st[0] < _MAX_STRIDE


def plain(x: torch.Tensor, modules=(), norms=(), linears=()) -> bool:
    """True when calling `modules`, `norms` (over x's last dimension) and
    `linears` would do nothing but their own arithmetic on weights that the
    kernels can read."""
    if _module._has_any_global_hook() or not _unpatched():
        return False
    index, shape = x.get_device(), (x.shape[-1],)
    for m in modules:
        if not _bare(m):
            return False
    for m in norms:
        if not (type(m) is _RMSNorm and _bare(m) and m.normalized_shape == shape
                and _plain_weight(m._parameters.get("weight"), index, 1)):
            return False
    for m in linears:
        if type(m) is not _Linear or not _bare(m):
            return False
        p = m.__dict__["_parameters"]
        if p.get("bias") is not None or not _plain_weight(p.get("weight"), index, 2):
            return False
    return True


def norm_fits(k: int, rows: int) -> bool:
    """Sizes hy_norm_linear takes."""
    return k % 64 == 0 and 512 <= k <= 4096 and rows <= (MAX_ROWS if k <= 3072 else 16)


def add_fits(k: int, rows: int) -> bool:
    """Sizes hy_linear_add takes."""
    return k % 128 == 0 and k > 0 and rows <= MAX_ROWS


def tiles_fit(d: int, heads: int, mid: int, rows: int) -> bool:
    """Sizes hy_row_norm and hy_linear_tiles take for a block of d inputs, `heads`
    values of attention and `mid` of the MLP (x's rows are at most _MAX_STRIDE
    apart, which rows_of sees to)."""
    n = d if d > mid else mid
    return ((d | heads | mid) % 64 == 0 and 0 < d <= 4096 and 0 < heads < _MAX_STRIDE
            and 0 < mid < _MAX_STRIDE and (rows // 64 + 1) * (n // 48 + 1) < 1 << 23)


def tiles_add_pays(k: int, n: int, rows: int) -> bool:
    """Whether hy_linear_tiles with a residual keeps up with the library's product
    and addition. Its tiles and their split of k are for outputs that do not fill
    the chip; on many the library's kernels are ahead. Measured on MI355X over n =
    1024 .. 4096 and k = n .. 4 n (time over the library's, by millions of outputs):
    below 4 0.75-1.1, mean 0.95; 4 to 5.5 0.91-1.15, mean 1.03; 6 to 9 1.05; 13 to
    16 up to 1.33 (9728 -> 2560, 512 rows 35 / 47 us, 2064 109 / 111, 6000 283 /
    215). With a very long k the library falls behind for longer (25600 -> 5120:
    1700 rows 0.63, 2064 1.31)."""
    return rows * n <= (11 << 19 if k <= 16_384 else 1 << 23)


def rows_of(x: torch.Tensor) -> torch.Tensor:
    """x (..., d) as (rows, d) with rows the kernels can read."""
    x = x.reshape(-1, x.shape[-1])
    row, one = x.stride()
    if one != 1 or row & 7 or row >= _MAX_STRIDE or x.data_ptr() & 15:
        x = x.contiguous()
        if x.data_ptr() & 15:
            x = x.clone()
    return x


def norm_linear(x: torch.Tensor, norm_weight: Optional[torch.Tensor], eps: float,
                weight: torch.Tensor, up_weight: Optional[torch.Tensor] = None) -> torch.Tensor:
    """norm(x) W^T, or silu(norm(x) W^T) * (norm(x) U^T); x is (rows, k)."""
    m, k = x.shape
    n = weight.shape[0]
    y = x.new_empty((m, n))
    rc = _native.lib().hy_norm_linear(
        x.data_ptr(), x.stride(0), m, k, None if norm_weight is None else norm_weight.data_ptr(),
        eps, weight.data_ptr(), None if up_weight is None else up_weight.data_ptr(),
        weight.stride(0), n, y.data_ptr(), n, _native.stream_of(x.get_device()))
    if rc:
        _native.check(rc, "hy_norm_linear")
    return y


def linear_add(x: torch.Tensor, weight: torch.Tensor,
               residual: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x W^T + residual; x is (rows, k)."""
    m, k = x.shape
    n = weight.shape[0]
    y = x.new_empty((m, n))
    rc = _native.lib().hy_linear_add(
        x.data_ptr(), x.stride(0), m, k, weight.data_ptr(), weight.stride(0), n,
        None if residual is None else residual.data_ptr(),
        0 if residual is None else residual.stride(0), y.data_ptr(), n,
        _native.stream_of(x.get_device()))
    if rc:
        _native.check(rc, "hy_linear_add")
    return y


def row_norm(x: torch.Tensor, norm_weight: torch.Tensor, eps: float) -> torch.Tensor:
    """RMSNorm of x (rows, k)."""
    m, k = x.shape
    y = x.new_empty((m, k))
    rc = _native.lib().hy_row_norm(x.data_ptr(), x.stride(0), m, k, norm_weight.data_ptr(), eps,
                                   y.data_ptr(), _native.stream_of(x.get_device()))
    if rc:
        _native.check(rc, "hy_row_norm")
    return y


def tile_linear(x: torch.Tensor, weight: torch.Tensor, up_weight: Optional[torch.Tensor] = None,
                residual: Optional[torch.Tensor] = None) -> torch.Tensor:
    """x W^T + residual, or silu(x W^T) * (x U^T); x is (rows, k), any rows."""
    m, k = x.shape
    n = weight.shape[0]
    lib = _native.lib()
    y = x.new_empty((m, n))
    size = lib.hy_linear_tiles_workspace_bytes(m, n, k, up_weight is not None)
    work = torch.empty(size, dtype=torch.uint8, device=x.device) if size else None
    rc = lib.hy_linear_tiles(
        x.data_ptr(), x.stride(0), m, k, weight.data_ptr(),
        None if up_weight is None else up_weight.data_ptr(), weight.stride(0), n,
        None if residual is None else residual.data_ptr(),
        0 if residual is None else residual.stride(0), y.data_ptr(), n,
        None if work is None else work.data_ptr(), size,
        _native.stream_of(x.get_device()))
    if rc:
        _native.check(rc, "hy_linear_tiles")
    return y
