"""Tensor plumbing shared by the kernel wrappers: dtype codes, device checks,
strides and the HIP stream of the calling thread."""

from __future__ import annotations

import torch
from torch import _C, _ops
from torch.autograd import forward_ad
from torch.utils._device import DeviceContext

from kernels import MLS_BF16, MLS_F16, MLS_F32

_DT = {torch.float32: MLS_F32, torch.float16: MLS_F16, torch.bfloat16: MLS_BF16}


def dt_code(dtype: torch.dtype, what: str) -> int:
    try:
        return _DT[dtype]
    except KeyError:
        raise TypeError(f"{what}: dtype {dtype} not supported (float32, float16, bfloat16)") from None


def require_hip(fn: str, *tensors: torch.Tensor) -> torch.device:
    """All tensors on one HIP device; the kernels have no host implementation."""
    dev = None
    for t in tensors:
        if not isinstance(t, torch.Tensor):
            raise TypeError(f"{fn}: expected tensors, got {type(t).__name__}")
        d = t.device
        if d.type != "cuda":
            raise TypeError(f"{fn}: tensors must be on a HIP device (got {d}); "
                            "the gfx950 kernels have no CPU implementation")
        if dev is None:
            dev = d
        elif d != dev:
            raise ValueError(f"{fn}: tensors on different devices ({dev} and {d})")
    return dev


def rows(t: torch.Tensor) -> torch.Tensor:
    """A 2-D view with unit inner stride (copying only if needed)."""
    if t.dim() != 2:
        raise ValueError(f"expected a 2-D tensor, got shape {tuple(t.shape)}")
    if t.stride(1) != 1 or t.stride(0) < max(1, t.shape[1]):
        t = t.contiguous()
    return t


def ld(t: torch.Tensor) -> int:
    return max(int(t.stride(0)), int(t.shape[1]), 1)


def stream(dev: torch.device) -> int:
    """The calling thread's current stream on dev, a tensor's device (so it has an index). The
    handle itself, 0.2 us a call: making torch.cuda.current_stream's Stream object takes 2.0
    (an eager INT8 layer, fp32, 8 x 512 -> 2048: 18.4 -> 15.9 us)."""
    return torch._C._cuda_getCurrentRawStream(dev.index)


def scale_vector(scale: torch.Tensor) -> tuple[torch.Tensor, int]:
    """Per-row scales as fp32 or fp16 (kept as stored); other dtypes become fp32,
    which is what the reference does for every scale (dequant_matmul.py:147)."""
    if scale.dtype not in (torch.float32, torch.float16):
        scale = scale.to(torch.float32)
    return scale, _DT[scale.dtype]


def _watched() -> bool:
    """Whether something records, rewrites or intercepts this thread's torch calls: a trace, a function
    transform, forward mode, a dispatch mode, or a function mode other than torch's default device."""
    return (_C._is_tracing() or _C._len_torch_dispatch_stack() > 0 or forward_ad._current_level >= 0
            or _C._functorch.peek_interpreter_stack() is not None or _ops._len_torch_dispatch_stack_pre_dispatch() > 0
            or torch.compiler.is_compiling()
            or _C._len_torch_function_stack() > 0
            and not all(isinstance(m, DeviceContext) for m in torch.overrides._get_current_function_mode_stack()))


def plain(t: torch.Tensor) -> bool:
    """An ordinary device tensor whose values are as stored, from which no gradient is asked for, in
    code that nothing watches: one whose memory a kernel may read in place of torch ops."""
    return (type(t) is torch.Tensor and t.device.type == "cuda" and not (t.requires_grad and torch.is_grad_enabled())
            and not t.is_neg() and not _watched())
