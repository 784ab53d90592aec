"""Torch tensor plumbing for the C-ABI: device pointers, dtype enums and streams."""
from __future__ import annotations

import torch
from torch.autograd import forward_ad

from . import _lib

_DTYPES = {torch.float32: _lib.K3_F32, torch.bfloat16: _lib.K3_BF16}


def dtype_code(dt: torch.dtype) -> int:
    try:
        return _DTYPES[dt]
    except KeyError:
        raise TypeError(f"unsupported dtype {dt}; k3hip takes float32 or bfloat16") from None


def ptr(t: torch.Tensor | None) -> int:
    """The device address (0 for None), as the ctypes argument types take it."""
    return 0 if t is None else t.data_ptr()


def _stream_handle(device_index: int) -> int:
    return torch.cuda.current_stream(device_index).cuda_stream


# The raw handle of the current stream, without the Stream object that
# torch.cuda.current_stream builds around it (about 1 us per call) where torch offers it.
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", _stream_handle)


def stream(t: torch.Tensor) -> int:
    """The current HIP stream of t's device."""
    return _raw_stream(t.get_device())


def stream_of(device: torch.device) -> int:
    """The current HIP stream of a device (the current device where it has no index)."""
    return _raw_stream(torch.cuda.current_device() if device.index is None else device.index)


def require_device(*ts: torch.Tensor) -> None:
    dev = None
    for t in ts:
        if t is None:
            continue
        if not t.is_cuda:
            raise ValueError(f"k3hip kernels take device tensors; got {t.device}")
        d = t.get_device()
        if dev is None:
            dev, first = d, t
        elif d != dev:
            raise ValueError(f"tensors on different devices: {first.device} vs {t.device}")


def tracked(*ts: torch.Tensor | None) -> bool:
    """A gradient, or a forward-mode tangent, of one of these is asked for: the launches carry
    neither, so such a call stays on the tensor operations that do."""
    if torch.is_grad_enabled():
        for t in ts:
            if t is not None and t.requires_grad:
                return True
    # (unpack_dual takes half a microsecond a tensor: only inside a dual level, or where torch no longer says)
    if getattr(forward_ad, "_current_level", 0) >= 0:
        return any(t is not None and forward_ad.unpack_dual(t).tangent is not None for t in ts)
    return False


def contiguous_aligned(t: torch.Tensor) -> torch.Tensor:
    """Row-contiguous with a 16-byte aligned base (the 128-bit load paths need it);
    the counterpart of ensure_row_contiguous=True (mxfp4_matvec.py:71)."""
    if not t.is_contiguous():
        t = t.contiguous()
    if t.data_ptr() % 16:
        t = t.clone()
    return t
