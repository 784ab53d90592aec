"""Dense projections for the multi-token paths.

``mm_f32(a, w)`` is ``a @ w.T`` with fp32 output, exact products and fp32 accumulation for
bf16 or fp32 ``a`` against bf16 or fp32 ``w``, without copying the weight:

* bf16 ``a``, bf16 ``w``: one GEMM with fp32 output on the BLAS library;
* fp32 ``a``, bf16 ``w``: ``k3_dense`` (``a`` as the exact sum of three bf16 terms against the
  weight in one launch);
* fp32 ``w``: an fp32 GEMM.

This is the arithmetic of the reference's fp32 router and of MLX's promotion of a bf16
weight against an fp32 activation (``air_llm/models/kimi_k3/moe.py:67-68``).

``dense(a, ws)`` is ``k3_dense`` itself: several bf16 weight matrices against one ``a``.

``mm_ref(a, w)`` keeps the reference's dtype promotion instead: operands of one dtype give
that dtype (a bf16 GEMM returns bf16, as MLX's bf16 matmul does), mixed operands give fp32.
The paths that restate the reference's own unfused definitions use it.
"""
from __future__ import annotations

import ctypes

import torch

from . import _lib
from . import _torch as T


def bf16_terms(a: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Three bf16 tensors whose fp32 sum is exactly ``a`` (fp32) for normal values."""
    t1 = a.to(torch.bfloat16)
    r = a - t1.float()
    t2 = r.to(torch.bfloat16)
    t3 = (r - t2.float()).to(torch.bfloat16)
    return t1, t2, t3


def _mm_bf16_f32(a2: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return torch.mm(a2, w.t(), out_dtype=torch.float32)


# what k3_dense takes: rows of a and of one weight matrix, and their width and pitch
MAX_ROWS, MAX_WIDTH = 1 << 24, 1 << 20


def _rows_ok(w: torch.Tensor) -> bool:
    return (w.is_cuda and w.dtype == torch.bfloat16 and w.dim() == 2 and w.is_contiguous() and w.data_ptr() % 16 == 0
            and w.shape[1] % 8 == 0 and w.shape[1] <= MAX_WIDTH and 0 < w.shape[0] <= MAX_ROWS)


def weights_ok(*ws: torch.Tensor) -> bool:
    """k3_dense takes these weights as they are: bf16 device matrices of whole 16-byte rows."""
    for w in ws:
        if not _rows_ok(w):
            return False
    return not T.tracked(*ws)


def dense_ok(a: torch.Tensor, *ws: torch.Tensor) -> bool:
    """k3_dense takes a against these weights as they are, and no gradient is asked for."""
    if not a.is_cuda or a.dtype not in (torch.float32, torch.bfloat16) or T.tracked(a, *ws):
        return False
    K, dev = a.shape[-1], a.get_device()
    if a.numel() > MAX_ROWS * K:
        return False
    for w in ws:
        if not _rows_ok(w) or w.shape[1] != K or w.get_device() != dev:
            return False
    return True


def dense(a: torch.Tensor, ws, add: torch.Tensor | None = None) -> list[torch.Tensor]:
    """[a [M, K] @ w[N, K]^T in fp32 for w in ws] (k3_dense; a and ws checked by dense_ok), plus
    ``add`` [M, N] fp32 where one weight is given."""
    M, K = a.shape
    if add is not None:
        if len(ws) != 1 or tuple(add.shape) != (M, ws[0].shape[0]) or add.dtype != torch.float32:
            raise ValueError(f"add must be float32 [{M}, N] beside one weight [N, {K}]; got {add.dtype} {tuple(add.shape)}")
        T.require_device(a, add)
        add = T.contiguous_aligned(add)
    if (a.stride(1) != 1 or (a.stride(0) * a.element_size()) % 16 or not K <= a.stride(0) <= MAX_WIDTH
            or a.data_ptr() % 16):
        a = T.contiguous_aligned(a)
    n = len(ws)
    outs = [torch.empty((M, w.shape[0]), dtype=torch.float32, device=a.device) for w in ws]
    N = (ctypes.c_int64 * n)(*(w.shape[0] for w in ws))
    code = T.dtype_code(a.dtype)
    nbytes = int(_lib.lib().k3_dense_workspace_size(M, K, N, n, code))
    # the partial sums are the call's own: calls of several threads on one stream, and a captured
    # graph whose call is followed by a larger one, must not meet in a kept buffer
    buf = torch.empty(nbytes, dtype=torch.uint8, device=a.device) if nbytes else None
    _lib.call("k3_dense", T.ptr(a), code, a.stride(0) if M > 1 else K, (ctypes.c_void_p * n)(*(w.data_ptr() for w in ws)),
              (ctypes.c_void_p * n)(*(o.data_ptr() for o in outs)), N, n, T.ptr(add), M, K, T.ptr(buf), nbytes,
              T.stream(a))
    return outs


def one_launch(M: int, n: int) -> bool:
    """Whether one k3_dense launch takes n bf16 matrices against M bf16 tokens (one matrix-core pass)
    instead of a library GEMM each.

    On the device (weights not yet cached, library / k3_dense us) it is shorter up to 64 tokens (1536 +
    576 + 8192 rows of 7168 at 2 tokens 48.6 / 36.1, at 64 64 / 41; 512 + 512 of 1024 11.2 / 10.5; at worst
    6144 + 6144 of 7168 at 2 tokens 40.2 / 42.0), for three matrices or more (768 + 576 + 2048 of 2048 at 256
    tokens 33.5 / 29.7) and for long rows, whose K it splits over blocks (2048 + 2048 of 7168 at 700 tokens
    82.7 / 66.9).  Two matrices of short rows are shorter on the library beyond 64 tokens, by 14 us
    at most of 559 measured points (512 + 512 of 1024 at 1000 tokens 17.3 / 28.2, 5632 + 5632 of 2048 at 274
    35.0 / 48.8).  But every library call costs the host more than that, and a layer of such sizes
    waits for the host: 162 tokens through a layer with 1024 + 1024 rows of 1792 140.5 us with one
    launch, 166.7 with two library calls.  Beyond 1024 tokens neither leads (1536 + 576 + 8192 of 7168 at 1500
    tokens 236 / 193, at 2048 288 / 343) and the library stays."""
    return n > 1 and M <= 1024


def project(a: torch.Tensor, ws, checked: bool = False) -> list[torch.Tensor]:
    """[a [M, K] @ w[N, K]^T in fp32 for w in ws], all against one activation: fp32 a in one k3_dense
    launch (three library products a matrix were slower at every size measured, 2 to 2048 tokens of
    64 to 12,288 rows); bf16 a where one_launch holds, on the library elsewhere.  checked: weights_ok
    holds for ws, and a is a device tensor of either type that nothing is asked of (tracked)."""
    M, K = a.shape
    if M and (a.dtype == torch.float32 or one_launch(M, len(ws))):
        dev = a.get_device()
        if all(w.shape[1] == K and w.get_device() == dev for w in ws) if checked else dense_ok(a, *ws):
            return dense(a, list(ws))
    return [mm_f32(a, w) for w in ws]


def mm_f32(a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """a [..., K] @ w[N, K]^T -> fp32 [..., N] with exact products and fp32 accumulation."""
    lead = a.shape[:-1]
    a2 = a.reshape(-1, a.shape[-1])
    if w.dtype == torch.float32:
        out = a2.to(torch.float32) @ w.t()
    elif w.dtype == torch.bfloat16:
        if a2.dtype == torch.bfloat16:
            out = _mm_bf16_f32(a2, w)
        elif a2.dtype == torch.float32 and a2.shape[0] > 0 and dense_ok(a2, w):
            out = dense(a2, [w])[0]
        else:
            t1, t2, t3 = bf16_terms(a2.to(torch.float32))
            out = _mm_bf16_f32(t1, w)
            out += _mm_bf16_f32(t2, w)
            out += _mm_bf16_f32(t3, w)
    else:
        raise TypeError(f"weights must be float32 or bfloat16; got {w.dtype}")
    return out.reshape(*lead, w.shape[0])


def mm_ref(a: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """a @ w.T with the reference's (MLX's) dtype promotion: same dtype in, same dtype out;
    bf16 against fp32 gives fp32."""
    if a.dtype == w.dtype:
        return a @ w.t()
    return mm_f32(a, w)
