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
    return not T.tracked(*ws) and all(map(_rows_ok, ws))


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


def one_launch(M: int, K: int, rows: list[int]) -> bool:
    """Whether one k3_dense launch takes several bf16 matrices against M bf16 tokens (one matrix-core
    pass) sooner than a library GEMM each.  Measured at 559 points, weights not yet cached (M 2..1100, K
    1024..7168, 2 to 4 matrices of 512 to 12,288 rows), it picks the sooner one within 11%
    (library / k3_dense us):

    * up to 64 tokens it does throughout: 1536 + 576 + 8192 rows of 7168 at 2 tokens 48.6 / 36.1, 512 + 512 of
      1024 11.2 / 10.5; at worst 6144 + 6144 of 7168 at 2 tokens 40.2 / 42.0;
    * to 1024 tokens for three matrices or more, whose launches add up (768 + 576 + 2048 of 2048 at 256 tokens
      33.5 / 29.7), and for long rows, whose K it splits over blocks (2048 + 2048 of 7168 at 700 tokens 82.7 /
      66.9); two matrices of short rows are shorter on the library (2048 + 2048 of 2048 at 256 tokens 23.5 /
      29.2, 5632 + 5632 of 2048 35.0 / 48.8);
    * between, for wide matrices to 256 tokens (4096 + 4096 of 4096 at 192 tokens 66.4 / 43.0; at 384 51.4 /
      55.4) and any but the smallest to 128 (3200 + 3200 of 2560 at 102 tokens 29.2 / 24.7; 768 + 576 of 2048
      at 128 16.3 / 18.4);
    * beyond 1024 tokens neither leads (1536 + 576 + 8192 of 7168 at 1500 tokens 236 / 193, at 2048 288 / 343)."""
    if len(rows) < 2 or M > 1024:
        return False
    widest = max(rows)
    return (M <= 64 or len(rows) > 2 or K >= 4800 or (M <= 256 and 3000 <= K <= 1.25 * widest)
            or (M <= 128 and sum(rows) * K >= 4_000_000 and widest <= 2 * K))


def project(a: torch.Tensor, ws) -> list[torch.Tensor]:
    """[a [M, K] @ w[N, K]^T in fp32 for w in ws], all against one activation: fp32 a in one k3_dense
    launch (three library products a matrix were slower at every size measured, 2 to 2048 tokens of
    64 to 12,288 rows); bf16 a where one_launch holds, on the library elsewhere."""
    M = a.shape[0]
    if M and dense_ok(a, *ws) and (a.dtype == torch.float32 or one_launch(M, a.shape[1], [w.shape[0] for w in ws])):
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
