"""Kimi Delta Attention on MI355X -- the counterpart of ``KDAAttention``
(air_llm/models/kimi_k3/attention_kda.py:32-115).

``KDAAttention(cfg, w)`` keeps the reference constructor, weight names and
``__call__(x, state=None, conv=None) -> (out, state, (cq, ck, cv))``.  One token of one
sequence is one ``k3_kda_step_decode`` (projections, short convolutions, norms, gate,
recurrence, gated RMSNorm, o_proj in four launches); more take ``prefill``, which reads every
weight once for all tokens: the projections (``_blas.project``), ``k3_kda_prefill_inputs``,
one ``k3_kda_recurrent`` launch and ``k3_kda_gated_norm``.  For inference: no gradient passes
through the recurrence, and the output carries none.  The recurrent state is fp32
[B, H, 128, 128], updated in place; the convolution states come back as fp32 [B, k-1, C].

``kda_recurrent(q, k, v, g, beta, scale, state)`` takes the reference's tensors
(q, k [B, T, H, K]; v [B, T, HV, V]; g [B, T, HV, K] log decay; beta [B, T, HV]; state
[B, HV, K, V] or None) and returns ``(o [B, T, HV, V] fp32, state [B, HV, K, V] fp32)``.
All tokens are one launch of ``k3_kda_recurrent`` over all B * HV heads, the state kept in
registers between tokens and updated in place once (the reference allocates a new state
per step).  A state passed in is
used as the output state when it is a contiguous fp32 device tensor, else copied once.
"""
from __future__ import annotations

import torch

from . import _blas, _lib, _workspace
from . import _torch as T


def kda_recurrent(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, g: torch.Tensor, beta: torch.Tensor,
                  scale: float | None = None, state: torch.Tensor | None = None):
    T.require_device(q, k, v, g, beta, state)
    if q.dim() != 4 or k.shape != q.shape or v.dim() != 4 or g.dim() != 4 or beta.dim() != 3:
        raise ValueError("q, k [B, T, H, K], v [B, T, HV, V], g [B, T, HV, K], beta [B, T, HV] expected")
    B, Tn, H, K = q.shape
    HV, V = v.shape[2], v.shape[3]
    if tuple(v.shape[:2]) != (B, Tn) or tuple(g.shape) != (B, Tn, HV, K) or tuple(beta.shape) != (B, Tn, HV):
        raise ValueError(f"shape mismatch: q {tuple(q.shape)}, v {tuple(v.shape)}, g {tuple(g.shape)}, "
                         f"beta {tuple(beta.shape)}")
    if HV % H:
        raise ValueError(f"value heads {HV} must be a multiple of q/k heads {H}")
    if scale is None:
        scale = K ** -0.5
    dt = torch.bfloat16 if all(t.dtype == torch.bfloat16 for t in (q, k, v, g, beta)) else torch.float32
    # time-major, so each step's [B, heads, dim] slice is contiguous
    q, k, v, g, beta = (t.to(dt).transpose(0, 1).contiguous() for t in (q, k, v, g, beta))
    S = _state(state, (B, HV, K, V), q.device)
    return _recurrent(q, k, v, g, beta, float(scale), S).transpose(0, 1), S


def _state(state: torch.Tensor | None, shape: tuple, device) -> torch.Tensor:
    """The state to update in place: the given one where the kernels can, else a copy, or zeros."""
    if state is None:
        return torch.zeros(shape, dtype=torch.float32, device=device)
    if tuple(state.shape) != shape:
        raise ValueError(f"state must be {list(shape)}; got {tuple(state.shape)}")
    if state.dtype == torch.float32 and state.is_contiguous() and state.data_ptr() % 16 == 0:
        return state
    return state.to(torch.float32).contiguous().clone()


def _recurrent(q, k, v, g, beta, scale: float, S: torch.Tensor) -> torch.Tensor:
    """All tokens of contiguous time-major q, k [T, B, H, K], v [T, B, HV, V], g [T, B, HV, K], beta
    [T, B, HV] on the state S in one launch -> o [T, B, HV, V] fp32."""
    Tn, B, H, K = q.shape
    HV, V = v.shape[2], v.shape[3]
    o = torch.empty((Tn, B, HV, V), dtype=torch.float32, device=q.device)
    # B sequences are B * HV independent heads: q/k head b * H + h serves value heads
    # (b * HV + h * G) .. + G, the same grouping as within one sequence; all tokens in one
    # launch, the state kept in registers between them
    _lib.call("k3_kda_recurrent", T.ptr(q), T.ptr(k), T.ptr(v), T.ptr(g), T.ptr(beta), T.dtype_code(q.dtype), T.ptr(S),
              T.ptr(o), _lib.K3_F32, Tn, B * H, B * HV, K, V, scale, T.stream(q))
    return o


class KDAAttention:
    """Drop-in for KDAAttention (attention_kda.py:32-115) on bf16 projection weights."""

    KEYS = ("q_proj.weight", "k_proj.weight", "v_proj.weight", "g_proj.weight",
            "o_proj.weight", "q_conv1d.weight", "k_conv1d.weight", "v_conv1d.weight",
            "f_a_proj.weight", "f_b_proj.weight", "b_proj.weight", "o_norm.weight",
            "A_log", "dt_bias")

    def __init__(self, cfg, w: dict):
        self.cfg = cfg
        H, D, K = cfg.kda_num_heads, cfg.kda_head_dim, cfg.kda_conv_size
        self.H, self.D, self.K = H, D, K
        bf = lambda n: T.contiguous_aligned(w[n].to(torch.bfloat16))  # noqa: E731
        f32 = lambda n: T.contiguous_aligned(w[n].to(torch.float32))  # noqa: E731
        self.q_w, self.k_w, self.v_w = bf("q_proj.weight"), bf("k_proj.weight"), bf("v_proj.weight")
        self.g_w, self.o_w = bf("g_proj.weight"), bf("o_proj.weight")
        self.fa, self.fb, self.b_w = bf("f_a_proj.weight"), bf("f_b_proj.weight"), bf("b_proj.weight")
        self.qc, self.kc, self.vc = (f32(n).reshape(H * D, K) for n in ("q_conv1d.weight", "k_conv1d.weight",
                                                                         "v_conv1d.weight"))
        self.o_norm_w, self.dt_bias = f32("o_norm.weight"), f32("dt_bias").reshape(-1)
        A = f32("A_log").reshape(-1)
        if A.shape[0] != D or (A.shape[0] > H and float(A[H:].abs().max()) != 0.0):
            raise ValueError("A_log must be [head_dim] with zeros past num_heads (attention_kda.py:50-54)")
        self.A_log = A

    def decode_step(self, x1, state, conv_in, conv_out, out) -> None:
        """One token of one sequence: x1 [hidden], state [H, D, D] fp32 (in place),
        conv_in / conv_out [3, k-1, H*D] fp32, out [hidden] fp32."""
        c = self.cfg
        nbytes = _lib.size("k3_kda_step_workspace_size", self.H)
        ws = _workspace.get(x1.device, nbytes, "kda_step")
        _lib.call("k3_kda_step_decode", T.ptr(x1), T.dtype_code(x1.dtype), T.ptr(self.q_w), T.ptr(self.k_w),
                  T.ptr(self.v_w), T.ptr(self.g_w), T.ptr(self.o_w), T.ptr(self.fa), T.ptr(self.fb), T.ptr(self.b_w),
                  T.ptr(self.qc), T.ptr(self.kc), T.ptr(self.vc), T.ptr(conv_in), T.ptr(conv_out),
                  T.ptr(self.o_norm_w), T.ptr(self.A_log), T.ptr(self.dt_bias), T.ptr(state), T.ptr(out),
                  _lib.K3_F32, x1.shape[-1], self.H, self.D, self.K, float(c.kda_gate_lower_bound),
                  float(c.rms_norm_eps), T.ptr(ws), ws.numel(), T.stream(x1))

    def _check_widths(self) -> None:
        """The launches of prefill read these weights at the layer's widths, whatever their shapes."""
        H, D = self.H, self.D
        P = H * D
        if (self.q_w.shape[0] == self.k_w.shape[0] == self.v_w.shape[0] == self.g_w.shape[0] == self.fb.shape[0] == P
                and self.b_w.shape[0] == H and self.dt_bias.numel() == P and self.o_norm_w.numel() == D
                and self.A_log.numel() >= H):
            return
        raise ValueError(f"{H} heads of {D} do not match " + ", ".join(f"{n} {tuple(w.shape)}" for n, w in (
            ("q_proj", self.q_w), ("k_proj", self.k_w), ("v_proj", self.v_w), ("g_proj", self.g_w), ("f_b_proj", self.fb),
            ("b_proj", self.b_w), ("dt_bias", self.dt_bias), ("o_norm", self.o_norm_w), ("A_log", self.A_log))))

    def prefill(self, x: torch.Tensor, state: torch.Tensor | None = None, conv: tuple | None = None):
        """Many tokens (attention_kda.py:94-115): the projections of all tokens (each weight
        read once), the convolutions, norms and gates in one launch, the recurrence over every
        token in one, the gated RMSNorm, and o_proj."""
        c = self.cfg
        B, Tn, hid = x.shape
        H, D, K = self.H, self.D, self.K
        P = H * D
        self._check_widths()
        dev = x.device
        xf = x.reshape(B * Tn, hid)
        if xf.dtype not in (torch.float32, torch.bfloat16):
            xf = xf.to(torch.float32)
        xf = xf.detach()
        mats = [self.q_w, self.k_w, self.v_w, self.g_w, self.fa, self.b_w]
        if B * Tn <= 32:
            yq, yk, yv, og, fa, br = _blas.project(xf, mats)
        else:
            # exp(A_log) multiplies the rounding of the gates' matrices: they take the library's
            # split reduction (the state's error 1.1e-6 -> 8.5e-7 of 64 bits, for 20 us)
            yq, yk, yv, og = _blas.project(xf, mats[:4])
            fa, br = (_blas.mm_f32(xf, w) for w in mats[4:])
        fb = _blas.project(fa, [self.fb])[0]
        wins = [None] * 3 if conv is None else [
            T.contiguous_aligned(conv[m].detach().to(dev, torch.float32).reshape(B, K - 1, P)) for m in range(3)]
        T.require_device(x, state)
        states = tuple(torch.empty((B, K - 1, P), dtype=torch.float32, device=dev) for _ in range(3))
        q, k, v, g = (torch.empty((Tn, B, H, D), dtype=torch.float32, device=dev) for _ in range(4))
        beta = torch.empty((Tn, B, H), dtype=torch.float32, device=dev)
        st = T.stream(x)
        _lib.call("k3_kda_prefill_inputs", *(T.ptr(t) for t in (yq, yk, yv, fb, br, self.qc, self.kc, self.vc, *wins,
                                                                *states, self.A_log, self.dt_bias, q, k, v, g, beta)),
                  B, Tn, H, D, K, float(c.kda_gate_lower_bound), st)
        state = _state(state, (B, H, D, D), dev)
        o = _recurrent(q, k, v, g, beta, D ** -0.5, state)
        y = torch.empty((B * Tn, P), dtype=torch.float32, device=dev)
        _lib.call("k3_kda_gated_norm", T.ptr(o), T.ptr(og), T.ptr(self.o_norm_w), float(c.rms_norm_eps), T.ptr(y), B, Tn,
                  H, D, st)
        return _blas.project(y, [self.o_w])[0].reshape(B, Tn, hid), state, states

    def __call__(self, x: torch.Tensor, state: torch.Tensor | None = None, conv: tuple | None = None):
        T.require_device(x, state)
        B, Tn, hid = x.shape
        if B * Tn > 1:
            return self.prefill(x, state, conv)
        H, D, K = self.H, self.D, self.K
        P = H * D
        state = _state(state, (B, H, D, D), x.device)
        if B * Tn == 0:      # nothing to do: the state and the windows as they came
            wins = [torch.zeros((B, K - 1, P), dtype=torch.float32, device=x.device) if conv is None
                    else conv[m].to(x.device, torch.float32).reshape(B, K - 1, P).clone() for m in range(3)]
            return torch.empty((B, Tn, hid), dtype=torch.float32, device=x.device), state, tuple(wins)
        # the windows of q, k and v in one buffer (one launch, or none where a caller passes back
        # the views a call returned); the step writes every element of the next ones
        fin = torch.empty((1, 3, K - 1, P), dtype=torch.float32, device=x.device)
        if conv is None:
            cin = torch.zeros((3, K - 1, P), dtype=torch.float32, device=x.device)
        else:
            wins = [c.to(x.device, torch.float32).reshape(1, K - 1, P) for c in conv]
            step = (K - 1) * P * 4
            if (all(c.is_contiguous() for c in wins) and wins[0].data_ptr() % 16 == 0
                    and all(wins[m].data_ptr() == wins[0].data_ptr() + m * step for m in (1, 2))):
                cin = wins[0]
            else:
                cin = torch.cat(wins)
        xin = x if x.dtype in (torch.float32, torch.bfloat16) else x.to(torch.float32)
        out = torch.empty((1, 1, hid), dtype=torch.float32, device=x.device)
        self.decode_step(T.contiguous_aligned(xin[0, 0]), state[0], cin, fin[0], out[0, 0])
        return out, state, (fin[:, 0], fin[:, 1], fin[:, 2])
