"""What this library is measured on: the calls a serving program makes, layer by layer.

Three kinds of layer make up a model of this class -- MXFP4 expert layers (plain and with the
latent wrapper), latent attention (MLA) and delta attention (KDA) -- and each runs in two
directions: decode (one token, or a few) and prefill (a prompt).  Every case is one layer, or
one projection or expert for programs that dispatch experts themselves, called through the
package's public entry points on a fresh state made from a seed.

Values: hidden states are unit-variance, dense weights have variance 1 / fan_in and the E8M0
scale bytes are set so that the MXFP4 weights have about that variance too, so activations
stay in the range in which SiLU / SiTU, the gates and the softmax actually bend.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path
from types import SimpleNamespace

import torch

_PKG = Path(__file__).resolve().parent.parent / "kimi-k3-mlx-macmini_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

from k3hip.kda import KDAAttention  # noqa: E402
from k3hip.mla import MLAAttention, MLACache, new_cache  # noqa: E402
from k3hip.moe import LatentMoE, MoEConfig, RoutedMoE, expert_ffn_fused  # noqa: E402
from k3hip.mxfp4_matvec import mxfp4_matvec_fused  # noqa: E402

DEV = "cuda"
BF16 = torch.bfloat16
KEY_GAP = 2e-5   # smallest distance kept between the last selected and the first rejected expert
EPS = 1e-5


# ------------------------------------------------------------------------------- the cases
def listed() -> list[dict]:
    return [
        # One MXFP4 projection of one decode token: the smallest call, what a program that
        # dispatches experts itself issues three times per selected expert.
        {"name": "matvec_one_token", "kind": "matvec", "tokens": 1, "n": 2048, "k": 7168, "x": "bf16"},
        # The same call on the tokens gathered for one expert of a short prompt or a batch of
        # sequences (an odd count: routing gives what it gives).
        {"name": "matvec_gathered_tokens", "kind": "matvec", "tokens": 37, "n": 3072, "k": 3584, "x": "bf16"},
        # One whole SwiGLU expert on one token.
        {"name": "expert_one_token", "kind": "expert", "hidden": 7168, "inter": 2048, "act": "silu", "x": "bf16"},
        # A decode step of one sequence through the 384-expert layer with its shared expert.
        {"name": "moe_layer_one_token", "kind": "moe", "tokens": 1, "hidden": 7168, "inter": 2048, "shared": 2048,
         "experts": 384, "top_k": 8, "router": "softmax", "act": "silu", "x": "bf16"},
        # A decode step of four sequences (or a speculative step of four tokens).
        {"name": "moe_layer_four_tokens", "kind": "moe", "tokens": 4, "hidden": 7168, "inter": 2048, "shared": 2048,
         "experts": 384, "top_k": 8, "router": "softmax", "act": "silu", "x": "bf16"},
        # An ordinary prompt through that layer; a length that fills no tile evenly.
        {"name": "moe_layer_prompt", "kind": "moe", "tokens": 700, "hidden": 7168, "inter": 2048, "shared": 2048,
         "experts": 384, "top_k": 8, "router": "softmax", "act": "silu", "x": "bf16"},
        # A decode step through the 896-expert layer with the latent wrapper.
        {"name": "latent_layer_one_token", "kind": "latent", "tokens": 1, "hidden": 7168, "latent": 3584,
         "inter": 3072, "shared": 6144, "experts": 896, "top_k": 16, "x": "bf16"},
        # A long prompt through it: the largest case.
        {"name": "latent_layer_prompt", "kind": "latent", "tokens": 2048, "hidden": 7168, "latent": 3584,
         "inter": 3072, "shared": 6144, "experts": 896, "top_k": 16, "x": "bf16"},
        # A decode step through a latent attention layer late in a long conversation.
        {"name": "mla_layer_one_token", "kind": "mla", "tokens": 1, "past": 32767, "hidden": 7168, "heads": 64,
         "q_rank": 1536, "gate": True, "x": "bf16", "cache": "bf16"},
        # A prompt through it.
        {"name": "mla_layer_prompt", "kind": "mla", "tokens": 1000, "past": 0, "hidden": 7168, "heads": 64,
         "q_rank": 1536, "gate": True, "x": "bf16", "cache": "bf16"},
        # A decode step through a delta attention layer, from a kept state.
        {"name": "kda_layer_one_token", "kind": "kda", "tokens": 1, "hidden": 7168, "heads": 96, "x": "bf16"},
        # A prompt through it.
        {"name": "kda_layer_prompt", "kind": "kda", "tokens": 256, "hidden": 7168, "heads": 96, "x": "bf16"},
    ]


def _log(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo: int, hi: int, step: int) -> int:
    return step * _log(rng, lo / step, hi / step)


def draw(rng) -> dict:
    """One more case: any of the calls above at sizes, dtypes and options of their ranges."""
    kind = rng.choice(["matvec", "matvec", "expert", "moe", "moe", "latent", "latent", "mla", "mla", "kda", "kda"])
    x = rng.choice(["bf16", "bf16", "bf16", "fp32"])
    if kind == "matvec":
        # a few rows, or the tokens one expert gets of a prompt; rows and columns of any
        # expert projection, N of any parity, K of whole 32-element groups
        return {"kind": kind, "tokens": rng.choice([1, _log(rng, 2, 8), _log(rng, 9, 256)]),
                "n": _log(rng, 300, 8192), "k": _mult(rng, 256, 7168, 32), "x": x}
    if kind == "expert":
        return {"kind": kind, "hidden": _mult(rng, 1024, 7168, 128), "inter": _mult(rng, 512, 4096, 128),
                "act": rng.choice(["silu", "situ"]), "x": x}
    if kind == "moe":
        return {"kind": kind, "tokens": rng.choice([1, rng.randint(2, 8), _log(rng, 9, 2048)]),
                "hidden": _mult(rng, 1024, 7168, 256), "inter": _mult(rng, 512, 2048, 128),
                "shared": rng.choice([0, _mult(rng, 512, 2048, 128)]), "experts": _log(rng, 32, 384),
                "top_k": rng.choice([2, 4, 6, 8]), "router": rng.choice(["softmax", "sigmoid_bias"]),
                "act": rng.choice(["silu", "situ"]), "x": x}
    if kind == "latent":
        return {"kind": kind, "tokens": rng.choice([1, rng.randint(2, 8), _log(rng, 9, 2048)]),
                "hidden": _mult(rng, 2048, 7168, 256), "latent": _mult(rng, 1024, 3584, 128),
                "inter": _mult(rng, 512, 3072, 128), "shared": _mult(rng, 1024, 6144, 128),
                "experts": _log(rng, 64, 512), "top_k": rng.choice([4, 8, 16]), "x": x}
    if kind == "mla":
        one = rng.random() < 0.5
        return {"kind": kind, "tokens": 1 if one else _log(rng, 2, 1000),
                "past": _log(rng, 16, 32767) if one else rng.choice([0, _log(rng, 16, 1000)]),
                "hidden": rng.choice([2048, 4096, 7168]), "heads": rng.choice([16, 32, 64]),
                "q_rank": rng.choice([768, 1536]), "gate": rng.random() < 0.7, "x": "bf16",
                "cache": rng.choice(["bf16", "bf16", "fp32"])}
    return {"kind": kind, "tokens": rng.choice([1, rng.randint(2, 8), _log(rng, 9, 256)]),
            "hidden": rng.choice([2048, 4096, 7168]), "heads": rng.choice([16, 32, 64, 96]), "x": "bf16"}


# ------------------------------------------------------------------------------- the inputs
class _Rand:
    def __init__(self, seed: int):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def n(self, *s, std: float = 1.0):
        return torch.randn(*s, device=DEV, generator=self.g) * std

    def lin(self, o: int, i: int):
        return self.n(o, i, std=i ** -0.5).to(BF16)

    def mxfp4(self, n: int, k: int):
        """Random codes with scales that put the weights' deviation at about k ** -0.5 (the
        root mean square of the eight E2M1 magnitudes is 2.93)."""
        packed = torch.randint(-2 ** 31, 2 ** 31, ((n * k // 2 + 3) // 4,), dtype=torch.int32, device=DEV,
                               generator=self.g).view(torch.uint8)[:n * k // 2].view(n, k // 2)
        mid = 127 - round(math.log2(2.93 * k ** 0.5))
        scales = torch.randint(mid - 1, mid + 2, (n, k // 32), dtype=torch.uint8, device=DEV, generator=self.g)
        return packed, scales

    def expert(self, hidden: int, inter: int):
        return self.mxfp4(inter, hidden), self.mxfp4(inter, hidden), self.mxfp4(hidden, inter)


def _dt(case):
    return BF16 if case.get("x", "bf16") == "bf16" else torch.float32


_SITU = {"situ_beta": 2.0, "situ_linear_beta": 3.0}
_WHICH = {"w1": 0, "w3": 1, "w2": 2}


def _routed_x(r: _Rand, case, gate_w, bias):
    """Hidden states whose routing is not decided by rounding: of the tokens drawn, those
    whose last selected expert is further than KEY_GAP above the first rejected one."""
    T, k = case["tokens"], case["top_k"]
    if k >= case["experts"]:
        return r.n(T, case["hidden"]).to(_dt(case))
    x = r.n(T + 16 + T // 16, case["hidden"]).to(_dt(case))
    key = x.double() @ gate_w.double().T
    if bias is not None:
        key = torch.sigmoid(key) + bias.double()
    top = key.topk(k + 1, dim=1).values
    keep = (top[:, k - 1] - top[:, k] > KEY_GAP).nonzero().flatten()[:T]
    return x[keep].contiguous()


def _mla_cfg(case):
    return SimpleNamespace(hidden_size=case["hidden"], num_attention_heads=case["heads"], q_lora_rank=case["q_rank"],
                           kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64, v_head_dim=128,
                           q_head_dim=192, rms_norm_eps=EPS, mla_use_output_gate=case["gate"],
                           mla_cache_dtype=BF16 if case["cache"] == "bf16" else torch.float32)


def prepare(case: dict, seed: int):
    r = _Rand(seed)
    kind = case["kind"]
    s = SimpleNamespace(case=case)
    if kind == "matvec":
        s.w = r.mxfp4(case["n"], case["k"])
        s.x = r.n(case["tokens"], case["k"]).to(_dt(case))
    elif kind == "expert":
        s.e = r.expert(case["hidden"], case["inter"])
        s.x = r.n(1, case["hidden"]).to(_dt(case))
    elif kind in ("moe", "latent"):
        H, E, Is = case["hidden"], case["experts"], case["shared"]
        width = case["latent"] if kind == "latent" else H
        experts = [r.expert(width, case["inter"]) for _ in range(E)]
        # the router's rows differ in length, so the experts' loads differ as trained ones' do
        w = {"gate.weight": (r.n(E, H, std=1.7 * H ** -0.5) * (1 + 0.1 * r.n(E, 1))).to(BF16)}
        bias = None
        if kind == "latent" or case["router"] == "sigmoid_bias":
            bias = r.n(E, std=0.05)
            w["gate.e_score_correction_bias"] = bias
        if Is:
            w.update({"shared_experts.gate_proj.weight": r.lin(Is, H), "shared_experts.up_proj.weight": r.lin(Is, H),
                      "shared_experts.down_proj.weight": r.lin(H, Is)})
        source = lambda layer, e, which: experts[e][_WHICH[which]]  # noqa: E731
        if kind == "latent":
            w.update({"routed_expert_down_proj.weight": r.lin(width, H), "routed_expert_up_proj.weight": r.lin(H, width),
                      "routed_expert_norm.weight": 1 + 0.1 * r.n(width)})
            cfg = SimpleNamespace(hidden_size=H, routed_expert_hidden_size=width, moe_intermediate_size=case["inter"],
                                  num_experts=E, num_experts_per_token=case["top_k"], moe_renormalize=True,
                                  routed_scaling_factor=2.5, rms_norm_eps=EPS, **_SITU)
            s.layer = LatentMoE(cfg, 0, w, source)
            s.layer._routed.expert_table()
        else:
            cfg = MoEConfig(hidden_size=H, moe_intermediate_size=case["inter"], num_experts=E,
                            num_experts_per_token=case["top_k"], shared_intermediate_size=Is, router=case["router"],
                            activation=case["act"], routed_scaling_factor=2.5 if bias is not None else 1.0, **_SITU)
            s.layer = RoutedMoE(cfg, 0, w, source)
            s.layer.expert_table()
        s.experts, s.w = experts, w
        s.x = _routed_x(r, case, w["gate.weight"], bias)
    elif kind == "mla":
        H, hid, ql = case["heads"], case["hidden"], case["q_rank"]
        s.w = {"q_a_proj.weight": r.lin(ql, hid), "q_a_layernorm.weight": 1 + 0.1 * r.n(ql),
               "q_b_proj.weight": r.lin(H * 192, ql), "kv_a_proj_with_mqa.weight": r.lin(576, hid),
               "kv_a_layernorm.weight": 1 + 0.1 * r.n(512), "kv_b_proj.weight": r.lin(H * 256, 512),
               "g_proj.weight": r.lin(H * 128, hid), "o_proj.weight": r.lin(hid, H * 128)}
        cfg = _mla_cfg(case)
        s.layer = MLAAttention(cfg, s.w)
        past, T = case["past"], case["tokens"]
        s.past = (r.n(1, past, 512), r.n(1, past, 64)) if past else None
        s.cache = new_cache(1, 512, 64, past + T, cfg.mla_cache_dtype, DEV)
        if past:
            s.cache.append(*s.past)
            s.past = tuple(t.to(cfg.mla_cache_dtype) for t in s.past)
        s.x = r.n(1, T, hid).to(_dt(case))
    elif kind == "kda":
        H, hid, P = case["heads"], case["hidden"], case["heads"] * 128
        a = torch.zeros(128, device=DEV)
        a[:H] = torch.log(1 + 15 * torch.rand(H, device=DEV, generator=r.g))
        s.w = {f"{n}_proj.weight": r.lin(P, hid) for n in "qkvg"}
        s.w.update({"o_proj.weight": r.lin(hid, P), "f_a_proj.weight": r.lin(128, hid),
                    "f_b_proj.weight": r.lin(P, 128), "b_proj.weight": r.lin(H, hid),
                    "o_norm.weight": 1 + 0.1 * r.n(128), "A_log": a, "dt_bias": r.n(P)})
        s.w.update({f"{n}_conv1d.weight": r.n(P, 1, 4, std=0.3) for n in "qkv"})
        cfg = SimpleNamespace(hidden_size=hid, kda_num_heads=H, kda_head_dim=128, kda_conv_size=4,
                              kda_gate_lower_bound=-5.0, rms_norm_eps=EPS)
        s.layer = KDAAttention(cfg, s.w)
        # the state and convolution windows kept after a prefix; each pass continues from them
        s.kept = r.n(1, H, 128, 128, std=0.1)
        s.state = torch.empty_like(s.kept)
        s.conv = tuple(r.n(1, 3, P) for _ in range(3))
        s.x = r.n(1, case["tokens"], hid).to(_dt(case))
    return s


def run(s):
    c = s.case
    kind = c["kind"]
    if kind == "matvec":
        return mxfp4_matvec_fused(s.x, *s.w)
    if kind == "expert":
        if c["act"] == "situ":
            return expert_ffn_fused(s.x, *s.e, act="situ", beta=2.0, linear_beta=3.0)
        return expert_ffn_fused(s.x, *s.e)
    if kind in ("moe", "latent"):
        return s.layer(s.x)
    if kind == "mla":
        s.cache.length = c["past"]      # continue from the kept prefix (the cache rows stay)
        out, cache = s.layer(s.x, s.cache)
        return out, *(t[:, c["past"]:] for t in cache.view())
    s.state.copy_(s.kept)               # the layer updates the state it is given
    out, state, conv = s.layer(s.x, s.state, s.conv)
    return out, state, *conv


# ---------------------------------------------------------------------- bytes and operations
def _mx(n, k):
    return n * k // 2 + n * k // 32


def work(case: dict) -> dict:
    c, kind = case, case["kind"]
    T, xs = c.get("tokens", 1), 2 if c.get("x", "bf16") == "bf16" else 4
    if kind == "matvec":
        return {"bytes": _mx(c["n"], c["k"]) + T * (c["k"] * xs + c["n"] * 4), "flops": 2 * T * c["n"] * c["k"]}
    if kind == "expert":
        H, i = c["hidden"], c["inter"]
        return {"bytes": 3 * _mx(i, H) + H * (xs + 4), "flops": 6 * H * i}
    if kind in ("moe", "latent"):
        H, i, E, k, Is = c["hidden"], c["inter"], c["experts"], c["top_k"], c["shared"]
        width = c["latent"] if kind == "latent" else H
        used = E * (1 - (1 - k / E) ** T)          # distinct experts T tokens select
        dense = E * H + 3 * Is * H + (2 * width * H if kind == "latent" else 0)
        return {"bytes": int(used * 3 * _mx(i, width)) + 2 * dense + T * H * (xs + 4),
                "flops": 2 * T * (k * 3 * i * width + dense)}
    if kind == "mla":
        H, hid, ql, past = c["heads"], c["hidden"], c["q_rank"], c["past"]
        dense = ql * hid + H * 192 * ql + 576 * hid + hid * H * 128 + (H * 128 * hid if c["gate"] else 0)
        pairs = T * past + T * (T + 1) // 2        # (query, key) pairs under the causal mask
        # one token: the absorbed form (scores and context at the latent width); a prompt:
        # keys and values expanded once, scores over 192 and context over 128 columns
        absorbed = T * H * 256 * 512 + pairs * H * (576 + 512)
        expanded = (past + T) * H * 256 * 512 + pairs * H * (192 + 128)
        row = 576 * (2 if c["cache"] == "bf16" else 4)
        return {"bytes": 2 * (dense + H * 256 * 512) + (past + T) * row + T * hid * (xs + 4),
                "flops": 2 * (T * dense + min(absorbed, expanded))}
    H, hid, P = c["heads"], c["hidden"], c["heads"] * 128
    dense = 5 * P * hid + 128 * hid + P * 128 + H * hid
    state = 2 * H * 128 * 128 * 4 + 2 * 3 * 3 * P * 4
    return {"bytes": 2 * dense + state + T * hid * (xs + 4), "flops": 2 * T * dense + T * H * 128 * 128 * 7}


def tolerance(case: dict) -> dict:
    """About four times the largest distance from 64 bits that the ranges above showed."""
    kind, T = case["kind"], case.get("tokens", 1)
    if kind in ("matvec", "expert") or (kind == "moe" and T <= 8):
        return {"rel": 1e-6}      # fp32 sums over exact weights: up to 2.5e-7
    if kind == "moe":
        return {"rel": 8e-5}      # prompts: 12-bit activations and matrix-core sums, 2.0e-5
    if kind == "latent":
        # a latent state of bf16: an element whose sum falls on the other side of a rounding
        # boundary moves its token's output; 7.3e-5
        return {"rel": 3e-4}
    if kind == "mla":
        return {"rel": 4.5e-4}    # the same of a bf16 cache row: 1.1e-4
    return {"rel": 1.2e-6} if T <= 8 else {"rel": 1e-5}   # fp32 sums: 2.9e-7 and 2.3e-6


# ------------------------------------------------------------- the same outputs in 64 bits
_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _decode(w):
    packed, scales = w
    lut = torch.tensor(_E2M1 + [-v for v in _E2M1], dtype=torch.float64, device=packed.device)
    codes = torch.stack([packed & 15, packed >> 4], dim=-1).flatten(1).int()
    return lut[codes] * torch.exp2(scales.double() - 127).repeat_interleave(32, dim=1)


def _act(g, u, act):
    if act == "situ":
        b, lb = _SITU["situ_beta"], _SITU["situ_linear_beta"]
        return b * torch.tanh(g / b) * torch.sigmoid(g) * (lb * torch.tanh(u / lb))
    return g * torch.sigmoid(g) * u


def _expert64(x, e, act):
    return _act(x @ _decode(e[0]).T, x @ _decode(e[1]).T, act) @ _decode(e[2]).T


def _rms(x, w):
    return w.double() * x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)


def _moe64(s):
    c, w, x = s.case, {n: t.double() for n, t in s.w.items()}, s.x.double()
    logits = x @ w["gate.weight"].T
    latent = c["kind"] == "latent"
    if "gate.e_score_correction_bias" in w:
        raw = torch.sigmoid(logits)
        idx = (raw + w["gate.e_score_correction_bias"]).topk(c["top_k"], dim=1).indices
        scaling = 2.5
    else:
        raw = torch.softmax(logits, dim=1)
        idx = raw.topk(c["top_k"], dim=1).indices
        scaling = 1.0
    wt = raw.gather(1, idx)
    wt = wt / (wt.sum(1, keepdim=True) + 1e-20) * scaling
    h, act = x, "situ" if latent else c["act"]
    if latent:
        h = x @ w["routed_expert_down_proj.weight"].T
        if s.x.dtype == BF16:
            h = h.to(BF16).double()      # the layer keeps its latent state in x's dtype
    y = torch.zeros_like(h)
    for e in idx.unique().tolist():
        tok, slot = (idx == e).nonzero(as_tuple=True)
        y.index_add_(0, tok, _expert64(h[tok], s.experts[e], act) * wt[tok, slot, None])
    if latent:
        y = _rms(y, s.w["routed_expert_norm.weight"]) @ w["routed_expert_up_proj.weight"].T
    if c["shared"]:
        y = y + _act(x @ w["shared_experts.gate_proj.weight"].T, x @ w["shared_experts.up_proj.weight"].T,
                     act) @ w["shared_experts.down_proj.weight"].T
    return y


def _mla64(s):
    c, x, T, H, past = s.case, s.x[0].double(), s.case["tokens"], s.case["heads"], s.case["past"]
    w = {n: t.double() for n, t in s.w.items()}
    q = (_rms(x @ w["q_a_proj.weight"].T, s.w["q_a_layernorm.weight"]) @ w["q_b_proj.weight"].T).view(T, H, 192)
    ckv = x @ w["kv_a_proj_with_mqa.weight"].T
    cdt = s.cache.latent.dtype
    lat = _rms(ckv[:, :512], s.w["kv_a_layernorm.weight"]).to(cdt)
    rot = ckv[:, 512:].to(cdt)
    new = (lat.double()[None], rot.double()[None])
    if past:
        lat, rot = torch.cat([s.past[0][0], lat]), torch.cat([s.past[1][0], rot])
    lat, rot = lat.double(), rot.double()
    kb = w["kv_b_proj.weight"].view(H, 256, 512)
    mask = torch.arange(past + T, device=x.device)[None] > torch.arange(past, past + T, device=x.device)[:, None]
    o = torch.empty(T, H, 128, dtype=torch.float64, device=x.device)
    for h in range(H):
        sc = ((q[:, h, :128] @ kb[h, :128]) @ lat.T + q[:, h, 128:] @ rot.T) * 192 ** -0.5
        p = torch.softmax(sc.masked_fill(mask, -math.inf), dim=-1)
        o[:, h] = (p @ lat) @ kb[h, 128:].T
    o = o.view(T, H * 128)
    if c["gate"]:
        o = o * torch.sigmoid(x @ w["g_proj.weight"].T)
    return (o @ w["o_proj.weight"].T)[None], *new


def _kda64(s):
    c, x, T, H = s.case, s.x[0].double(), s.case["tokens"], s.case["heads"]
    w = {n: t.double() for n, t in s.w.items()}
    streams, windows = [], []
    for n, win in zip("qkv", s.conv):
        xp = torch.cat([win[0].double(), x @ w[f"{n}_proj.weight"].T])
        cw = w[f"{n}_conv1d.weight"].view(-1, 4)
        z = sum(cw[:, j] * xp[j:j + T] for j in range(4))
        streams.append((z * torch.sigmoid(z)).view(T, H, 128))
        windows.append(xp[T:][None])
    q, k, v = streams
    q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) * 128 ** -0.5
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    g = ((x @ w["f_a_proj.weight"].T) @ w["f_b_proj.weight"].T + w["dt_bias"]).view(T, H, 128)
    g = -5.0 * torch.sigmoid(torch.exp(w["A_log"][:H, None]) * g)
    beta = torch.sigmoid(x @ w["b_proj.weight"].T)
    S = s.kept[0].double()
    o = torch.empty(T, H, 128, dtype=torch.float64, device=x.device)
    for t in range(T):
        S = S * g[t].exp()[..., None]
        d = (v[t] - (k[t][..., None] * S).sum(1)) * beta[t][:, None]
        S = S + k[t][..., None] * d[:, None]
        o[t] = (q[t][..., None] * S).sum(1)
    o = _rms(o, s.w["o_norm.weight"]) * torch.sigmoid(x @ w["g_proj.weight"].T).view(T, H, 128)
    return (o.reshape(T, -1) @ w["o_proj.weight"].T)[None], S[None], *windows


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "matvec":
        return s.x.double() @ _decode(s.w).T
    if kind == "expert":
        return _expert64(s.x.double(), s.e, case["act"])
    return {"moe": _moe64, "latent": _moe64, "mla": _mla64, "kda": _kda64}[kind](s)
