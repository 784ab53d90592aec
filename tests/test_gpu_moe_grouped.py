"""GPU parity of the grouped (prefill) routed-expert path against the fp64 oracle.

Tolerance: normwise max-relative error <= 2e-5.  The weights are exact in bf16, bf16 x is
exact; an fp32 x and the activation enter as two bf16 terms, 16 bits, so each is off by at
most 2^-17 = 7.6e-6 of itself and of either sign, and sums are fp32 (observed 1.4e-6 ..
3.9e-6 on these cases).
"""
from __future__ import annotations

import os

import numpy as np
import pytest
import torch

from oracle import moe as omoe
from oracle import mxfp4 as om

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 2e-5


def make_experts(rng, D, H, I):
    ex_np = [(om.random_mxfp4(rng, I, H), om.random_mxfp4(rng, I, H), om.random_mxfp4(rng, H, I)) for _ in range(D)]
    ex_dev = [tuple(tuple(torch.from_numpy(a).to(DEV) for a in pair) for pair in ex) for ex in ex_np]
    return ex_np, ex_dev


def table_of(ex_dev, E):
    D = len(ex_dev)
    rows = []
    for e in range(E):
        (gp, gs), (upk, us), (dp, ds) = ex_dev[e % D]
        rows.append([t.data_ptr() for t in (gp, gs, upk, us, dp, ds)])
    return torch.tensor(rows, dtype=torch.int64, device=DEV)


def distinct_routing(rng, T, E, k):
    idx = np.stack([rng.choice(E, size=k, replace=False) for _ in range(T)]).astype(np.int32)
    w = rng.random((T, k)).astype(np.float32)
    return idx, w / w.sum(axis=1, keepdims=True)


def zipf_routing(rng, T, E, k, s=1.1):
    """Gumbel-top-k on log r^-s over a seeded permutation: k distinct experts per token,
    drawn without replacement with probability proportional to the Zipf weights."""
    perm = rng.permutation(E)
    logw = -s * np.log(np.arange(1, E + 1, dtype=np.float64))[np.argsort(perm)]
    g = logw[None, :] - np.log(-np.log(rng.random((T, E))))
    idx = np.argsort(-g, axis=1)[:, :k].astype(np.int32)
    z = rng.standard_normal((T, k))
    w = np.exp(z - z.max(axis=1, keepdims=True))
    return idx, (w / w.sum(axis=1, keepdims=True)).astype(np.float32)


def run(x32, idx, w, ex_dev, E, I, act="silu", beta=1.0, lbeta=None, out_dtype=torch.float32):
    from k3hip.moe import moe_grouped_ffn
    x = torch.from_numpy(x32).to(DEV).to(torch.bfloat16)
    y = moe_grouped_ffn(x, torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV), table_of(ex_dev, E), I,
                        act, beta, lbeta, out_dtype=out_dtype)
    torch.cuda.synchronize()
    return y.float().cpu().numpy()


CASES = [
    # T, H, I, E, k, D, routing, act
    (40, 512, 256, 8, 2, 8, "distinct", "silu"),
    (130, 1024, 384, 16, 4, 16, "hot", "situ"),
    (77, 768, 192, 64, 3, 5, "few", "silu"),
    (300, 2048, 512, 32, 8, 4, "distinct", "silu"),
]


@pytest.mark.parametrize("T,H,I,E,k,D,routing,act", CASES)
def test_grouped_matches_oracle(T, H, I, E, k, D, routing, act):
    rng = np.random.default_rng(4000 + T)
    ex_np, ex_dev = make_experts(rng, D, H, I)
    if routing == "hot":      # expert 3 in every token: 130 rows = 4 full tiles + 1 partial
        idx, w = distinct_routing(rng, T, E, k)
        for t in range(T):
            if 3 not in idx[t]:
                idx[t, 0] = 3
    elif routing == "few":    # most experts empty
        idx = np.stack([rng.choice(5, size=k, replace=False) * 7 for _ in range(T)]).astype(np.int32)
        w = rng.random((T, k)).astype(np.float32)
    else:
        idx, w = distinct_routing(rng, T, E, k)
    x32 = om.bf16_round(rng.standard_normal((T, H)).astype(np.float32))
    beta, lbeta = (1.5, 3.0) if act == "situ" else (1.0, None)
    got = run(x32, idx, w, ex_dev, E, I, act, beta, lbeta)
    experts = {e: ex_np[e % D] for e in range(E)}
    want = omoe.moe_layer(x32, idx, w, experts, None, kind=act, beta=beta, linear_beta=lbeta)
    rel = om.normwise_rel(got, want)
    print(f"T={T} H={H} I={I} E={E} k={k} rel={rel:.3e}")
    assert rel <= TOL


def device_experts(E, H, I, seed):
    """E distinct MXFP4 experts drawn on the device (scale bytes in [118, 130], as the
    benchmark's generator), so no two table rows alias one weight set."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)

    def mx(n, kk):
        return (torch.randint(0, 256, (n, kk // 2), dtype=torch.uint8, device=DEV, generator=g),
                torch.randint(118, 131, (n, kk // 32), dtype=torch.uint8, device=DEV, generator=g))

    return [(mx(I, H), mx(I, H), mx(H, I)) for _ in range(E)]


class HostExperts:
    """experts[e] for the oracle: the device expert's (packed, scales) pairs copied to host
    memory on access (only the experts the sampled tokens use are ever copied)."""

    def __init__(self, ex_dev):
        self.ex_dev = ex_dev

    def __getitem__(self, e):
        return tuple(tuple(a.cpu().numpy() for a in pair) for pair in self.ex_dev[e])


def oracle_workers():
    return max(1, min(16, len(os.sched_getaffinity(0))))


def test_grouped_full_shape_every_expert_distinct():
    """2048 tokens x top-8 over 384 distinct experts (9 GB of weights drawn on the device),
    Zipf(1.1) load, hidden 7168, intermediate 2048.  At least 320 tokens against the fp64
    oracle: the first and last token of every 64-token tile of the four hottest experts (in
    the grouped order, which is token order), the token of every expert routed exactly
    once, the first and last tokens, and a random draw; two runs bit-identical.  Every
    (token, slot) pair of the sample reaches its own expert's weights, so a wrong
    expert-to-weight mapping fails."""
    T, H, I, E, k = 2048, 7168, 2048, 384, 8
    ex_dev = device_experts(E, H, I, seed=1004)
    rng = np.random.default_rng(1004)
    idx, w = zipf_routing(rng, T, E, k)
    x32 = om.bf16_round(rng.standard_normal((T, H)).astype(np.float32))
    counts = np.bincount(idx.ravel(), minlength=E)
    assert counts.max() > 1000 and (counts == 0).sum() < E  # skewed, with a hot head
    got = run(x32, idx, w, ex_dev, E, I)
    again = run(x32, idx, w, ex_dev, E, I)
    assert np.array_equal(got, again)
    edges = set()
    for hot in np.argsort(-counts, kind="stable")[:4]:
        toks = np.nonzero((idx == hot).any(axis=1))[0]        # grouped rows of the expert, in order
        edges |= {int(toks[m]) for m0 in range(0, len(toks), 64) for m in (m0, min(m0 + 63, len(toks) - 1))}
    singles = {int(np.nonzero((idx == e).any(axis=1))[0][0]) for e in np.nonzero(counts == 1)[0]}
    sample = edges | singles | {0, 1, T - 2, T - 1}
    rest = np.setdiff1d(np.arange(T), sorted(sample))
    sample = sorted(sample | {int(t) for t in rng.choice(rest, max(0, 320 - len(sample)), replace=False)})
    want = omoe.moe_layer(x32[sample], idx[sample], w[sample], HostExperts(ex_dev), workers=oracle_workers())
    rel = om.normwise_rel(got[sample], want)
    used = len(set(idx[sample].ravel().tolist()))
    print(f"full shape: {len(sample)} sampled tokens ({len(edges)} hot-tile edges, {len(singles)} single-token "
          f"experts) over {used} distinct experts, rel={rel:.3e}")
    assert len(sample) >= 320 and used > 280
    assert rel <= TOL


def test_grouped_bf16_output_and_errors():
    from k3hip.moe import moe_grouped_ffn
    rng = np.random.default_rng(9)
    ex_np, ex_dev = make_experts(rng, 2, 256, 128)
    idx, w = distinct_routing(rng, 10, 2, 2)
    x32 = om.bf16_round(rng.standard_normal((10, 256)).astype(np.float32))
    y32 = run(x32, idx, w, ex_dev, 2, 128)
    y16 = run(x32, idx, w, ex_dev, 2, 128, out_dtype=torch.bfloat16)
    assert np.array_equal(y16, om.bf16_round(y32))
    x = torch.from_numpy(x32).to(DEV).to(torch.bfloat16)
    tab = table_of(ex_dev, 2)
    with pytest.raises(ValueError):   # expert id out of range
        moe_grouped_ffn(x, torch.full((10, 2), 5, device=DEV), torch.ones(10, 2, device=DEV), tab, 128)
    # fp32 hidden states take two bf16 terms; for bf16-exact values the second is zero, so
    # the result equals the bf16 path's
    ti, tw = torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV)
    yf = moe_grouped_ffn(x.float(), ti, tw, tab, 128).cpu().numpy()
    assert np.allclose(yf, moe_grouped_ffn(x, ti, tw, tab, 128).cpu().numpy(), rtol=1e-6, atol=1e-6)
    with pytest.raises(ValueError):   # H not a multiple of 64
        moe_grouped_ffn(x[:, :200], torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV), tab, 128)


def test_routed_moe_grouped_forward_matches_decode_path():
    """RoutedMoE.grouped_forward (prefill) vs its own per-token decode kernels, shared
    expert included: the two device paths agree to the tolerance."""
    from k3hip.moe import MoEConfig, RoutedMoE
    H, I, E, k, Is = 1024, 256, 16, 4, 256
    rng = np.random.default_rng(12)
    ex_np, ex_dev = make_experts(rng, E, H, I)
    w = {"gate.weight": torch.from_numpy(om.bf16_round((rng.standard_normal((E, H)) * 0.02).astype(np.float32))
                                         ).to(DEV).to(torch.bfloat16)}
    for name, shape in (("gate", (Is, H)), ("up", (Is, H)), ("down", (H, Is))):
        w[f"shared_experts.{name}_proj.weight"] = (torch.randn(*shape, device=DEV) * 0.02).to(torch.bfloat16)
    which = {"w1": 0, "w3": 1, "w2": 2}
    cfg = MoEConfig(hidden_size=H, moe_intermediate_size=I, num_experts=E, num_experts_per_token=k,
                    shared_intermediate_size=Is)
    moe = RoutedMoE(cfg, 0, w, lambda L, e, wh: ex_dev[e][which[wh]])
    x = torch.from_numpy(om.bf16_round(rng.standard_normal((48, H)).astype(np.float32))).to(DEV).to(torch.bfloat16)
    a = moe.grouped_forward(x).cpu().numpy()
    b = moe(x).cpu().numpy()
    assert om.normwise_rel(a, b) <= TOL


@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,I,off", [(320, 192, 0), (256, 128, 1), (1088, 448, 3), (64, 64, 2)])
def test_grouped_tile_edges(H, I, off, xdt):
    """Experts of 1, 15, 16, 17, 33, 48, 49, 64, 65 and 130 rows (every column-group count, full
    and part tiles), K of whole and part 256-steps, row blocks that end past the last weight
    row, scale rows at every byte alignment, bf16 and fp32 x, against fp64 torch.  Products are
    exact; x in fp32 and the activation keep 16 bits (2^-17 each), sums are fp32: 2e-5."""
    from k3hip.moe import moe_grouped_ffn
    g = torch.Generator(device=DEV)
    g.manual_seed(H + I + off)
    counts = [1, 15, 16, 17, 33, 48, 49, 64, 65, 130, 0]
    E = len(counts)
    ids = torch.cat([torch.full((c,), e, device=DEV) for e, c in enumerate(counts)])
    ids = ids[torch.randperm(len(ids), device=DEV, generator=g)].view(-1, 2)      # top-2, an id twice at times
    T = ids.shape[0]
    lut = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], dtype=torch.float64, device=DEV)
    lut = torch.cat([lut, -lut])

    def mx(n, k):
        p = torch.randint(0, 256, (n, k // 2), dtype=torch.uint8, device=DEV, generator=g)
        buf = torch.randint(118, 124, (n * (k // 32) + 4,), dtype=torch.uint8, device=DEV, generator=g)
        return p, buf[off:off + n * (k // 32)].view(n, k // 32)

    def dec(w):
        codes = torch.stack([w[0] & 15, w[0] >> 4], dim=-1).flatten(1).int()
        return lut[codes] * torch.exp2(w[1].double() - 127).repeat_interleave(32, dim=1)

    ex = [(mx(I, H), mx(I, H), mx(H, I)) for _ in range(E)]
    table = torch.tensor([[t.data_ptr() for pair in e for t in pair] for e in ex], dtype=torch.int64, device=DEV)
    x = torch.randn(T, H, device=DEV, generator=g).to(xdt)
    w = torch.rand(T, 2, device=DEV, generator=g)
    got = moe_grouped_ffn(x, ids, w, table, I, "situ", 2.0, 3.0)
    want = torch.zeros(T, H, dtype=torch.float64, device=DEV)
    for j in range(2):
        for e in range(E):
            t = (ids[:, j] == e).nonzero().flatten()
            a, u = x[t].double() @ dec(ex[e][0]).T, x[t].double() @ dec(ex[e][1]).T
            act = 2 * torch.tanh(a / 2) * torch.sigmoid(a) * 3 * torch.tanh(u / 3)
            want.index_add_(0, t, act @ dec(ex[e][2]).T * w[t, j, None].double())
    rel = float((got.double() - want).norm() / want.norm())
    print(f"H={H} I={I} scale offset {off} {xdt}: {rel:.2e}")
    assert rel <= 2e-5
    assert torch.equal(got, moe_grouped_ffn(x, ids, w, table, I, "situ", 2.0, 3.0))


def _prompts(E, H, I, k, sizes):
    from k3hip.moe import moe_grouped_ffn
    rng = np.random.default_rng(31)
    _, ex_dev = make_experts(rng, 4, H, I)
    table = table_of(ex_dev, E)
    calls = []
    for T in sizes:
        idx, w = distinct_routing(rng, T, E, k)
        args = [torch.from_numpy(om.bf16_round(rng.standard_normal((T, H)).astype(np.float32))).to(DEV).to(torch.bfloat16),
                torch.from_numpy(idx).to(DEV), torch.from_numpy(w).to(DEV), table, I]
        calls.append(lambda a=args: moe_grouped_ffn(*a, validate=False))
    return calls, (ex_dev, table)


def test_grouped_replay_after_larger_calls():
    """A captured prompt keeps its own scratch: later, larger prompts on its stream and whatever takes
    the memory they free leave its replays as the eager result."""
    (small, big, bigger), keep = _prompts(16, 256, 128, 4, (20, 150, 700))
    want = small().clone()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        small()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = small()
    for call in (big, bigger, small):
        with torch.cuda.stream(stream):
            call()
            junk = [torch.full((n,), 0x7f, dtype=torch.uint8, device=DEV) for n in (1 << 17, 1 << 19, 1 << 21, 1 << 23)]
        torch.cuda.synchronize()
        del junk
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(small(), want)


def test_grouped_threads_on_one_stream():
    """Two threads run prompts of different sizes on one stream, their launches in any order."""
    import threading
    calls, keep = _prompts(16, 256, 128, 4, (40, 150))
    want = [c().clone() for c in calls]
    torch.cuda.synchronize()
    stream, got, errors = torch.cuda.Stream(), [[], []], []
    start = threading.Barrier(2)

    def work(i):
        try:
            start.wait()
            with torch.cuda.stream(stream):
                for _ in range(40):
                    got[i].append(calls[i]())
        except Exception as e:  # reported below
            errors.append(repr(e))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    stream.synchronize()
    assert not errors and not any(t.is_alive() for t in threads)
    for i in range(2):
        assert len(got[i]) == 40 and all(torch.equal(y, want[i]) for y in got[i])
