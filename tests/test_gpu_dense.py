"""GPU parity of the dense projections for many tokens (k3_dense, k3_rmsnorm_rows, k3_act_rows)
against fp64.  Every product is exact (an fp32 value enters as three bf16 terms whose sum is
exact) and sums are fp32, so the error is at most K 2^-24 of the sum of |products| for any
order, and in practice a few 2^-24 sqrt(K) of it; the bar is 2e-6 of that sum per element."""
from __future__ import annotations

import pytest
import torch

from k3hip import _blas, _lib
from k3hip import _torch as T

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _g(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


# token tiles 32 / 64 / 128 (/ 256 for bf16) and their remainders, weight tiles of 256 and
# their remainders, K of whole and part 64-steps, K split over blocks or not
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,K,Ns", [(1, 8, [8]), (2, 72, [5, 300]), (33, 1536, [256]), (64, 4104, [257]),
                                    (65, 512, [96, 512, 1, 128]), (129, 2048, [700]), (300, 1000, [1024, 256]),
                                    (1000, 1536, [512])])
def test_dense_matches_fp64(M, K, Ns, dtype):
    g = _g(M * 7 + K)
    a = torch.randn(M, K, device=DEV, generator=g).to(dtype)
    ws = [torch.randn(n, K, device=DEV, generator=g).to(torch.bfloat16) for n in Ns]
    outs = _blas.dense(a, ws)
    for w, o in zip(ws, outs):
        want = a.double() @ w.double().T
        mag = a.double().abs() @ w.double().abs().T
        worst = float(((o.double() - want).abs() / mag).max())
        assert worst <= 2e-6, (w.shape, worst)
    assert all(torch.equal(x, y) for x, y in zip(outs, _blas.dense(a, ws)))
    if len(ws) == 1:   # rows of a wider matrix, and an added matrix
        wide = torch.randn(M, K + 64, device=DEV, generator=g).to(dtype)
        wide[:, 64:] = a
        add = torch.randn_like(outs[0])
        got = _blas.dense(wide[:, 64:], ws, add)[0]
        assert torch.equal(got, outs[0] + add)


def test_dense_wide_range_and_non_finite():
    """Values over the whole fp32 range keep their products (no term overflows, no term is
    dropped), and a non-finite activation reaches its own token only."""
    g = _g(5)
    a = torch.randn(40, 256, device=DEV, generator=g) * torch.exp2(torch.randint(-60, 60, (40, 1), device=DEV, generator=g).float())
    a[3, 7], a[5, 9], a[6, 0] = float("inf"), float("nan"), 3.4e38
    w = torch.randn(64, 256, device=DEV, generator=g).to(torch.bfloat16)
    w[:, 7] = w[:, 7].abs() + 0.5
    w[:, 0] = 0.25
    o = _blas.dense(a, [w])[0]
    want = a.double() @ w.double().T
    ok = [i for i in range(40) if i not in (3, 5)]
    mag = a.double().abs() @ w.double().abs().T
    assert float(((o.double() - want).abs() / mag)[ok].max()) <= 2e-6
    assert torch.isposinf(o[3]).all() and torch.isnan(o[5]).all()


def test_rmsnorm_and_act_rows():
    g = _g(6)
    x = torch.randn(37, 1000, device=DEV, generator=g)[:, 4:]
    w = torch.rand(996, device=DEV, generator=g) + 0.5
    out = torch.empty(37, 996, device=DEV)
    _lib.call("k3_rmsnorm_rows", T.ptr(x), 1000, T.ptr(w), 1e-5, T.ptr(out), 37, 996, T.stream(x))
    xd = x.double()
    want = w.double() * xd * torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-5)
    assert float(((out.double() - want).abs() / want.abs().clamp_min(1e-6)).max()) <= 2e-6
    gt, u = torch.randn(2, 5, 68, device=DEV, generator=g) * 3
    o = torch.empty_like(gt)
    gd, ud = gt.double(), u.double()
    for kind, ref in ((_lib.K3_ACT_SILU, gd * torch.sigmoid(gd) * ud),
                      (_lib.K3_ACT_SITU, 2 * torch.tanh(gd / 2) * torch.sigmoid(gd) * 3 * torch.tanh(ud / 3))):
        _lib.call("k3_act_rows", T.ptr(gt), T.ptr(u), T.ptr(o), gt.numel(), kind, 2.0, 3.0, T.stream(gt))
        assert float((o.double() - ref).abs().max()) <= 2e-6 * float(ref.abs().max())


def test_dense_replay_after_larger_calls():
    """A captured call (K split over blocks, so with partial sums) keeps its own scratch: later
    larger calls and whatever takes freed memory leave its replays as the eager result."""
    g = _g(11)
    a = torch.randn(40, 4096, device=DEV, generator=g)
    w = torch.randn(512, 4096, device=DEV, generator=g).to(torch.bfloat16)
    big = torch.randn(200, 4096, device=DEV, generator=g)
    wide = torch.randn(2048, 4096, device=DEV, generator=g).to(torch.bfloat16)
    want = _blas.dense(a, [w])[0].clone()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        _blas.dense(a, [w])
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = _blas.dense(a, [w])[0]
    for i in range(3):
        with torch.cuda.stream(stream):
            _blas.dense(big[:100 + 50 * i], [wide])
            junk = [torch.full((n,), float("nan"), device=DEV) for n in (1 << 18, 1 << 20, 1 << 22)]
        torch.cuda.synchronize()
        del junk
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        assert torch.equal(_blas.dense(a, [w])[0], want)
