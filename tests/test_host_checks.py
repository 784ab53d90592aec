"""What the Python layer settles before anything is launched: shapes that the kernels take on
trust, and which path a call goes to.  No GPU: a call that should be refused is refused by the
shape check and not by the check for device tensors, which comes after it."""
from __future__ import annotations

from types import SimpleNamespace

import pytest
import torch

BF16 = torch.bfloat16


def _kda(H=2, hid=64, K=4, **other):
    from k3hip.kda import KDAAttention
    P, D = H * 128, 128
    z = lambda *s: torch.zeros(*s, dtype=BF16)  # noqa: E731
    w = {"q_proj.weight": z(P, hid), "k_proj.weight": z(P, hid), "v_proj.weight": z(P, hid), "g_proj.weight": z(P, hid),
         "o_proj.weight": z(hid, P), "q_conv1d.weight": z(P, 1, K), "k_conv1d.weight": z(P, 1, K),
         "v_conv1d.weight": z(P, 1, K), "f_a_proj.weight": z(D, hid), "f_b_proj.weight": z(P, D), "b_proj.weight": z(H, hid),
         "o_norm.weight": z(D), "A_log": torch.zeros(D), "dt_bias": torch.zeros(P)}
    w.update(other)
    cfg = SimpleNamespace(kda_num_heads=H, kda_head_dim=D, kda_conv_size=K, kda_gate_lower_bound=-5.0, rms_norm_eps=1e-5)
    return KDAAttention(cfg, w)


@pytest.mark.parametrize("name,shape", [("q_proj.weight", (128, 64)), ("v_proj.weight", (512, 64)), ("g_proj.weight", (255, 64)),
                                        ("f_b_proj.weight", (128, 128)), ("b_proj.weight", (1, 64)), ("dt_bias", (255,)),
                                        ("o_norm.weight", (64,))])
def test_kda_many_tokens_refuse_weights_of_other_widths(name, shape):
    with pytest.raises(ValueError, match=name.split(".")[0]):
        _kda(**{name: torch.zeros(*shape)}).prefill(torch.zeros(1, 3, 64))


def test_kda_many_tokens_refuse_more_heads_than_A_log_holds():
    with pytest.raises(ValueError, match="A_log"):
        _kda(H=129).prefill(torch.zeros(1, 2, 64))


def _layer(Is=64, hid=32, up=None, down=None):
    from k3hip.moe import MoEConfig, RoutedMoE
    z = lambda *s: torch.zeros(*s, dtype=BF16)  # noqa: E731
    w = {"gate.weight": z(4, hid), "shared_experts.gate_proj.weight": z(Is, hid),
         "shared_experts.up_proj.weight": z(*(up or (Is, hid))), "shared_experts.down_proj.weight": z(*(down or (hid, Is)))}
    return RoutedMoE(MoEConfig(hid, 32, 4, 2), 0, w, lambda *a: None)


def _no_device(monkeypatch, launches):
    """The layers' own checks without a GPU: device checks pass, launches are recorded and the
    matrix products are torch's."""
    from k3hip import _blas, _lib
    from k3hip import _torch as T
    monkeypatch.setattr(T, "require_device", lambda *ts: None)
    monkeypatch.setattr(T, "stream", lambda t: 0)
    monkeypatch.setattr(_blas, "weights_ok", lambda *ws: True)
    monkeypatch.setattr(_blas, "dense_ok", lambda a, *ws: all(w.shape[1] == a.shape[-1] for w in ws))
    monkeypatch.setattr(_blas, "_mm_bf16_f32", lambda a, w: a.float() @ w.float().t())
    monkeypatch.setattr(_lib, "call", lambda name, *a: launches.append(name))


@pytest.mark.parametrize("kw", [dict(up=(48, 32)), dict(down=(32, 48)), dict(down=(32, 72))])
def test_shared_expert_refuses_matrices_that_do_not_match(monkeypatch, kw):
    """gate and up of different rows, and a down projection of another width."""
    launches = []
    _no_device(monkeypatch, launches)
    with pytest.raises((ValueError, RuntimeError)):
        _layer(**kw).shared_forward(torch.zeros(3, 32, dtype=BF16))
    if "up" in kw:
        assert "k3_act_rows" not in launches
    assert launches.count("k3_dense") <= 1


@pytest.mark.parametrize("add", [torch.zeros(3, 15), torch.zeros(2, 16), torch.zeros(3, 16, dtype=BF16), torch.zeros(16)])
def test_dense_refuses_an_added_matrix_of_another_form(add):
    from k3hip import _blas
    with pytest.raises(ValueError, match="add"):
        _blas.dense(torch.zeros(3, 32), [torch.zeros(16, 32, dtype=BF16)], add)


def test_dense_reads_an_added_view_at_its_own_strides(monkeypatch):
    from k3hip import _blas, _lib
    _no_device(monkeypatch, [])
    seen = {}
    monkeypatch.setattr(_lib, "lib", lambda: SimpleNamespace(k3_dense_workspace_size=lambda *a: 0))
    monkeypatch.setattr(_lib, "call", lambda name, *a: seen.update(add=a[7]))
    add = torch.arange(3 * 40, dtype=torch.float32).view(3, 40)[:, 1:17]
    _blas.dense(torch.zeros(3, 32), [torch.zeros(16, 32, dtype=BF16)], add)
    assert seen["add"] != add.data_ptr() and seen["add"] % 16 == 0


def test_shared_forward_takes_the_hidden_state_alone():
    import inspect
    from k3hip.moe import LatentMoE, RoutedMoE
    for cls in (RoutedMoE, LatentMoE):
        assert list(inspect.signature(cls.shared_forward).parameters) == ["self", "x"]


@pytest.mark.parametrize("mod", ["mla", "moe"])
def test_norm_of_rows_refuses_a_weight_of_another_length(monkeypatch, mod):
    import importlib
    m = importlib.import_module(f"k3hip.{mod}")
    launches = []
    _no_device(monkeypatch, launches)
    x = torch.randn(3, 32)
    with pytest.raises(RuntimeError):
        m._rmsnorm_rows(x, torch.ones(16), 1e-5)
    assert torch.equal(m._rmsnorm_rows(x, torch.full((1,), 2.0), 1e-5), m._rmsnorm_rows(x, torch.ones(1), 1e-5) * 2)
    assert not launches
    m._rmsnorm_rows(x, torch.ones(32), 1e-5)
    assert launches == ["k3_rmsnorm_rows"]


def _mla_stub(heads=4):
    """MLAAttention's route, with tensors that claim to be on the device."""
    from k3hip.mla import MLAAttention
    attn = MLAAttention.__new__(MLAAttention)
    attn.cfg = SimpleNamespace(num_attention_heads=heads, kv_lora_rank=512, qk_rope_head_dim=64, qk_nope_head_dim=128,
                               v_head_dim=128, q_head_dim=192)
    attn.kv_b = _dev(torch.zeros(1, 1, dtype=BF16))
    return attn


class _Dev:
    """A CPU tensor that says it is a device tensor."""
    def __init__(self, t, requires_grad=False):
        self._t, self.is_cuda, self.requires_grad = t, True, requires_grad

    def __getattr__(self, name):
        return getattr(self._t, name)


def _dev(t, **kw):
    return _Dev(t, **kw)


def _rows(B, Tk, width, **kw):
    return _dev(torch.zeros(1, dtype=BF16).expand(B, Tk, width), **kw)


def test_mla_prompt_takes_one_sequence_of_one_length():
    attn = _mla_stub()
    q = _dev(torch.zeros(1).expand(1, 20, 4, 192))
    assert attn._expanded_ok(q, _rows(1, 20, 512), _rows(1, 20, 64))
    assert not attn._expanded_ok(q, _rows(2, 20, 512), _rows(2, 20, 64))   # a cache of two sequences
    assert not attn._expanded_ok(q, _rows(1, 20, 512), _rows(1, 19, 64))
    assert not attn._expanded_ok(_dev(torch.zeros(1).expand(2, 20, 4, 192)), _rows(1, 20, 512), _rows(1, 20, 64))


@pytest.mark.parametrize("mod", ["mla", "moe"])
def test_norm_of_rows_keeps_gradients_and_tangents(monkeypatch, mod):
    import importlib
    from torch.autograd import forward_ad
    m = importlib.import_module(f"k3hip.{mod}")
    launches = []
    _no_device(monkeypatch, launches)
    x, w = torch.randn(3, 32), torch.ones(32, requires_grad=True)
    m._rmsnorm_rows(x, w, 1e-5).sum().backward()
    assert w.grad is not None and torch.isfinite(w.grad).all()
    with forward_ad.dual_level():
        y = m._rmsnorm_rows(forward_ad.make_dual(x, torch.ones_like(x)), torch.ones(32), 1e-5)
        assert forward_ad.unpack_dual(y).tangent is not None
    assert not launches
    with torch.no_grad():
        m._rmsnorm_rows(x, w, 1e-5)
    assert launches == ["k3_rmsnorm_rows"]


def test_routes_leave_tracked_tensors_to_tensor_operations(monkeypatch):
    from torch.autograd import forward_ad
    from k3hip import _blas
    from k3hip import _torch as T
    attn = _mla_stub()
    q, lat, rot = _dev(torch.zeros(1).expand(1, 20, 4, 192)), _rows(1, 20, 512), _rows(1, 20, 64)
    for args in ((_dev(q._t, requires_grad=True), lat, rot), (q, _rows(1, 20, 512, requires_grad=True), rot),
                 (q, lat, _rows(1, 20, 64, requires_grad=True))):
        assert not attn._expanded_ok(*args)
    w, v = torch.zeros(16, 32, dtype=BF16), torch.zeros(16, 32, dtype=BF16)
    assert _blas.weights_ok(_dev(w)) and not _blas.weights_ok(_dev(w), _dev(v, requires_grad=True))
    a = torch.zeros(3, 32)
    with forward_ad.dual_level():
        dual = forward_ad.make_dual(a, torch.ones_like(a))
        assert T.tracked(None, dual) and not T.tracked(None, a)
    # a gradient of what the shared expert is added to
    _no_device(monkeypatch, [])
    monkeypatch.setattr(_blas, "dense", lambda a, ws, add=None: pytest.fail("a launch cuts the gradient")
                        if add is not None else [a @ w.float().t() for w in ws])
    add = torch.zeros(3, 32, requires_grad=True)
    y = _layer()._shared(torch.zeros(3, 32), add)
    assert y.requires_grad


# (heads, fp32 cache, cached positions, queries, masked form us, expanded form us)
MLA_FORMS = [(64, False, 256, 2, 218, 51), (64, False, 1024, 16, 220, 115), (64, False, 1024, 128, 336, 138),
             (64, False, 2048, 128, 531, 256), (64, False, 4096, 2, 224, 442), (64, False, 4096, 16, 247, 443),
             (64, False, 4096, 128, 939, 545), (64, False, 8192, 16, 443, 860), (64, False, 8192, 128, 1791, 1065),
             (64, False, 16384, 64, 1831, 2667), (64, False, 16384, 256, 7071, 3375), (64, False, 32768, 16, 1488, 8852),
             (64, False, 32768, 96, 5782, 11407), (64, False, 32768, 256, 15225, 11969), (64, False, 65536, 16, 2982, 31724),
             (64, False, 65536, 192, 32909, 44087), (64, True, 1024, 16, 203, 148), (64, True, 2048, 2, 203, 269),
             (64, True, 4096, 16, 236, 544), (64, True, 4096, 128, 935, 661), (64, True, 32768, 48, 3361, 10594),
             (16, False, 1024, 8, 214, 92), (16, False, 4096, 128, 336, 376), (16, False, 4096, 256, 558, 376),
             (16, False, 32768, 16, 539, 2205), (16, False, 32768, 256, 3647, 2974), (96, True, 918, 70, 448, 189),
             (96, False, 2904, 50, 614, 380), (64, True, 1637, 60, 344, 256), (8, False, 2784, 256, 318, 249),
             (64, False, 44255, 337, 35996, 29605), (48, False, 37410, 119, 8902, 10215), (96, False, 6172, 5, 437, 777)]


@pytest.mark.parametrize("heads,f32,Tk,T,masked,expanded", MLA_FORMS)
def test_mla_form_for_several_tokens_is_the_shorter_one(heads, f32, Tk, T, masked, expanded):
    """Both forms were measured at each of these; the rule takes the one that was shorter."""
    assert _mla_stub(heads)._expand_pays(T, Tk, f32) == (expanded < masked)


# (bf16 x, K, N, tokens, GEMV launches us, one matmul us)
MATVEC_FORMS = [(False, 7168, 300, 5, 9.0, 17.5), (False, 7168, 2048, 8, 23.1, 17.4), (False, 8192, 300, 8, 13.2, 22.0),
                (False, 8192, 300, 16, 25.3, 21.9), (False, 8192, 2048, 8, 24.3, 22.6), (False, 12288, 64, 5, 19.1, 30.1),
                (False, 12288, 1024, 5, 20.3, 31.2), (False, 12288, 2048, 5, 25.9, 31.4), (False, 12288, 4096, 5, 37.6, 32.7),
                (False, 12288, 300, 12, 45.6, 30.9), (False, 16384, 300, 5, 20.8, 39.5), (False, 16384, 1024, 8, 33.9, 40.4),
                (False, 16384, 1024, 12, 49.9, 40.2), (False, 16384, 4096, 8, 68.1, 41.1), (True, 8192, 1024, 8, 10.0, 11.5),
                (True, 8192, 1024, 12, 14.6, 11.6), (True, 8192, 2048, 5, 9.5, 11.6), (True, 12288, 64, 8, 12.2, 14.9),
                (True, 12288, 1024, 5, 10.5, 15.4), (True, 12288, 4096, 5, 21.7, 15.7), (True, 16384, 300, 8, 14.3, 18.8),
                (True, 16384, 1024, 12, 22.0, 19.1), (True, 16384, 2048, 8, 26.3, 19.2), (True, 24576, 300, 5, 23.2, 26.3)]


@pytest.mark.parametrize("bf,K,N,M,gemv,matmul", MATVEC_FORMS)
def test_matvec_form_for_a_few_tokens_is_the_shorter_one(bf, K, N, M, gemv, matmul):
    """Both forms were measured at each of these; k3_mxfp4_matvec takes the one that was shorter."""
    from k3hip import _lib
    n = _lib.lib().k3_mxfp4_matvec_launches(M, N, K, _lib.K3_BF16 if bf else _lib.K3_F32)
    assert (n > 1) == (gemv < matmul)


def test_matvec_launches_of_refused_sizes():
    from k3hip import _lib
    f = _lib.lib().k3_mxfp4_matvec_launches
    assert f(1, 64, 4096, 0) == 1 and f(3, 64, 16384, 0) == 3 and f(4, 64, 16384, 1) == 1
    assert [f(0, 64, 64, 0), f(1, 64, 48, 0), f(1, 64, 1 << 20, 0), f(1, 64, 64, 7)] == [0] * 4


def test_projections_of_bf16_tokens(monkeypatch):
    """Several matrices in one launch up to 1024 tokens; one matrix, and more tokens, on the library;
    fp32 tokens in one launch always; and operands that do not match never reach the launch."""
    from k3hip import _blas
    _no_device(monkeypatch, [])
    took = []
    monkeypatch.setattr(_blas, "dense", lambda a, ws, add=None: took.append("launch") or [a.float() @ w.float().t() for w in ws])
    monkeypatch.setattr(_blas, "mm_f32", lambda a, w: took.append("library") or a.float() @ w.float().t())
    w = [torch.zeros(16, 32, dtype=BF16)] * 2
    for M, dt, ws, want in ((2, BF16, w, ["launch"]), (1024, BF16, w, ["launch"]), (1025, BF16, w, ["library"] * 2),
                            (200, BF16, w[:1], ["library"]), (2000, torch.float32, w, ["launch"]),
                            (7, torch.float32, w[:1], ["launch"])):
        for checked in (False, True):
            took.clear()
            _blas.project(torch.zeros(M, 32, dtype=dt), ws, checked)
            assert took == want
    took.clear()
    with pytest.raises(RuntimeError):
        _blas.project(torch.zeros(3, 24), w, True)
    assert "launch" not in took


@pytest.mark.parametrize("B,T", [(1, 0), (2, 0), (0, 3)])
def test_kda_without_tokens_returns_the_state_and_windows(monkeypatch, B, T):
    launches = []
    _no_device(monkeypatch, launches)
    kda = _kda()
    x = torch.zeros(B, T, 64)
    out, state, conv = kda(x)
    assert out.shape == (B, T, 64) and state.shape == (B, 2, 128, 128) and not state.any()
    assert [tuple(c.shape) for c in conv] == [(B, 3, 256)] * 3 and not any(c.any() for c in conv)
    S, wins = torch.randn(B, 2, 128, 128), tuple(torch.randn(B, 3, 256) for _ in range(3))
    out, state, conv = kda(x, S, wins)
    assert state is S and all(torch.equal(a, b) and a.dtype == torch.float32 for a, b in zip(conv, wins))
    assert not launches


def test_sizes_beyond_a_launch_stay_where_they_ran(monkeypatch):
    """More rows, wider rows or wider pitches than the launches take go the way they went before."""
    from k3hip import _blas, _lib, mla
    z = lambda *s, dt=torch.float32: _dev(torch.zeros((1,) * len(s), dtype=dt).expand(*s))  # noqa: E731
    w = _dev(torch.zeros(16, 8, dtype=BF16))
    assert _blas.dense_ok(z(1 << 24, 8), w) and not _blas.dense_ok(z((1 << 24) + 1, 8), w)
    wide = _dev(torch.zeros(1, (1 << 20) + 8, dtype=BF16))
    assert not _blas.weights_ok(wide) and not _blas.dense_ok(z(2, (1 << 20) + 8), wide)
    attn = _mla_stub()
    for heads, Tk, ok in ((4, 1 << 24, True), (4, (1 << 24) + 1, False), (4097, 64, False)):
        attn.cfg.num_attention_heads = heads
        assert attn._expanded_ok(z(1, 20, heads, 192), _rows(1, Tk, 512), _rows(1, Tk, 64)) == ok
    launches = _lib.lib().k3_mxfp4_matvec_launches
    assert launches(5, 1 << 26, 32, 0) == 1 and launches(5, 1 << 28, 32, 0) == 2
    launched = []
    _no_device(monkeypatch, launched)
    x = z((1 << 24) + 1, 4)._t
    monkeypatch.setattr(mla, "_rmsnorm", lambda *a: "tensor operations")
    assert mla._rmsnorm_rows(x, torch.ones(4), 1e-5) == "tensor operations" and not launched


def test_dense_copies_rows_of_a_pitch_it_does_not_take(monkeypatch):
    from k3hip import _blas, _lib
    _no_device(monkeypatch, [])
    seen = {}
    monkeypatch.setattr(_lib, "lib", lambda: SimpleNamespace(k3_dense_workspace_size=lambda *a: 0))
    monkeypatch.setattr(_lib, "call", lambda name, *a: seen.update(ptr=a[0], lda=a[2]))
    a = torch.zeros(3, (1 << 20) + 64)[:, :32]
    _blas.dense(a, [torch.zeros(16, 32, dtype=BF16)])
    assert seen["lda"] == 32 and seen["ptr"] != a.data_ptr()


def test_grouped_prompts_do_not_share_scratch(monkeypatch):
    """Every prompt through the grouped experts brings scratch of its own (a captured graph and a later
    call, or two threads on one stream, would meet in a kept buffer)."""
    from k3hip import _lib, _workspace, moe
    seen = []
    _no_device(monkeypatch, [])
    monkeypatch.setattr(_lib, "call", lambda name, *a: seen.append((name, a[-3])))
    monkeypatch.setattr(_workspace, "get", lambda *a: pytest.fail("a kept buffer"))
    x, idx, w = torch.zeros(9, 64), torch.zeros(9, 2, dtype=torch.int64), torch.zeros(9, 2)
    moe.moe_grouped_ffn(x, idx, w, torch.zeros(4, 6, dtype=torch.int64), 64, validate=False)
    assert [n for n, _ in seen] == ["k3_moe_grouped_ffn"] and seen[0][1]


@pytest.fixture
def workspaces(monkeypatch):
    """k3hip._workspace on the host: one stream, and a capture that the test opens and closes."""
    from k3hip import _lib, _workspace
    from k3hip import _torch as T
    state = SimpleNamespace(capture=0, get=lambda n, tag="t": _workspace.get(torch.device("cpu"), n, tag), mod=_workspace)
    monkeypatch.setattr(T, "stream_of", lambda device: 7)
    monkeypatch.setattr(_lib, "lib", lambda: SimpleNamespace(k3_stream_capture_id=lambda stream: state.capture))
    for name in ("_cache", "_captured", "_outgrown"):
        monkeypatch.setattr(_workspace, name, type(getattr(_workspace, name, {}))())
    return state


def test_an_outgrown_workspace_stays(workspaces):
    """A captured graph may go on writing it.  All outgrown ones together are smaller than the one in use."""
    import weakref
    sizes = [5000, 9000, 9001, 30000, 200000]
    seen = [weakref.ref(workspaces.get(n)) for n in sizes]
    assert all(r() is not None for r in seen)
    kept = workspaces.mod._outgrown
    assert sum(b.numel() for b in kept) < workspaces.get(1).numel() and not workspaces.get(1).any()
    del kept
    workspaces.mod.clear()
    assert all(r() is None for r in seen)


def test_a_workspace_made_in_a_capture_is_that_captures_own(workspaces):
    workspaces.capture = 3
    a = workspaces.get(5000)
    assert workspaces.get(4000).data_ptr() == a.data_ptr() and not a[:4096].any()
    workspaces.capture = 4                  # another graph, which may replay before the first ever does
    b = workspaces.get(5000)
    workspaces.capture = 0                  # an eager call, the same
    c = workspaces.get(5000)
    assert len({a.data_ptr(), b.data_ptr(), c.data_ptr()}) == 3 and not c.any()
    workspaces.capture = 5                  # a buffer in use outside is taken by captures too, as it is
    assert workspaces.get(5000).data_ptr() == c.data_ptr()


def test_threads_on_one_stream_have_workspaces_of_their_own(workspaces):
    import threading
    got, both = {}, threading.Barrier(2)

    def work(i):
        got[i] = workspaces.get(5000)
        both.wait()                        # both threads are alive: their numbers differ
        assert workspaces.get(5000).data_ptr() == got[i].data_ptr()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert got[0].data_ptr() != got[1].data_ptr()


def test_import_without_the_raw_stream_getter(monkeypatch):
    """A torch that lacks it imports the package and takes the handle from its Stream objects."""
    import importlib.util
    from k3hip import _torch as T
    monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device: SimpleNamespace(cuda_stream=1000 + device))
    spec = importlib.util.spec_from_file_location("k3hip._torch_again", T.__file__)
    again = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(again)
    assert again.stream_of(torch.device("cuda", 3)) == 1003
    assert again.stream(SimpleNamespace(get_device=lambda: 2)) == 1002
