"""Which calls the fused kernels take, and what they leave to the general ones: alignment, transforms of a call, sizes."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops import seq_ops as S
from k8s_llm_rca_amd.ops._lib import unwatched

BF = torch.bfloat16
gpu = pytest.mark.gpu


def meta(n, dev="cpu"):
    """``n`` sequences of one token each, past their first."""
    def i32(v):
        return torch.tensor(list(v), dtype=torch.int32, device=dev)
    return S.SegMeta(n, i32(range(n)), i32(range(n + 1)), i32([3] * n), i32(range(n)), i32([0] * n).view(n, 1),
                     list(range(n + 1)), [3] * n, list(range(n)), n_single=n)


def off(t, by=1):
    """The same numbers ``by`` entries behind an aligned address."""
    buf = torch.empty(t.numel() + by, dtype=t.dtype, device=t.device)
    v = buf[by:].view(t.shape)
    return v.copy_(t)


def test_states_off_16_bytes_are_not_read_by_16(monkeypatch):
    monkeypatch.setattr(S, "use_hip", lambda *t: True)
    x, gate, state, w = torch.zeros(2, 384), torch.zeros(2, 128), torch.zeros(2, 2, 64, 64), torch.zeros(128)
    assert S._step_ok(x, meta(2), 64, 64, state, gate, w)
    for bad in ((off(x), state, gate, w), (x, off(state), gate, w), (x, state, off(gate), w), (x, state, gate, off(w))):
        assert not S._step_ok(bad[0], meta(2), 64, 64, *bad[1:])


@gpu
def test_unaligned_states_and_pages_give_the_same():
    """Layers of one token each with states at an odd number, and pages of mixed values at an odd entry."""
    g, H, D, V = torch.Generator().manual_seed(0), 2, 64, 64

    def rnd(*shape):
        return torch.randn(*shape, generator=g).cuda()
    x, a, rate, db, beta = rnd(3, 4 * D + H * V), rnd(3, H * D), rnd(H).abs(), rnd(H * D), rnd(3, H)
    gate, w, state, xm, gb = rnd(3, H * V), rnd(V), rnd(3, H, D, V), rnd(3, 2 * H * (D + V) + 2 * H), rnd(2 * H)
    n, m, xd, dec, wd = rnd(3, H, D), rnd(3, H), rnd(3, H * (2 * D + 2 * V)), torch.rand(H).cuda(), rnd(H * V)
    got = []
    for move in (lambda t: t.clone(), off):
        st = [move(state) for _ in range(3)]
        o = [S.delta_layer(x, H, H, D, V, a, rate, db, beta, st[0], meta(3, "cuda"), gate, w, 1e-5, torch.float32),
             S.memory_layer(xm, H, D, V, gb, 9.0, st[1], n.clone(), m.clone(), meta(3, "cuda"), w, 1e-5, torch.float32)]
        y, rms = S.decay_layer(xd, H, D, V, dec, st[2], meta(3, "cuda"), xd[:, -H * V:], wd, 1e-5, torch.float32)
        if rms is not None:
            y = y * torch.rsqrt(rms[0].sum(1, keepdim=True) / rms[1] + rms[2])
        got.append(o + [y] + st)
    for p, q in zip(*got):
        assert float((p - q).abs().max()) < 1e-5 * float(q.abs().max())
    planes, other, slots = rnd(2, 3, 4 * D), rnd(3, D), torch.tensor([0, 40, 7], dtype=torch.int32).cuda()
    bias, pages = rnd(4 * D), []
    for move in (lambda t: t, off):
        kc, vc = move(torch.zeros(2, 32, D, dtype=BF).cuda()), torch.zeros(2, 32, D, dtype=BF).cuda()
        q = S.attn_prep(planes, bias, 2, 1, D, D, slots, slots, kc, vc, BF, norm=True, eps=1e-5, lam=0.5, v_other=other)
        pages.append([t.float() for t in (q, kc, vc)])
    for p, q in zip(*pages):
        assert float((p - q).abs().max()) <= 2.0 ** -7 * float(q.abs().max())


def test_head_products_that_do_not_fit_are_refused(monkeypatch):
    """Weights of other heads, other sizes or another device go to torch's batched product, as before there was a kernel; a
    launch by address would read past them."""
    monkeypatch.setattr(S, "use_hip", lambda *t: True)
    monkeypatch.setattr(S, "lib", lambda: pytest.fail("launched"))
    monkeypatch.setattr(S, "rotated_tail", lambda *a: None)
    x, out = torch.zeros(2, 4, 16), torch.zeros(2, 4, 64)
    assert S._small_heads(x, torch.zeros(4, 16, 64), 4, 16, out)
    for w in (torch.zeros(3, 16, 64), torch.zeros(4, 8, 64), torch.zeros(4, 24, 64), torch.zeros(8, 16, 64)):
        with pytest.raises(RuntimeError):
            S.head_proj(x, w, out)
        with pytest.raises(RuntimeError):
            S.latent_queries(x.view(2, 64), w, None, 4, 16, 0)
    with pytest.raises(RuntimeError):
        S.latent_queries(torch.zeros(2, 48), torch.zeros(4, 16, 64), None, 4, 16, 0)      # rows shorter than their heads
    assert not S._small_heads(x, torch.empty(4, 16, 64, device="meta"), 4, 16, out)
    assert not S.head_proj(x[:, :, :0], torch.zeros(4, 0, 64), torch.ones(2, 4, 64)).any()        # a sum of nothing
    assert S.head_proj(x, torch.zeros(4, 16, 0), out[:, :, :0]).numel() == 0
    for bad in (torch.zeros(1, 4, 64), torch.zeros(2, 4, 128)):
        S.head_proj(x, torch.zeros(4, 16, 64), bad)                                        # (torch sizes it anew)
    with pytest.raises(RuntimeError):
        S.head_proj(x, torch.zeros(4, 16, 64), torch.zeros(2, 4, 64, requires_grad=True))


def test_calls_that_something_watches():
    """Every way in which torch has more to do with an operator than its numbers."""
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    x, w, seen = torch.randn(2, 4), torch.nn.Parameter(torch.randn(3, 4)), []

    def look(*_):
        seen.append(unwatched(x))
        return x
    assert unwatched(x, w.detach()) and not unwatched(x, w)
    with torch.no_grad():
        assert unwatched(x, w)
    with forward_ad.dual_level():
        assert unwatched(x, w.detach()) and not unwatched(forward_ad.make_dual(x, x), w.detach())
    torch.func.vmap(look)(x)
    torch.func.jvp(look, (x,), (x,))
    torch.jit.trace(look, (x,), check_trace=False)
    torch.set_autocast_enabled("cuda", True)              # (torch.autocast is off without a device)
    look()
    torch.set_autocast_enabled("cuda", False)
    with TorchDispatchMode():
        look()
    with TorchFunctionMode():
        look()
    seen.append(unwatched(x.as_subclass(type("Sub", (torch.Tensor,), {}))))
    assert len(seen) >= 7 and not any(seen)


@gpu
def test_transforms_of_products_in_fp32():
    """Tangents, batched calls, traces and casts of fp32 products are torch's own, as of its operators."""
    from torch.autograd import forward_ad
    g = torch.Generator().manual_seed(1)
    x, w, t = (torch.randn(*s, generator=g).cuda() for s in ((4, 64), (96, 64), (4, 64)))
    q, uk, tq = (torch.randn(*s, generator=g).cuda() for s in ((4, 2 * 64), (2, 64, 64), (4, 2 * 64)))
    calls = [(lambda a: L.linear(a, w), lambda a: a @ w.T, x, t),
             (lambda a: S.latent_queries(a, uk, None, 2, 64, 0)[0],
              lambda a: torch.bmm(a.view(-1, 2, 64).transpose(0, 1), uk).transpose(0, 1), q, tq)]
    for f, ref, a, da in calls:
        with forward_ad.dual_level():
            d = forward_ad.unpack_dual(f(forward_ad.make_dual(a, da))).tangent
        assert d is not None and torch.allclose(d, ref(da), atol=1e-4)
        assert torch.allclose(torch.func.vmap(f)(torch.stack([a, da])), torch.stack([ref(a), ref(da)]), atol=1e-4)
        assert torch.allclose(torch.func.jvp(f, (a,), (da,))[1], ref(da), atol=1e-4)
        assert torch.allclose(torch.jit.trace(f, (a,), check_trace=False)(da), ref(da), atol=1e-4)
        with torch.autocast("cuda", dtype=BF):
            assert f(a).dtype == BF
        v = a.clone().requires_grad_()
        f(v).sum().backward()
        assert torch.allclose(v.grad, torch.autograd.grad(ref(v).sum(), v)[0], atol=1e-4)


def test_sizes_of_small_products():
    """The vector pipes take what they were measured faster at, over heads and sizes: (rows, heads, K, N) in bf16."""
    for case, fast in {(1, 16, 128, 256): 1, (64, 16, 128, 256): 1, (128, 16, 128, 256): 1, (128, 16, 256, 128): 1,
                       (16, 128, 128, 512): 0, (64, 32, 64, 512): 0, (1, 8, 1024, 1024): 0, (16, 4, 1024, 64): 0,
                       (64, 64, 512, 512): 0, (2, 16, 512, 512): 0, (64, 64, 128, 128): 0, (16, 64, 128, 128): 1,
                       (64, 64, 64, 64): 1, (128, 128, 64, 64): 0, (8, 16, 512, 128): 1, (16, 4, 512, 128): 0}.items():
        assert S._few_heads(*case, False) == bool(fast), case
    for case, fast in {(128, 16, 256, 256): 1, (16, 16, 512, 128): 1, (16, 128, 512, 128): 0, (128, 16, 256, 128): 1}.items():
        assert S._few_heads(*case, True) == bool(fast), case
    for case, fast in {(128, 64, 2048, 64, 2048): 1, (128, 128, 4096, 256, 4096): 0, (16, 1024, 8192, 1024, 8192): 0,
                       (64, 512, 2048, 512, 2048): 1, (16, 512, 2048, 512, 2048): 0, (1, 512, 2048, 512, 2048): 1, (32, 256, 8192, 256, 8192): 1}.items():
        assert S._few_ranks(*case) == bool(fast), case


def test_products_of_few_rows_by_shape():
    """Planes and narrow strips where they were measured faster: (rows, columns, K)."""
    for case, cut in {(1, 2048, 2048): 1, (1, 2048, 1024): 0, (16, 1024, 512): 0, (24, 2048, 512): 1, (24, 2048, 256): 0,
                      (1, 4096, 1024): 0, (8, 3072, 3072): 0, (16, 5120, 2048): 1, (17, 4096, 1024): 1, (8, 2560, 4096): 1, (8, 4096, 8192): 0,
                      (1, 2048, 8192): 1, (64, 2560, 1024): 1}.items():
        assert (L.plane_plan(*case)[1] > 1) == bool(cut), case
    assert L._skinny_f32(32, 8192, 1024) and not L._skinny_f32(32, 8192, 2048) and L._skinny_f32(17, 8192, 2048)
