"""An attention's input product of many rows with its preparation (csrc/kernels/gemm_prep.hip) against 64 bits: every size of tiles, rows
that end within a tile and within a group of eight, pages that rows enter anywhere, slots without a place; and its rule."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops import seq_ops as S
from k8s_llm_rca_amd.ops._lib import lib, ptr, stream_ptr

BF = torch.bfloat16


def test_plan():
    assert L.prep_plan(4096, 2560, 2048) == 6 and L.prep_plan(3517, 2560, 2048) == 5 and L.prep_plan(16384, 2560, 2048) == 8
    assert L.prep_plan(1280, 2560, 2048) == 4 and L.prep_plan(24730, 8736, 2048) == 8
    for bad in ((1279, 8736, 2048), (4096, 2560, 1000), (4096, 2560, 512), (4096, 2560, 16384), (1300, 1280, 2048)):
        assert L.prep_plan(*bad) is None


def test_plan_of_long_k():
    """Product and pass stay apart where the library has a wave that is not full the quicker: sizes timed on both sides."""
    def took(m, n, k, prepared):
        return L.prep_plan(m, n, k, prepared) is not None
    for n, k, prepared, line in ((2576, 2048, 2560, 1280), (2576, 3072, 2560, 1400), (2576, 4096, 2560, 1800), (2576, 6144, 2560, 2048),
                                 (2560, 8192, 2560, 2048), (2048, 2048, 1536, 2048), (2048, 4096, 1536, 2600), (8736, 8192, 2560, 1280)):
        for rows in (1280, 1400, 1536, 1800, 2048, 2600, 3517):
            assert took(rows, n, k, prepared) == (rows >= line), (rows, n, k)


def oracle(h, w, bias, H, G, D, NV, cs, rot, norm, qw, kw, eps, lam, vo):
    x = h.double() @ w.double().T
    n = (H + G) * D + NV
    rest, x = x[:, n:], x[:, :n] + (bias.double() if bias is not None else 0)
    qk, v = x[:, :(H + G) * D].reshape(len(x), H + G, D).clone(), x[:, (H + G) * D:]
    if rot:
        a, b = qk[..., :rot // 2].clone(), qk[..., rot // 2:rot].clone()
        co, si = cs[:, None, :rot // 2].double(), cs[:, None, rot // 2:].double()
        qk[..., :rot // 2], qk[..., rot // 2:rot] = a * co - b * si, b * co + a * si
    if norm:
        qk = qk / torch.sqrt((qk * qk).mean(-1, keepdim=True) + eps)
    q, k = qk[:, :H] * (qw.double() if qw is not None else 1), qk[:, H:] * (kw.double() if kw is not None else 1)
    return q.flatten(1), k.flatten(1), v, (1 - lam) * v + lam * vo.double() if vo is not None else v, rest


def close(got, want, rel):
    # fp32 sums of k products of size k^(-1/2), through rotation, norm and weights of up to four; bf16's half unit
    assert bool(((got.double() - want).abs() <= rel * want.abs() + 1e-4).all()), float((got.double() - want).abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("f", [4, 5, 6, 8])
@pytest.mark.parametrize("M,H,G,D,NV,K,over,rot,norm,extras", [
    (257, 4, 2, 128, 256, 192, 0, 128, 1, False), (300, 2, 2, 128, 512, 128, 16, 0, 1, True), (70, 4, 4, 64, 256, 64, 260, 64, 1, True),
    (129, 8, 4, 64, 256, 320, 4, 16, 0, False), (1, 2, 2, 128, 256, 128, 300, 64, 1, True), (531, 4, 2, 128, 256, 256, 36, 8, 1, True)])
def test_against_64_bits(f, M, H, G, D, NV, K, over, rot, norm, extras):
    g = torch.Generator().manual_seed(M + K)
    BS, n = 64, (H + G) * D + NV
    h = torch.randn(M, K + 8, generator=g).to(BF).cuda()[:, :K]
    w = (torch.randn(n + over, K, generator=g) * K ** -0.5).to(BF).cuda()
    cs = torch.randn(M, rot, generator=g).cuda() if rot else None
    bias, qw, kw, vo = ((torch.randn(*s, generator=g).cuda() if extras else None) for s in ((n,), (D,), (D,), (M, NV)))
    keep = torch.full((M, NV), float("nan"), device="cuda") if extras else None
    # sequences that enter their pages anywhere, and rows without a place
    pages = M // 16 + 4
    slots, at = [], 5
    for r in range(M):
        if r % 97 == 40:
            at = (at // BS + 1) * BS + r % 7
        slots.append(-1 if r % 61 == 13 else at)
        at += 1
    assert max(slots) < pages * BS
    sl = torch.tensor(slots, dtype=torch.int32, device="cuda")
    kc, vt, vc = (torch.full(s, 7.0, device="cuda", dtype=BF) for s in ((pages, BS, G * D), (pages, NV, BS), (pages, BS, NV)))
    q, rest = torch.empty(M, H * D, device="cuda", dtype=BF), torch.full((M + 1, max(over, 4)), float("nan"), device="cuda")
    assert lib().k8s_gemm_prep(ptr(h), h.stride(0), ptr(w), M, n + over, K, f, ptr(bias), ptr(cs), rot, norm, ptr(qw), ptr(kw), 1e-5, 0.3,
                               ptr(vo), ptr(keep), ptr(sl), ptr(q), ptr(kc), ptr(vt), ptr(vc) if extras else 0, BS, H * D, G * D, NV, D,
                               ptr(rest), rest.shape[1], stream_ptr(q)) == 0
    wq, wk, wv, wmix, wrest = oracle(h, w, bias, H, G, D, NV, cs, rot, norm, qw, kw, 1e-5, 0.3, vo)
    rel = 2.0 ** -8 * 1.01
    close(q, wq, rel)
    ok = sl >= 0
    where = sl[ok].long()
    for pool, want in ((kc.view(-1, G * D), wk), (vt.transpose(1, 2).reshape(-1, NV), wmix), (vc.view(-1, NV), wmix)):
        if pool.data_ptr() == vc.data_ptr() and not extras:
            assert bool((pool == 7).all())
            continue
        close(pool[where], want[ok], rel)
        other = torch.ones(pool.shape[0], dtype=torch.bool, device="cuda")
        other[where] = False
        assert bool((pool[other] == 7).all())               # nothing else was written
    if keep is not None:
        close(keep, wv, 1e-6)
    if over:
        close(rest[:M, :over], wrest, 1e-6)
    assert bool(torch.isnan(rest[M]).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [(1500,), (700, 900, 1), (4097,)])
@pytest.mark.parametrize("D,over,pairs", [(128, 16, False), (64, 0, False), (128, 0, True)])
def test_entry_point(rows, D, over, pairs):
    """What it gives is what product and pass give, to a unit of bf16, and nothing where it does not fit."""
    H, G, V, K, BS, T = 1024 // D, 256 // D, D, 1024, 64, sum(rows)
    g = torch.Generator().manual_seed(T + D)
    h, w = torch.randn(T, K, generator=g).to(BF).cuda(), (torch.randn((H + 2 * G) * D + over, K, generator=g) / 32).to(BF).cuda()
    bias = torch.randn((H + 2 * G) * D, generator=g).cuda()
    pos = torch.cat([torch.arange(r) for r in rows]).to(torch.int32).cuda()
    slots = torch.arange(T, dtype=torch.int32, device="cuda") + 3
    rope = S.make_rope(D, 1e4, "cuda", pairs=pairs)
    cs = S.rope_table(pos, rope)
    row0 = [sum(rows[:i]) for i in range(len(rows) + 1)]

    class Seg:
        n_seg = len(rows)
    assert row0[-1] == T
    out = []
    for fused in (True, False):
        kc, vt = (torch.zeros(T // BS + 2, *s, device="cuda", dtype=BF) for s in ((BS, G * D), (G * V, BS)))
        kw = dict(norm=True, eps=1e-5, rope=rope, rope_cs=cs)
        if fused:
            made = S.proj_prep(h, w, bias, H, G, D, V, slots, kc, None, vt, Seg, **kw)
            if pairs or L.prep_plan(T, w.shape[0], K) is None:
                assert made is None
                return
            q, rest = made
            assert (rest is None) == (over == 0)
        else:
            x = L.proj_f32out(h, w)
            q, rest = S.attn_prep(x[:, :bias.numel()], bias, H, G, D, V, pos, slots, kc, None, BF, vt=vt, **kw), x[:, bias.numel():]
        out.append((q, kc, vt) + ((rest,) if over else ()))
    for a, b in zip(*out):
        assert float((a.float() - b.float()).abs().max()) <= 2.0 ** -7 * float(b.float().abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,D,over,extras", [((700, 1, 599), 128, 0, False), ((1250, 50), 128, 16, True), ((1900, 900, 700), 128, 16, True),
                                                ((3500,), 64, 0, True), ((2000, 1, 1499), 64, 512, False)])
def test_entry_point_in_one_launch(rows, D, over, extras):
    """Sizes that the rule gives to it, every sequence on pages of its own: what it gives against 64 bits, entry by entry, and against
    product and pass of the same rows."""
    H, G, V, K, BS, T = 2048 // D, 256 // D, D, 2048, 64, sum(rows)
    NV, n = G * V, (H + 2 * G) * D
    assert L.prep_plan(T, n + over, K, n) is not None
    g = torch.Generator().manual_seed(T + D + over)
    h, w = torch.randn(T, K, generator=g).to(BF).cuda(), (torch.randn(n + over, K, generator=g) * K ** -0.5).to(BF).cuda()
    bias, qw, kw, vo = ((torch.randn(*s, generator=g).cuda() if extras else None) for s in ((n,), (D,), (D,), (T, NV)))
    page0 = [sum(-(-r // BS) + 1 for r in rows[:i]) for i in range(len(rows) + 1)]
    pages = page0[-1]
    slots = torch.cat([torch.arange(r) + p * BS for r, p in zip(rows, page0)]).to(torch.int32).cuda()
    pos = torch.cat([torch.arange(r) for r in rows]).to(torch.int32).cuda()
    rope = None if extras and D == 128 else S.make_rope(D // 2, 1e4, "cuda")
    cs = S.rope_table(pos, rope) if rope is not None else None

    class Seg:
        n_seg = len(rows)
    out = []
    for fused in (True, False):
        kc, vt, vc = (torch.full(s, 7.0, device="cuda", dtype=BF) for s in ((pages, BS, G * D), (pages, NV, BS), (pages, BS, NV)))
        keep = torch.empty(T, NV, device="cuda") if extras else None
        prep = dict(norm=True, q_w=qw, k_w=kw, eps=1e-5, lam=0.3, v_other=vo, v_keep=keep, rope=rope, rope_cs=cs)
        if fused:
            made = S.proj_prep(h, w, bias, H, G, D, V, slots, kc, vc, vt, Seg, **prep)
            assert made is not None and (made[1] is None) == (over == 0)
            q, rest = made
        else:
            x = L.proj_f32out(h, w)
            q, rest = S.attn_prep(x[:, :n], bias, H, G, D, V, pos, slots, kc, vc, BF, vt=vt, **prep), x[:, n:]
        out.append((q, kc.view(-1, G * D)[slots.long()], vt.transpose(1, 2).reshape(-1, NV)[slots.long()], vc.view(-1, NV)[slots.long()],
                    keep, rest if over else None))
        written = torch.zeros(pages * BS, dtype=torch.bool, device="cuda")
        written[slots.long()] = True
        assert all(bool((t[~written] == 7).all()) for t in (kc.view(-1, G * D), vt.transpose(1, 2).reshape(-1, NV), vc.view(-1, NV)))
    wq, wk, wv, wmix, wrest = oracle(h, w, bias, H, G, D, NV, cs, rope.dims if rope is not None else 0, True, qw, kw, 1e-5, 0.3, vo)
    rel = 2.0 ** -8 * 1.01
    for got in out:
        for t, want, r in zip(got, (wq, wk, wmix, wmix, wv, wrest), (rel, rel, rel, rel, 1e-6, 1e-6)):
            if t is not None:
                close(t, want, r)
    for a, b in zip(*out):
        if a is not None:                                # two roundings of sums in different orders: a unit of bf16 apart
            assert bool(((a.float() - b.float()).abs() <= 2.0 ** -7 * b.float().abs() + 2e-4).all())


@pytest.mark.gpu
def test_refused():
    z = torch.zeros(1 << 16, device="cuda", dtype=BF)
    f = torch.zeros(1 << 14, device="cuda")
    sl = torch.zeros(4, dtype=torch.int32, device="cuda")
    ok = [ptr(z), 64, ptr(z), 4, 768, 64, 4, 0, 0, 0, 1, 0, 0, 1e-5, 0.0, 0, 0, ptr(sl), ptr(z), ptr(z), ptr(z), 0, 64, 256, 256, 256, 64, 0,
          0, stream_ptr(z)]
    for at, bad in ((0, 0), (0, ptr(z) + 2), (1, 60), (1, 56), (2, 0), (3, 0), (4, 770), (4, 512), (4, 772), (5, 96), (6, 3), (6, 7), (7, ptr(f) + 4),
                    (9, 12), (9, 16), (9, 128), (10, 2), (17, 0), (18, 0), (19, 0), (20, 0), (22, 0), (23, 128), (24, 128), (25, 0), (26, 96),
                    (26, 32)):
        assert lib().k8s_gemm_prep(*ok[:at], bad, *ok[at + 1:]) != 0, (at, bad)


@pytest.mark.gpu
@pytest.mark.parametrize("stride,flat", [(0, False), (1024, False), (2048, True)])
def test_left_to_product_and_pass(stride, flat):
    """Rows that overlap, and another layer's values in another shape, are not taken: product and pass say what they say of them."""
    T, K, H, G, D, NV, BS = 1300, 2048, 16, 2, 128, 256, 64
    h = torch.zeros(T * stride + K, device="cuda", dtype=BF).as_strided((T, K), (stride, 1))
    w, vo = torch.zeros(2560, K, device="cuda", dtype=BF), torch.zeros(T, NV, device="cuda")
    kc, vt = (torch.zeros(T // BS + 1, *s, device="cuda", dtype=BF) for s in ((BS, G * D), (NV, BS)))
    slots = torch.arange(T, dtype=torch.int32, device="cuda")

    class Seg:
        n_seg = 1
    assert L.prep_plan(T, 2560, K, 2560) is not None
    args = (w, None, H, G, D, 128, slots, kc, None, vt, Seg)
    good = S.proj_prep(torch.zeros(T, K, device="cuda", dtype=BF), *args, norm=True, v_other=vo, lam=0.5)
    assert good is not None
    assert S.proj_prep(h, *args, norm=True, v_other=vo.view(-1) if flat else vo, lam=0.5) is None
