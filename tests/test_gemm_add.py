"""A prompt's products added to the fp32 residual with what reads it next (csrc/kernels/gemm_add.hip), against 64 bits: rows that
end within a tile, a half and a wave's share of it; K of fewer tiles than are staged; several columns' tiles; the rest behind whole
waves; and the gated product that divides its rows."""
import itertools

import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops import norm as NO
from k8s_llm_rca_amd.ops import row_step as R
from k8s_llm_rca_amd.ops._lib import check, lib, ptr, stream_ptr

BF = torch.bfloat16


def test_plan():
    for then, m, n, k in itertools.product((0, 1, 2), (512, 1000, 2600, 3517, 4096, 6143, 6144, 24730, 30001), (256, 1024, 2048, 3072, 5120),
                                           (1024, 2048, 8192, 14336)):
        plan = L.add_plan(m, n, k, then)
        if plan is None:
            continue
        assert plan[0][0] == 0 and plan[-1][1] == m and len(plan) <= 2
        for lo, hi, f in plan:
            assert lo < hi and (f in (4, 5, 6, 8) or f == 0 and hi - lo < 512)
        if len(plan) == 2:
            assert plan[0][1] == plan[1][0] and plan[0][2]
    # sizes on each side of the lines
    assert L.add_plan(4096, 2048, 2048, L.THEN_DYT) == ((0, 4096, 4),) and L.add_plan(4850, 2048, 8192, L.THEN_SCALED) == ((0, 4850, 5),)
    assert L.add_plan(24730, 2048, 8192, L.THEN_DYT) == ((0, 24576, 8), (24576, 24730, 0))
    assert L.add_plan(1000, 1024, 2048, L.THEN_DYT) is None and L.add_plan(2048, 2048, 8192, L.THEN_DYT) is None
    assert L.add_plan(16384, 2048, 2048, L.THEN_NOTHING) is None and L.add_plan(4096, 2048, 2048, L.THEN_NOTHING)
    for bad in ((4096, 2000, 2048), (4096, 2048, 1000), (4096, 2048, 512), (511, 2048, 2048), (4096, 8192, 2048)):
        assert L.add_plan(*bad, L.THEN_DYT) is None


def test_plan_cuts():
    """A second launch has to earn its start: never the same tiles twice, but at 4096 columns, where one launch would have every XCD at the
    same half of them, and of 256 rows with tanh, which gain by it."""
    for then, m, n, k in itertools.product((0, 1, 2), (700, 1234, 2600, 4630, 6143, 8192, 10000, 12288, 16384, 24730, 32768), range(256, 5121, 256),
                                           (1024, 2048, 4096, 8192)):
        plan = L.add_plan(m, n, k, then)
        if plan is not None and len(plan) == 2 and plan[0][2] == plan[1][2] and not (then == L.THEN_DYT and plan[0][2] == 8 and 65536 % n == 0):
            assert n == 4096 and -(-m // (32 * plan[0][2])) % 32 == 0 and -(-plan[0][1] // (32 * plan[0][2])) % 32, (m, n, k)
    for m, n, k, f in ((16384, 2048, 2048, 8), (16384, 2048, 8192, 8), (10000, 2048, 2048, 5), (32768, 2048, 2048, 8), (12288, 2048, 2048, 6),
                       (24576, 1024, 2048, 6), (16384, 5120, 4096, 8)):
        assert L.add_plan(m, n, k, L.THEN_SCALED) == ((0, m, f),)
        assert (L.add_plan(m, n, k, L.THEN_DYT) == ((0, m, f),)) == (f != 8 or n == 5120)
    assert L.add_plan(20000, 2048, 8192, L.THEN_DYT) == ((0, 16384, 8), (16384, 20000, 4))
    assert L.add_plan(16384, 4096, 2048, L.THEN_DYT) == ((0, 4096, 8), (4096, 16384, 8))
    assert L.add_plan(12215, 4096, 2048, L.THEN_SCALED) == ((0, 12215, 8),)


def test_plan_of_long_k():
    """Product and pass apart while few of a wave's tiles have a long K: sizes on both sides of the line (nearly all of them timed)."""
    for n, k, yes, no in ((2048, 4096, 2400, 2048), (2048, 6144, 2800, 2400), (2048, 8192, 2600, 2400),
                          (3072, 11008, 2400, 2048), (4096, 11008, 1684, 1300), (2048, 14336, 3300, 2800), (5120, 14336, 1300, 1100)):
        assert L.add_plan(yes, n, k, L.THEN_DYT) and L.add_plan(yes, n, k, L.THEN_SCALED)
        assert L.add_plan(no, n, k, L.THEN_DYT) is None and L.add_plan(no, n, k, L.THEN_NOTHING) is None, (no, n, k)
    assert L.add_plan(1300, 4096, 8192, L.THEN_DYT)
    assert L.add_plan(3517, 2048, 8192, L.THEN_NOTHING) and L.add_plan(3072, 3072, 14336, L.THEN_NOTHING)
    assert L.add_plan(2048, 3072, 14336, L.THEN_NOTHING) is None and L.add_plan(2048, 3072, 8192, L.THEN_NOTHING)


def rnd(*shape, dtype=torch.float32, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed + sum(shape))).to(dtype).cuda()


def oracle(x, a, w, scale, then, alpha, nw, nb, rms, again):
    y = a.double() @ w.double().T
    if rms is not None:
        ss, width, eps = rms
        y = y / torch.sqrt(ss.double().sum(1, keepdim=True) / width + eps)
    x = x.double() + scale * y
    if again is not None:
        ids, emb, es = again
        x = x + es * emb.double()[ids.long()]
    if then == L.THEN_DYT:
        return x, torch.tanh(alpha * x) * nw.double() + nb.double()
    return x, x * nw.double()


def compare(x, h, part, want, k, bound=None):
    wx, wh = want
    n = wx.shape[1]
    # fp32 sums of k products of size k^(-1/2) each, and the residual's own rounding
    bound = bound or 4e-6 * k ** 0.5 + 2e-6
    assert float((x.double() - wx).abs().max()) < bound
    if h is not None:
        # bf16 rounds to 2^-9 of the value; the residual's difference goes through the norm with a slope of at most 4 here
        assert bool(((h.double() - wh).abs() <= 2.0 ** -8 * wh.abs() + 4 * bound).all())
    if part is not None:
        sums = (wx * wx).view(wx.shape[0], n // 256, 256).sum(2)
        assert float(((part.double() - sums).abs() / sums).max()) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("f", [4, 5, 6, 8])
@pytest.mark.parametrize("n,k", [(256, 64), (256, 128), (512, 192), (768, 256), (2048, 1088)])
@pytest.mark.parametrize("then", [0, 1, 2])
def test_tiles(f, n, k, then):
    bm = 32 * f
    for m in (1, 15, bm // 2 - 1, bm // 2 + 1, bm - 1, bm, bm + 1, 9 * bm + 40):
        wide = 8 if m % 2 else 0                       # rows that lie apart
        a, w = rnd(m, k + wide, dtype=BF)[:, :k], (rnd(n, k, seed=1) * k ** -0.5).to(BF)
        x0, nw, nb = rnd(m + 3, n, seed=2), 1 + 0.1 * rnd(n, seed=3), 0.1 * rnd(n, seed=4)
        x, h, part = x0.clone(), torch.full((m + 3, n), 7.0, device="cuda", dtype=BF), torch.full((m + 3, n // 256), 7.0, device="cuda")
        extra = then != L.THEN_DYT and m % 2 == 1
        rms = (rnd(m, 5, seed=5) ** 2 + 0.5, 4.0, 1e-3) if extra else None
        again = (torch.arange(m, device="cuda", dtype=torch.int32) % 7, rnd(7, n, dtype=BF, seed=6), 0.25) if extra else None
        check(lib().k8s_gemm_add(ptr(a), k + wide, ptr(w), ptr(x), 0.75, ptr(rms[0]) if extra else 0, 5 if extra else 0, 4.0, 1e-3,
                                 ptr(again[0]) if extra else 0, ptr(again[1]) if extra else 0, 0.25, then, 0.6, ptr(nw) if then else 0,
                                 ptr(nb) if then == 1 else 0, ptr(h) if then else 0, ptr(part) if then == 2 else 0, m, n, k, f,
                                 stream_ptr(x)), "gemm_add")
        compare(x[:m], h[:m] if then else None, part[:m] if then == 2 else None,
                oracle(x0[:m], a, w, 0.75, then, 0.6, nw, nb, rms, again), k)
        assert torch.equal(x[m:], x0[m:]) and bool((h[m:] == 7).all()) and bool((part[m:] == 7).all())      # nothing behind the rows


@pytest.mark.gpu
@pytest.mark.parametrize("then", [0, 1, 2])
@pytest.mark.parametrize("plan", [((0, 300, 5),), ((0, 256, 8), (256, 300, 0)), ((0, 128, 4), (128, 300, 6))])
def test_parts(then, plan):
    """Row ranges by different tiles, and by a product and a pass of their own."""
    m, n, k = 300, 512, 1024
    a, w, x0 = rnd(m, k, dtype=BF), (rnd(n, k, seed=1) * k ** -0.5).to(BF), rnd(m, n, seed=2)
    nw, nb = 1 + 0.1 * rnd(n, seed=3), 0.1 * rnd(n, seed=4)
    rms = again = None
    if then != L.THEN_DYT:
        rms = (rnd(m, 16, seed=5) ** 2 + 0.5, 16.0, 1e-5)
        again = (torch.arange(m, device="cuda", dtype=torch.int32) % 11, rnd(11, n, dtype=BF, seed=6), 3.0)
    x = x0.clone()
    h, part = L.gemm_add(x, a, w, 1.0, plan, then, 0.6, nw if then else None, nb if then == 1 else None, rms, again)
    compare(x, h, part, oracle(x0, a, w, 1.0, then, 0.6, nw, nb, rms, again), k)


@pytest.mark.gpu
def test_refused():
    a, w, x = rnd(64, 128, dtype=BF), rnd(256, 128, dtype=BF), rnd(64, 256)
    nw, h, part = rnd(256), torch.empty(64, 256, device="cuda", dtype=BF), torch.empty(64, 1, device="cuda")

    def call(a=a, lda=128, x=ptr(x), rn=0, rs=0, then=2, nw=ptr(nw), nb=0, h=ptr(h), part=ptr(part), n=256, k=128, f=4):
        return lib().k8s_gemm_add(ptr(a) if isinstance(a, torch.Tensor) else a, lda, ptr(w), x, 1.0, rs, rn, 1.0, 0.0, 0, 0, 0.0, then,
                                  1.0, nw, nb, h, part, 64, n, k, f, stream_ptr(w))
    assert call() == 0
    for bad in (dict(a=ptr(a) + 2), dict(lda=132), dict(lda=64), dict(x=ptr(x) + 4), dict(rs=ptr(nw), rn=65), dict(rs=ptr(nw), rn=0),
                dict(then=3), dict(then=1), dict(nw=0), dict(h=0), dict(part=0), dict(n=128), dict(k=96), dict(f=7), dict(nw=ptr(nw) + 4)):
        assert call(**bad) != 0, bad


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(257, 128, 256), (300, 384, 1024), (2100, 2048, 768)])
def test_gated(m, n, k):
    """The gated product behind a residual that was left in parts, against its rows divided first."""
    x, nw = rnd(m, k), 1 + 0.1 * rnd(k, seed=1)
    w = (rnd(2 * n, k, seed=2) * k ** -0.5).to(BF)
    h = (x * nw).to(BF)
    part = (x * x).view(m, k // 256, 256).sum(2).contiguous()
    got = L.gemm_big_silu_scaled(h, w, part, 1e-5)
    y = (h.double() @ w.double().T) / torch.sqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5)
    g, u = (t.float().to(BF).double() for t in y.split(n, 1))
    want = g * torch.sigmoid(g) * u
    # gate, up and their product are rounded to bf16; a sum that falls to the other side of a tie moves by an ulp
    assert bool(((got.double() - want).abs() <= 3 * 2.0 ** -8 * want.abs() + 1e-4).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,quarters", [(4000, 2560, 64), (4096, 2816, 96)])
def test_gated_in_a_split_tail(m, n, quarters):
    """The same where the last wave's tiles go in four and in two, whose sums meet before they are divided: 64 and 96 of them."""
    k = 4096
    assert -(-m // 256) * (n // 128) % 256 == quarters
    x, nw = rnd(m, k), 1 + 0.1 * rnd(k, seed=1)
    w = (rnd(2 * n, k, seed=2) * k ** -0.5).to(BF)
    h = (x * nw).to(BF)
    part = (x * x).view(m, k // 256, 256).sum(2).contiguous()
    L.reserve_big_ws(x.device)                           # (the workspace is the next stream's that asks for it: this one)
    foreign = L.big_tail_foreign(x.device)
    for _ in range(2):
        got = L.gemm_big_silu_scaled(h, w, part, 1e-5)
    assert L.big_tail_foreign(x.device) == foreign
    g, u = ((h.double() @ w.double().T) / torch.sqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5)).split(n, 1)
    # gate, up and the result are rounded to bf16 (2^-8 each), the sums in fp32 before that; the gate's slope is at most 1.1
    half, s = 2.0 ** -8 * 1.01, 4e-6 * k ** 0.5
    act = torch.nn.functional.silu(g)
    tol = 1.1 * (half * g.abs() + s) * u.abs() + act.abs() * (half * u.abs() + s) + half * (act * u).abs() + s * s + 1e-6
    assert float(((got.double() - act * u).abs() / tol).max()) < 1


@pytest.mark.gpu
def test_sublayers():
    """What the models call, at rows that take it: the pass and its product apart are the oracle."""
    m, W, F = 2600, 2048, 2048
    one = torch.ones(1, device="cuda")
    a, w, x0 = rnd(m, F, dtype=BF), (rnd(W, F, seed=1) * F ** -0.5).to(BF), rnd(m, 1, W, seed=2)
    nw, nb, w13 = 1 + 0.1 * rnd(W, seed=3), 0.1 * rnd(W, seed=4), (rnd(16384, W, seed=5) * W ** -0.5).to(BF)
    assert L.add_plan(m, W, F, L.THEN_SCALED) and L.silu_scales(m, w13)
    x = x0.clone()
    h = R.add_product(x, a, w, one, one.view(1, 1), nw, 1e-5, BF, glu=w13)
    assert isinstance(h, R.Scaled) and R.residual(h, x) is x
    want = x0[:, 0].double() + a.double() @ w.double().T
    assert float((x[:, 0].double() - want).abs().max()) < 4e-6 * F ** 0.5 + 2e-6
    n = (want / torch.sqrt((want * want).mean(1, keepdim=True) + 1e-5) * nw.double())
    assert float((h.read().double() - n).norm() / n.norm()) < 3e-3
    got, ref = R.glu_proj(h, w13), L.glu_proj(n.to(BF), w13)
    assert float((got.double() - ref.double()).norm() / ref.double().norm()) < 6e-3      # two more roundings to bf16
    x2 = x0[:, 0].clone()
    d = R.dyt_product(x2, a, w, 0.5, a, w, 0.25, 0.7, nw, nb, BF)
    want = x0[:, 0].double() + 0.75 * (a.double() @ w.double().T)
    assert float((x2.double() - want).abs().max()) < 4e-6 * F ** 0.5 + 4e-6
    ref = torch.tanh(0.7 * want) * nw.double() + nb.double()
    assert float((d.double() - ref).norm() / ref.norm()) < 3e-3
    y = x0.clone()
    R.add_rest(y, a, w, one, one.view(1, 1), (rnd(m, 16, seed=6) ** 2, 16.0, 1e-5))
    z = x0.clone()
    NO.hyper_step(z, L.proj_planes(a, w), one, one.view(1, 1), rms=(rnd(m, 16, seed=6) ** 2, 16.0, 1e-5))
    assert float((y - z).abs().max()) < 4e-5
