"""fp32 products of many rows as products of bf16 parts (csrc/kernels/gemm_split_f32.hip): against 64 bits, beside the library's
error, with infinities, NaN and numbers at both ends of the range."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops._lib import check, lib, ptr, stream_ptr

gpu = pytest.mark.gpu


def test_rule():
    assert L.split_plan(622, 16384, 2048, glu=True) is not None and L.split_plan(622, 2048, 8192, True)[1] > 1
    assert L.split_plan(166, 16384, 2048) is None and L.split_plan(333, 2048, 2048, True) is None
    for m, n, k in ((64, 16384, 2048), (5000, 16384, 2048), (622, 16382, 2048), (622, 16384, 2050), (622, 16384, 256)):
        assert L.split_plan(m, n, k) is None
    for m in range(128, 4097, 57):
        for n, k in ((2048, 8192), (2560, 2048), (1088, 4096), (8192, 512)):
            p = L.split_plan(m, n, k, True)
            assert p is None or p[0] in L.SPLIT_TILES and k % (32 * p[1]) == 0


def _split(x):
    m, k = x.shape
    p, f = torch.empty(3, m, k, dtype=torch.bfloat16, device=x.device), torch.empty(m, device=x.device)
    check(lib().k8s_split_rows_f32(ptr(x), x.stride(0), ptr(p), ptr(f), m, k, stream_ptr(x)), "split")
    return p, f


def _parts(x):
    return _split(x)[0]


def _product(x, w, mt, ranges):
    (m, k), n = x.shape, w.shape[0]
    y = torch.full((ranges, m, n), float("nan"), device=x.device)
    p, f = _split(x)
    check(lib().k8s_gemm_split_f32(ptr(p), ptr(f), ptr(w), ptr(y), m, n, k, mt, ranges, stream_ptr(x)), "product")
    return y


@gpu
@pytest.mark.parametrize("m", [1, 15, 64, 97, 160, 193])
@pytest.mark.parametrize("n,k", [(4, 32), (132, 64), (1100, 288), (128, 2048)])
@pytest.mark.parametrize("mt", L.SPLIT_TILES)
def test_product(m, n, k, mt):
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k + 4, generator=g).cuda()[:, :k], (torch.randn(n, k, generator=g) * k ** -0.5).cuda()
    x[0, 0], w[-1, -1] = 1e-30, 3e4
    want = x.double() @ w.double().T
    scale = x.double().abs() @ w.double().abs().T
    for ranges in (1, 2, 4):
        if k % (32 * ranges):
            continue
        y = _product(x, w, mt, ranges)
        # each sum of k products, in fp32: a share of the sum of their sizes
        assert bool(((y.double().sum(0) - want).abs() <= 2.0 ** -21 * scale).all())
    assert torch.equal(_parts(x).float().sum(0), x)                    # exactly three parts (1e-30 as well)


@gpu
@pytest.mark.parametrize("m,n,k", [(622, 1024, 2048), (333, 512, 8192)])
def test_no_further_off_than_the_library(m, n, k):
    g = torch.Generator().manual_seed(k)
    for heavy in (False, True):
        x, w = torch.randn(m, k, generator=g), torch.randn(n, k, generator=g) * k ** -0.5
        if heavy:                                                      # a few large entries a row
            x *= torch.exp(2.0 * torch.randn(m, k, generator=g))
        x, w = x.cuda(), w.cuda()
        want = x.double() @ w.double().T
        err = [float((y.double() - want).norm() / want.norm()) for y in (_product(x, w, 8, 1)[0], torch.nn.functional.linear(x, w))]
        assert err[0] <= err[1]


@gpu
def test_infinities_and_the_ends_of_the_range():
    g = torch.Generator().manual_seed(5)
    x, w = torch.randn(130, 96, generator=g).cuda(), torch.randn(140, 96, generator=g).cuda().abs()
    x[3, 7], x[4, 9], x[5, 11], x[6, 0], x[7] = float("inf"), float("-inf"), float("nan"), 3.4e38, 0.0
    w[9, 50], w[10, 0], w[11] = float("inf"), 3.402e38, 1e-3
    y, want = _product(x, w, 4, 1)[0], torch.nn.functional.linear(x, w)
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.isinf(), want.isinf())
    both = want.isinf()
    assert torch.equal(y[both], want[both])
    fin = want.isfinite()
    assert bool(((y - want)[fin].abs() <= 2e-5 * (want[fin].abs() + 30)).all())


@gpu
@pytest.mark.parametrize("sx,sw", [(-80, 0), (-112, 0), (-126, 0), (-140, 0), (0, -104), (0, -120), (0, -140), (-60, -60), (120, -118),
                                   (-118, 120), (100, -135), (-135, 100), (-40, 127), (127, -40)])
def test_small_and_large_numbers(sx, sw):
    """Rows of one size as exact as those of another, down to the least numbers there are; some rows only, too."""
    g = torch.Generator().manual_seed(9)
    x0, w0 = torch.rand(70, 512, generator=g) * 2 - 1, torch.rand(200, 512, generator=g) * 2 - 1
    for some in (False, True):
        x, w = (x0.double() * 2.0 ** sx).float(), (w0.double() * 2.0 ** sw).float()
        if some:
            x[::3], w[::5] = x0[::3], w0[::5]
        x, w = x.cuda(), w.cuda()
        want = x.double() @ w.double().T
        size = x.double().abs() @ w.double().abs().T
        for mt in L.SPLIT_TILES:
            for ranges in (1, 2):
                y = _product(x, w, mt, ranges).double().sum(0)
                # a share of the terms' sizes, and what fp32 cannot say below its least number;  terms that add up past its
                # largest number (2^128) may overflow on the way, as they do in a plain fp32 sum
                ok = ((y - want).abs() <= 2.0 ** -21 * size + 2.0 ** -148) | (size >= 2.0 ** 128)
                assert bool(ok.all()), (mt, ranges)
    (p, f), up = _split(x), 2.0 ** 64
    assert set(f.tolist()) <= {1.0, 1 / up} and torch.equal((p.double().sum(0) * f.double()[:, None]).float(), x)


@gpu
def test_numbers_that_are_not():
    """NaN where a number of either row is, without a sum of its own for each, and nowhere else."""
    g = torch.Generator().manual_seed(11)
    x, w = torch.randn(640, 2048, generator=g).cuda(), torch.randn(4096, 2048, generator=g).cuda() * 0.02
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]

    def us(x, w):
        best = 1e9
        for _ in range(4):
            ev[0].record()
            y = _product(x, w, 10, 1)
            ev[1].record()
            torch.cuda.synchronize()
            best = min(best, ev[0].elapsed_time(ev[1]) * 1e3)
        return best, y[0]
    plain, y0 = us(x, w)
    xn, wn = x.clone(), w.clone()
    xn[::2, 5], wn[1::2, 2047] = float("nan"), float("nan")
    for a, b in ((xn, w), (x, wn), (xn, wn)):
        t, y = us(a, b)
        bad = a.isnan().any(1)[:, None] | b.isnan().any(1)
        assert torch.equal(y.isnan(), bad) and torch.equal(y[~bad], y0[~bad])
        assert t < 8 * plain + 100
    # one infinity a row: a sum of its own each
    xi = x.clone()
    xi[7, 3], xi[639, 2000] = float("inf"), float("-inf")
    y = us(xi, w)[1]
    assert torch.equal(y[[7, 639]], torch.stack([xi[7, 3] * w[:, 3], xi[639, 2000] * w[:, 2000]]))


@gpu
def test_routes():
    """Where the rule takes it: the plain product, planes, and the gated unit; and what torch has to see stays with torch."""
    g = torch.Generator().manual_seed(7)
    x, w = torch.randn(640, 2048, generator=g).cuda(), (torch.randn(8192, 2048, generator=g) * 0.02).cuda()
    want = x.double() @ w.double().T
    assert L.split_plan(640, 8192, 2048) is not None
    assert float((L.linear(x, w).double() - want).norm() / want.norm()) < 1e-6
    y = L.proj_planes(x, w)
    assert float((y.double().sum(0) - want).norm() / want.norm()) < 1e-6
    gate, up = want.split(4096, 1)
    a = torch.nn.functional.silu(gate) * up
    assert float((L.glu_proj(x, w).double() - a).norm() / a.norm()) < 2e-6
    wg = w.clone().requires_grad_()
    L.linear(x, wg).sum().backward()
    assert wg.grad is not None
