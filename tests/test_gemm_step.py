"""A sublayer's last product with the residual's pass in its epilogue (csrc/kernels/gemm_step.hip) and the product that divides
by the root mean square afterwards (gemm_rows.hip, RowScale)."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops import norm as N
from k8s_llm_rca_amd.ops import row_step as R

BF = torch.bfloat16
gpu = pytest.mark.gpu
#: rows: one, both sides of the 8-row halves, the most
ROWS = [1, 2, 7, 8, 9, 16]
#: columns, K: the least, one of each number of loads that is a corner, an odd count of strips
SHAPES = [(128, 512), (1088, 1536), (2048, 2048), (2048, 4096)]


def test_rule():
    assert R.into_ok(8, 2048, 8192) and not R.into_ok(9, 2048, 8192) and R.into_ok(16, 2048, 4096)
    assert R.into_ok(16, 2048, 2048, True) and not R.into_ok(16, 2048, 4096, True)
    for m, n, k in ((0, 2048, 2048), (17, 2048, 2048), (1, 2044, 2048), (1, 2048, 2080), (1, 2048, 16384), (1, 512, 8192)):
        assert not R.into_ok(m, n, k)
    x, w = torch.ones(2, 1, 512), torch.ones(512, 512)
    one = torch.ones(1)
    h = R.add_product(x, torch.ones(2, 512), w, one, one.view(1, 1), torch.ones(512), 1e-5, torch.float32)   # on the CPU
    assert isinstance(h, torch.Tensor) and bool((x == 513.0).all())


def _close(got, want, k, scale=1.0):
    # fp32 sums of K products of size K^(-1/2) each, and what is added to them
    assert float((got.double() - want).abs().max()) < 4e-6 * (k ** 0.5 + scale)


def _rounded(got, want):
    # one rounding to bf16 of a value that may lie to either side of a boundary
    assert bool(((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())


def _rand(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=g).to(dtype).cuda()


@gpu
@pytest.mark.parametrize("m", ROWS)
@pytest.mark.parametrize("n,k", SHAPES)
def test_tanh_form(m, n, k):
    g = torch.Generator().manual_seed(m * k)
    a, w = _rand(g, m, k + 8, dtype=BF)[:, :k], (_rand(g, n, k) * k ** -0.5).to(BF)
    a2, w2 = _rand(g, m, k, dtype=BF), (_rand(g, n, k) * k ** -0.5).to(BF)
    x0, nw, nb = _rand(g, m, n) * 2, _rand(g, n), _rand(g, n)
    for two in (False, True):
        if not R.into_ok(m, n, k, two):
            continue
        x = x0.clone()
        h = R.dyt_product(x, a, w, 0.75, a2 if two else None, w2 if two else None, 0.5, 0.7, nw, nb, BF)
        want = x0.double() + 0.75 * (a.double() @ w.double().T) + (0.5 * (a2.double() @ w2.double().T) if two else 0)
        _close(x, want, k)
        _rounded(h, torch.tanh(0.7 * x.double()) * nw.double() + nb.double())


@gpu
@pytest.mark.parametrize("m", ROWS)
@pytest.mark.parametrize("n,k", [s for s in SHAPES if s[0] % 512 == 0 or s[0] == 1088])
@pytest.mark.parametrize("rn,add", [(0, False), (16, True), (64, False), (3, True)])
def test_norm_form_and_the_products_behind(m, n, k, rn, add):
    g = torch.Generator().manual_seed(m * k + rn)
    a, w = _rand(g, m, k, dtype=BF), (_rand(g, n, k) * k ** -0.5).to(BF)
    x0, nw, one = _rand(g, m, 1, n) * 2, 1 + 0.1 * _rand(g, n), torch.ones(1, device="cuda")
    ss = torch.rand(m, rn, generator=g).cuda() * 100 if rn else None
    ids, emb = torch.arange(m, dtype=torch.int32, device="cuda") % 5, _rand(g, 5, n, dtype=BF)
    x = x0.clone()
    h = R.add_product(x, a, w, one, one.view(1, 1), nw, 1e-5, BF, again=(ids, emb, 4.5) if add else None,
                      rms=(ss, 2048.0, 1e-5) if rn else None)
    y = a.double() @ w.double().T
    if rn:
        y = y / torch.sqrt(ss.double().sum(1, keepdim=True) / 2048.0 + 1e-5)
    want = x0[:, 0].double() + y + (4.5 * emb.double()[ids.long()] if add else 0)
    _close(x[:, 0], want, k, 10.0)
    assert isinstance(h, R.Scaled)
    _rounded(h.h, x[:, 0].double() * nw.double())
    full = h.read()
    assert torch.equal(full, N.hyper_read(x, None, nw, 1e-5, BF))
    idx = torch.tensor([m - 1, 0], device="cuda")
    _rounded(R.rows(h, idx).read(), full[idx].double())
    # what stands behind, against the same operand in 64 bits: sums, and results that are rounded once (SwiGLU: three times)
    r = 1.0 / torch.sqrt((x[:, 0].double() ** 2).mean(1, keepdim=True) + 1e-5)
    for cols in (2048, 1088):
        wn = (_rand(g, cols, n) * n ** -0.5).to(BF)
        exact = (h.h.double() @ wn.double().T) * r
        got = R.proj_f32out(h, wn), R.proj_planes(h, wn), R.proj(h, wn), R.glu_proj(h, wn)
        plans = [L.rows_plan(m, cols, n, L.ROWS_F32), L.rows_plan(m, cols, n, L.ROWS_F32, True), L.rows_plan(m, cols, n, L.ROWS_BF16),
                 L.rows_plan(m, cols // 2, n, L.ROWS_SILU)]
        assert [p is None for p in plans] == [n % 512 != 0] * 4
        if n % 512:                                         # a K that the dividing product does not take: normed rows, and the plain one
            for a, plain in zip(got, (L.proj_f32out, L.proj_planes, L.proj, L.glu_proj)):
                assert torch.equal(a, plain(full, wn))
            continue
        _close(got[0], exact, n)
        _close(got[1].sum(0), exact, n)
        _rounded(got[2], exact)
        gate, up = exact.split(cols // 2, 1)
        s = torch.nn.functional.silu(gate) * up
        assert bool(((got[3].double() - s).abs() <= 2.0 ** -6 * s.abs() + 2e-3).all())


@gpu
def test_what_is_refused():
    from k8s_llm_rca_amd.ops._lib import lib, ptr
    g = torch.Generator().manual_seed(1)
    a, w, x = _rand(g, 2, 512, dtype=BF), _rand(g, 512, 512, dtype=BF), _rand(g, 2, 512)
    nw, h, part = _rand(g, 512), _rand(g, 2, 512, dtype=BF), torch.empty(2, 64, device="cuda")
    ok = [ptr(a), 512, ptr(w), ptr(x), None, 0, 0.0, 0.0, None, None, 0.0, ptr(nw), ptr(h), ptr(part), 2, 512, 512, None]
    # (each is turned down before a launch: rows, columns, K, strides and addresses that the kernel does not take)
    for i, v in ((14, 17), (14, 0), (15, 508), (16, 520), (1, 500), (1, 256), (0, ptr(a) + 2), (2, ptr(w) + 2), (13, None), (11, None)):
        assert lib().k8s_gemm_step_rms(*(ok[:i] + [v] + ok[i + 1:])) != 0
