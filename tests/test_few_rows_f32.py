"""fp32 products of one to eight rows against float64, at remainders of every dimension, and the calls that stay with the
library."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L

pytestmark = pytest.mark.gpu


def operands(m, n, k):
    g = torch.Generator().manual_seed(m + n * 3 + k)
    return torch.randn(m, k, generator=g).cuda(), torch.randn(n, k, generator=g).cuda()


def close(y, x, w):
    """A sum is a chain of 4 ceil(K / 1024) terms, six exchanges in the wave and two over the waves (the library's is taken
    to be no longer than K / 16 + 16)."""
    k = x.shape[1]
    bound = (4 * -(-k // 1024) + 9 + (0 if L._few_f32_ok(x, w) else k / 16 + 16)) * 2.0 ** -24
    assert y.dtype == torch.float32 and y.shape == (x.shape[0], w.shape[0])
    err = (y.double() - x.double() @ w.double().T).abs()
    assert bool((err <= bound * (x.double().abs() @ w.double().abs().T)).all())


@pytest.mark.parametrize("n,k", [(1, 4), (3, 8), (5, 1020), (257, 1024), (130, 1028), (64, 2052), (2048, 768), (8191, 260),
                                 (8192, 64), (8195, 132)])
def test_rows(n, k):
    x, w = operands(9, n, k)
    most = 8 if n < 8192 else 5
    first = L.linear(x[:1], w)
    for m in range(1, 10):
        assert L._few_f32_ok(x[:m], w) == (m <= most)
        y = L.linear(x[:m], w)
        close(y, x[:m], w)
        if m <= most:       # a row's bits do not depend on its neighbours
            assert torch.equal(y[:1], first)
    for f in (L.proj, L.proj_f32out):
        assert torch.equal(f(x[:2], w), L.linear(x[:2], w))


def test_other_layouts():
    x, w = operands(4, 96, 256)
    wide = torch.randn(4, 300, device="cuda")
    assert L._few_f32_ok(wide[:, :256], w) and L._few_f32_ok(wide[:, 4:260], w)
    for a, b in ((wide[:, :256], w), (wide[:, 4:260], w), (wide[:, 1:257], w), (x.T.contiguous().T, w),
                 (x[:1].expand(4, 256), w), (x, w.T.contiguous().T), (x[:, :254], w[:, :254].contiguous())):
        close(L.linear(a, b), a, b)
    for a, b in ((wide[:, 1:257], w), (x[:1].expand(4, 256), w), (x, w.T.contiguous().T), (x.bfloat16(), w), (x[:0], w),
                 (x[:, :254], w[:, :254].contiguous())):
        assert not L._few_f32_ok(a, b)
    assert L.linear(x[:0], w).shape == (0, 96)
    v = w.clone().requires_grad_()
    L.linear(x, v).sum().backward()
    assert torch.allclose(v.grad, x.sum(0).expand(96, 256), atol=1e-5)
    out = torch.empty(4, 96, device="cuda")
    assert L.linear(x, w, out) is out


def test_infinities_stay_in_their_row():
    x, w = operands(3, 40, 512)
    x[1, 7] = float("inf")
    y = L.linear(x, w)
    assert torch.isfinite(y[[0, 2]]).all() and torch.isinf(y[1]).all()


@pytest.mark.parametrize("n,k", [(1, 4), (3, 8), (127, 1028), (1024, 2048), (4095, 260), (4096, 64)])
def test_gated_unit_is_product_and_pass(n, k):
    """The products' sums and the pass's arithmetic: the same bits, also where a sum is not finite."""
    x, w = operands(8, 2 * n, k)
    w *= k ** -0.5
    w[n - 1, 0] = float("nan")
    w[2 * n - 1, k - 1] = float("inf")
    most = 8 if 2 * n < 8192 else 5
    for m in range(1, most + 1):
        want = L.glu_clamp(L.linear(x[:m], w), 1.0, float("inf"), 0.0)
        got = L.glu_proj(x[:m], w)
        assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0), want.nan_to_num(7.0, 8.0, 9.0))
