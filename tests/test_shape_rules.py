"""Products whose kernel is chosen by shape (32-column strips, fused squared relu, fused SwiGLU) against float64, on both
sides of every border of their rules."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def operands(m, n, k):
    g = torch.Generator().manual_seed(m * 7 + n + k)
    x, w = torch.randn(m, k, generator=g).to(BF), (torch.randn(n, k, generator=g) * k ** -0.5).to(BF)
    return x.cuda(), w.cuda()


def close(y, want, ulps):
    """``ulps`` roundings to bf16 (2^-8 of the value each), and fp32 sums of a few units."""
    assert y.dtype == BF and y.shape == want.shape
    err = (y.double() - want).abs()
    assert bool((err <= ulps * 2.0 ** -8 * want.abs() + 1e-4).all()), float((err - ulps * 2.0 ** -8 * want.abs()).max())


ROWS = [1, 16, 17, 32, 33, 64, 65, 128, 129]


@pytest.mark.parametrize("n,k", [(8192, 2048), (8224, 2048), (32, 64), (96, 192), (4736, 2048), (100, 256), (512, 2112)])
@pytest.mark.parametrize("m", ROWS)
def test_proj_and_relu(m, n, k):
    x, w = operands(m, n, k)
    want = x.double() @ w.double().T
    close(L.proj(x, w), want, 1)
    # the unfused form rounds the product, squares it and rounds again: 2 + 1 roundings
    close(L.relu_sq_proj(x, w), want.clamp_min(0) ** 2, 3.1)


@pytest.mark.parametrize("i,k", [(8192, 2048), (4096, 2048), (4128, 2048), (3072, 2048), (2048, 2048), (16, 64), (640, 384),
                                 (48, 2112), (8192, 2112)])
@pytest.mark.parametrize("m", ROWS)
def test_glu_of_few_rows(m, i, k):
    x, w = operands(m, 2 * i, k)
    gu = x.double() @ w.double().T
    g, u = gu[:, :i], gu[:, i:]
    # gate, up and the result are rounded; a rounding of the gate moves silu by at most 1.1 of it and (1 + |g|) relative
    want = torch.nn.functional.silu(g) * u
    err = (L.glu_proj(x, w).double() - want).abs()
    bound = 2.0 ** -8 * (2.1 * want.abs() + 1.1 * (g * u).abs()) + 1e-4
    assert bool((err <= bound).all()), float((err - bound).max())


@pytest.mark.parametrize("m,n,k,fused", [(1345, 8192, 2048, False), (1345, 10240, 2048, True), (16384, 256, 256, True),
                                         (300, 1024, 384, False), (300, 1024, 640, False), (513, 768, 256, False),
                                         (5000, 768, 256, True), (4000, 1024, 512, False), (4200, 1024, 512, True)])
def test_prompt_rows(m, n, k, fused):
    assert L.big_fused(m, n, k, False) == fused == L.big_fused(m, n // 2, k, True) or k > 512
    assert L.big_fused(m, n, k, False) == fused
    x, w = operands(m, n, k)
    want = x.double() @ w.double().T
    close(L.relu_sq_proj(x, w), want.clamp_min(0) ** 2, 3.1)
    g, u = want[:, :n // 2], want[:, n // 2:]
    y = L.glu_proj(x, w).double()
    act = torch.nn.functional.silu(g) * u
    bound = 2.0 ** -8 * (2.1 * act.abs() + 1.1 * (g * u).abs()) + 1e-4
    assert bool(((y - act).abs() <= bound).all())


def test_values_that_are_not_finite():
    """A row with an infinity stays within its row and gives what the parts one by one give."""
    for m in (8, 40, 512):
        x, w = operands(m, 512, 256)
        x[m // 2, 3] = float("inf")
        u = L.linear(x, w)
        want = torch.relu(u.float()) ** 2
        y = L.relu_sq_proj(x, w).float()
        bad = m // 2
        assert torch.equal(torch.isinf(y[bad]), torch.isinf(want[bad]))
        assert bool(torch.isfinite(torch.cat([y[:bad], y[bad + 1:]])).all())
        assert bool(torch.isfinite(torch.cat([L.glu_proj(x, w)[:bad], L.glu_proj(x, w)[bad + 1:]])).all())
