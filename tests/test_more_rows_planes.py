"""Planes of products of 129 to 256 rows (ops/linear.py: _more_rows_plan): the rule, and the sums at its edges."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L

BF = torch.bfloat16


def test_rule():
    assert L.plane_plan(129, 2048, 8192) == (14, 8) and L.plane_plan(256, 2048, 8192) == (13, 8) and L.plane_plan(192, 4096, 4096) == (14, 4)
    for m, n, k in ((257, 2048, 8192), (154, 2048, 2048), (154, 8192, 8192), (154, 2048 + 16, 8192), (154, 2048, 4096 + 32)):
        assert L.plane_plan(m, n, k)[1] == 1


@pytest.mark.gpu
@pytest.mark.parametrize("m", [129, 192, 193, 256])
@pytest.mark.parametrize("n,k", [(2048, 8192), (64, 4096), (4096, 4096 + 512)])
def test_against_64_bits(m, n, k):
    g = torch.Generator().manual_seed(m + n)
    x, w = torch.randn(m, k + 8, generator=g).to(BF).cuda()[:, :k], (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()
    y = L.proj_planes(x, w)
    assert y.shape == (L.plane_plan(m, n, k)[1], m, n) and y.shape[0] > 1
    want = x.double() @ w.double().T
    assert float((y.double().sum(0) - want).abs().max()) < 4e-6 * k ** 0.5         # fp32 sums of k terms of size k^(-1/2), in ranges
