"""SwiGLU's gate at every bf16 number (csrc/kernels/common.h: silu_gate, silu_gate_near): the epilogue of the large products, which
divides by a short form where it can, has the separate pass's bits, and that has what 64 bits give."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops import norm as N

pytestmark = pytest.mark.gpu
BF, M, K = torch.bfloat16, 128, 128


def test_every_gate():
    z = torch.arange(-2 ** 15, 2 ** 15, dtype=torch.int32).to(torch.int16).view(BF).float()
    z = torch.where(torch.isfinite(z) & (z.abs() >= 2.0 ** -126), z, torch.zeros(()))
    z = z[z.abs().argsort()].cuda()                                    # near and far ones apart, so that both forms see their own
    u = (0.5 + 1.5 * torch.rand(M, generator=torch.Generator().manual_seed(1))).to(BF).cuda()
    # row m is the m-th unit vector: gate z[n], up u[m]
    x = torch.eye(M, K, dtype=BF, device="cuda")
    w = torch.cat([z.to(BF)[:, None].expand(-1, K), u.expand(len(z), K)]).contiguous()
    gu = torch.cat([z.to(BF).expand(M, -1), u[:, None].expand(-1, len(z))], 1).contiguous()
    want = N.silu_mul(gu)
    for pipe in (1, 5):
        assert torch.equal(L.gemm_big(x, w, silu=True, pipe=pipe), want)
    exact = z.double() * torch.sigmoid(z.double()) * u.double()[:, None]
    # the exponential (88 2^-24 at most) and the result's rounding; past -88.6 it overflows and the gate is zero
    far = torch.where(z < -88.6, 6e-37, 1e-38).double()
    fits = exact.abs() < 3.38e38                                       # (others round to an infinity)
    assert bool((((want.double() - exact).abs() <= 2.0 ** -8 * exact.abs() + far) | ~fits).all())
