"""Small products of few rows on the vector pipes against 64 bits, on both sides of their row rule and at odd sizes."""
import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed + sum(shape)))


def close(got, want, dt=BF):
    """One rounding of the result, and fp32 sums."""
    assert got.dtype == dt and got.shape == want.shape
    ulp = 2.0 ** -8 if dt == BF else 2.0 ** -24
    assert bool(((got.double().cpu() - want).abs() <= ulp * want.abs() + 1e-5 * float(want.abs().max())).all())


@pytest.mark.parametrize("T", [1, 3, 4, 5, 8, 9, 64, 128, 129])
@pytest.mark.parametrize("H,D,R,KR,pad", [(16, 128, 64, 256, 64), (3, 40, 6, 64, 32), (2, 200, 0, 128, 0), (5, 8, 32, 192, 64)])
@pytest.mark.parametrize("dt", [BF, torch.float32])
def test_heads(T, H, D, R, KR, pad, dt):
    q, uk = rnd(T, H * (D + R)).to(dt), (rnd(H, D, KR) * D ** -0.5).to(dt)
    cs = rnd(T, R) if R else None
    qa, qr = S.latent_queries(q.cuda(), uk.cuda(), cs.cuda() if R else None, H, D, pad)
    x = q.view(T, H, D + R)
    close(qa, torch.bmm(x[:, :, :D].double().transpose(0, 1), uk.double()).transpose(0, 1), dt)
    assert qa.transpose(0, 1).is_contiguous()
    if R:
        assert torch.equal(qr, S.rotated_tail(q.cuda(), cs.cuda(), H, D, pad))
    else:
        assert qr is None
    # out of latent space: head-major in, token-major out
    uv = (rnd(H, KR, 64) * KR ** -0.5).to(dt)
    out = torch.empty(T, H, 64, dtype=dt, device="cuda")
    close(S.head_proj(qa, uv.cuda(), out), torch.bmm(qa.double().cpu().transpose(0, 1), uv.double()).transpose(0, 1), dt)


@pytest.mark.parametrize("T", [1, 4, 7, 64, 128, 129])
@pytest.mark.parametrize("K0,N0,K1,N1", [(64, 2048, 64, 2048), (32, 100, 160, 7), (48, 64, 32, 64)])
def test_two_of_low_rank(T, K0, N0, K1, N1):
    x, w0, w1 = rnd(T, K0 + K1 + 3), (rnd(N0, K0) * K0 ** -0.5).to(BF), (rnd(N1, K1) * K1 ** -0.5).to(BF)
    got = S.low_rank_pair(x.cuda(), 2, w0.cuda(), 2 + K0, w1.cuda(), BF)
    for y, w, c in zip(got, (w0, w1), (2, 2 + K0)):
        want = x[:, c:c + w.shape[1]].to(BF).double() @ w.double().T
        assert y.dtype == torch.float32 and y.shape == want.shape
        assert float((y.double().cpu() - want).abs().max()) < 4e-6 * w.shape[1] ** 0.5
