"""Norm, pages and up projection of a latent layer's single tokens in one launch (csrc/kernels/latent_step.hip): the queries
against 64 bits, the pages against the separate pass."""
import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S
from k8s_llm_rca_amd.ops.linear import proj

pytestmark = pytest.mark.gpu
BF, BS = torch.bfloat16, 32


@pytest.mark.parametrize("T", [1, 2, 7, 8, 9, 16])
@pytest.mark.parametrize("QR,KR,R,pad,N", [(768, 256, 64, 64, 3072), (256, 64, 0, 0, 16), (512, 36, 2, 8, 48), (1024, 512, 64, 96, 256),
                                           (2048, 1984, 64, 64, 32), (1536, 128, 32, 32, 4096)])
@pytest.mark.parametrize("planes", [1, 2, 4])
def test_latent_up(monkeypatch, T, QR, KR, R, pad, N, planes):
    g = torch.Generator().manual_seed(T + QR)

    def rnd(*s):
        return torch.randn(*s, generator=g).cuda()
    dn = rnd(planes, T, QR + KR + R + 4)[..., :QR + KR + R]
    dn = dn[0] if planes == 1 else dn
    wq, wkv, w = rnd(QR).to(BF), rnd(KR).to(BF), (rnd(N, QR) / QR ** 0.5).to(BF)
    slots = torch.tensor([(5 * i + 3) % (T * BS) if i != 4 else -1 for i in range(T)], dtype=torch.int32, device="cuda")
    cs = S.rope_table(torch.arange(T, dtype=torch.int32, device="cuda"), S.make_rope(R, 1e4, "cuda", pairs=True)) if R else None
    c0, t0 = rnd(T, BS, KR + pad).to(BF), rnd(T, KR, BS).to(BF)
    monkeypatch.setattr(S, "LATENT_STEP_READ", 1 << 40)               # (sizes that the rule leaves to two launches, too)
    c1, t1 = c0.clone(), t0.clone()
    kw = dict(tail=R, tail_cs=cs)
    q = S.latent_up(dn, wq, wkv, w, slots, c0, QR, KR, 1e-5, BF, cache_t=t0, **kw)
    S.latent_norm(dn, wq, wkv, slots, c1, QR, KR, 1e-5, BF, cache_t=t1, **kw)
    # (the separate pass adds a single plane's squares in another order: a rounding of bf16 apart)
    for a, b in ((c0, c1), (t0, t1)):
        assert torch.equal(a, b) if planes > 1 else bool(((a.float() - b.float()).abs() <= 2.0 ** -7 * b.float().abs()).all())
    x = (dn.sum(0) if planes > 1 else dn).double()[:, :QR]
    cq = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * wq.double()
    want = cq @ w.double().T
    # the normed rows rounded to bf16 (2^-9 of each term), fp32 sums, the result rounded; twice that
    assert bool(((q.double() - want).abs() <= 2.0 ** -8 * (cq.abs() @ w.double().abs().T + want.abs())).all())


@pytest.mark.parametrize("T", [1, 16, 17])
def test_queries_alone(T):
    g = torch.Generator().manual_seed(T)
    dn, wq = torch.randn(T, 256 + 64, generator=g).cuda(), torch.randn(256, generator=g).to(BF).cuda()
    w, slots = torch.randn(64, 256, generator=g).to(BF).cuda(), torch.arange(T, dtype=torch.int32, device="cuda")
    q = S.latent_up(dn, wq, None, w, slots, None, 256, 64, 1e-5, BF)          # no latent to write: as latent_norm has it
    assert torch.equal(q, proj(S.latent_norm(dn, wq, None, slots, None, 256, 64, 1e-5, BF), w))
