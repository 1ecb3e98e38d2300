"""Products of a few rows as planes over ranges of K, and the consumers that add the planes where they read them."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops import norm as N
from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed + sum(shape)))


@pytest.mark.parametrize("n,k", [(2048, 2048), (2048, 8192), (1088, 2048), (2560, 2048), (64, 256), (384, 640), (4096, 4096),
                                 (100, 512), (16384, 2048)])
@pytest.mark.parametrize("m", [1, 7, 16, 17, 64, 65, 128, 129])
def test_planes_sum_to_the_product(n, k, m):
    x, w = rnd(m, k).to(BF), (rnd(n, k) * k ** -0.5).to(BF)
    y = L.proj_planes(x.cuda(), w.cuda())
    assert y.dtype == torch.float32 and y.shape[1:] == (m, n) and y.shape[0] == L.plane_plan(m, n, k)[1]
    want = x.double() @ w.double().T
    # fp32 sums of K terms of size K^(-1/2), in ranges
    assert float((y.double().sum(0).cpu() - want).abs().max()) < 4e-6 * k ** 0.5


@pytest.mark.parametrize("planes", [1, 2, 3, 4, 8])
@pytest.mark.parametrize("t,w", [(1, 2048), (5, 384), (64, 100), (3, 37)])
def test_residual_consumers(planes, t, w):
    y, y2, nw = rnd(planes, t, w), rnd(3, t, w, seed=1), rnd(w)
    x0 = rnd(t, 1, w, seed=2)
    one, mix = torch.ones(1), torch.ones(1, 1)
    res = {}
    for dev in ("cpu", "cuda"):
        x = x0.clone().to(dev)
        h = N.hyper_step(x, y.to(dev), one.to(dev), mix.to(dev), inn=one.to(dev), nw=nw.to(dev), eps=1e-5,
                         out_dtype=torch.float32)
        x2 = x0[:, 0].clone().to(dev)
        d = N.add_dyt(x2, y.to(dev), 0.7, y2.to(dev), 0.9, 0.8, nw.to(dev), nw.to(dev), out_dtype=torch.float32)
        x3 = x0[:, 0].clone().to(dev)
        N.add_dyt(x3, y.to(dev))
        res[dev] = [v.cpu() for v in (x, h, x2, d, x3)]
    for a, b in zip(res["cuda"], res["cpu"]):
        assert float((a - b).abs().max()) < 1e-5 * max(1.0, float(b.abs().max()))      # up to eleven fp32 terms, one norm


@pytest.mark.parametrize("planes", [2, 3, 8])
@pytest.mark.parametrize("t", [1, 6, 64])
def test_preparing_consumers(planes, t):
    H, G, D, V, QR, KR, R, BS = 4, 2, 64, 32, 80, 96, 32, 32
    x, dn = rnd(planes, t, (H + G) * D + G * V), rnd(planes, t, QR + KR + R)
    bias, wq, wkv = rnd((H + G) * D + G * V), rnd(QR), rnd(KR)
    slots, pos = torch.randperm(4 * BS)[:t].to(torch.int32), torch.arange(t, dtype=torch.int32) * 7
    res = {}
    for dev in ("cpu", "cuda"):
        kc, vc, cache = (torch.zeros(4, BS, n).to(dev) for n in (G * D, G * V, KR + 64))
        rope, pairs = S.make_rope(D, 1e4, dev), S.make_rope(R, 1e4, dev, pairs=True)
        q = S.attn_prep(x.to(dev), bias.to(dev), H, G, D, V, pos.to(dev), slots.to(dev), kc, vc, torch.float32, norm="head",
                        eps=1e-5, rope=rope, rope_cs=S.rope_table(pos.to(dev), rope))
        cq = S.latent_norm(dn.to(dev), wq.to(dev), wkv.to(dev), slots.to(dev), cache, QR, KR, 1e-5, torch.float32, tail=R,
                           tail_cs=S.rope_table(pos.to(dev), pairs))
        # a form the summing kernel does not take (no table): summed in front of it
        q2 = S.attn_prep(x.to(dev), None, H, G, D, V, pos.to(dev), slots.to(dev), kc.clone(), vc.clone(), torch.float32,
                         norm=True, eps=1e-5, rot_dims=16)
        res[dev] = [v.cpu() for v in (q, kc, vc, cq, cache, q2)]
    for a, b in zip(res["cuda"], res["cpu"]):
        assert float((a - b).abs().max()) < 1e-5 * max(1.0, float(b.abs().max()))
