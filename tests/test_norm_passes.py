"""Norm and preparation passes with wide loads against the CPU forms: many-row latent norm with its transposed pages, norms of
heads in lanes, aligned and unaligned gates, the convolution that keeps its own tail, the embedding read by fours."""
import pytest
import torch

from k8s_llm_rca_amd.ops import norm as N
from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
TYPES = [torch.bfloat16, torch.float32]


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed + sum(shape)))


def same(a, b, dt):
    """One rounding of ``dt`` apart, sums of up to 2048 fp32 terms in another order."""
    a, b = a.double().cpu(), b.double()
    eps = 2.0 ** -7 if dt == torch.bfloat16 else 1e-5
    assert bool(((a - b).abs() <= eps * b.abs() + 1e-5).all()), float((a - b).abs().max())


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("T", [1535, 1536, 1543])
@pytest.mark.parametrize("QR,KR,R,pad,shift", [(768, 256, 64, 64, 0), (100, 36, 6, 32, 3), (2048, 1024, 0, 0, 0), (64, 32, 8, 8, 1),
                                               (66, 30, 2, 2, 0)])
def test_latent_norm(T, QR, KR, R, pad, shift, dt):
    BS = 32
    pages = (T + shift) // BS + 2
    order = torch.randperm(pages, generator=torch.Generator().manual_seed(T))
    at = torch.arange(T) + shift
    slots = (order[at // BS] * BS + at % BS).to(torch.int32)
    slots[[5, 700, T - 1]] = -1
    dn, wq, wk = rnd(T, QR + KR + R), rnd(QR).to(dt), rnd(KR, seed=1).to(dt)
    cs = rnd(T, R) if R else None
    res = {}
    for dev in ("cpu", "cuda"):
        cache, ct = torch.full((pages, BS, KR + pad), 7.0, dtype=dt, device=dev), torch.full((pages, KR, BS), 7.0, dtype=dt, device=dev)
        cq = S.latent_norm(dn.to(dev), wq.to(dev), wk.to(dev), slots.to(dev), cache, QR, KR, 1e-5, dt, cache_t=ct, tail=R,
                           tail_cs=None if cs is None else cs.to(dev))
        res[dev] = (cq, cache, ct)
    for a, b in zip(res["cuda"], res["cpu"]):
        same(a, b, dt)
    assert torch.equal(res["cuda"][2].transpose(1, 2), res["cuda"][1][..., :KR])


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("gdt", TYPES)
@pytest.mark.parametrize("H,V", [(5, 64), (16, 128), (3, 256), (2, 96), (1, 2048), (1, 260)])
@pytest.mark.parametrize("T", [1, 7, 300])
def test_head_norm(T, H, V, gdt, dt):
    o, gate, mul = rnd(T, H * V), rnd(T, H * V + 8).to(gdt), rnd(T, H).abs() + 0.1
    for col in (0, 4, 1):                                   # aligned, aligned for 4-byte gates, not aligned
        for w in (None, rnd(V), rnd(H * V, seed=3)):
            for kw in (dict(), dict(mul=mul, out_scale=0.7)):
                def run(dev):
                    k = dict(kw, mul=kw["mul"].to(dev)) if "mul" in kw else kw
                    return S.head_norm_gate(o.to(dev), gate.to(dev)[:, col:], None if w is None else w.to(dev), H, V, 1e-5, dt, **k)
                same(run("cuda"), run("cpu"), dt)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("taps", [2, 3, 4, 5])
def test_convolution_tails(taps, dt):
    """Segments of one tile (the convolution leaves the tail itself), of several, and both: outputs and tails."""
    C = 300
    for lens, pos0 in (([1, 1, 1], [0, 9, 4]), ([3, 16, 1], [0, 5, 20]), ([17, 2, 40], [0, 6, 7])):
        T, row0 = sum(lens), [0]
        for n in lens:
            row0.append(row0[-1] + n)
        x, w, tail = rnd(T, C).to(dt), rnd(C, taps), rnd(4, taps - 1, C, seed=2)
        slots, res = [2, 0, 3], {}
        for dev in ("cpu", "cuda"):
            def i32(v):
                return torch.tensor(v, dtype=torch.int32, device=dev)
            m = S.SegMeta(3, i32([s for s, n in enumerate(lens) for _ in range(n)]), i32(row0), i32(pos0), i32(slots),
                          i32([[0]] * 3), row0, pos0, slots)
            t = tail.clone().to(dev)
            res[dev] = (S.short_conv(x.to(dev), w.to(dev), None, t, m), t)
        same(res["cuda"][0], res["cpu"][0], dt)
        assert torch.equal(res["cuda"][1].cpu(), res["cpu"][1])


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("W", [2048, 36, 37, 4096])
def test_embedding(W, dt):
    emb, w, b = rnd(50, W).to(dt), rnd(W), rnd(W, seed=1)
    ids, res = torch.tensor([3, 49, 0, 7, 7], dtype=torch.int32), {}
    for dev in ("cpu", "cuda"):
        x = torch.empty(5, W, device=dev)
        h = N.embed_scale_dyt(ids.to(dev), emb.to(dev), 3.0, x, 0.5, w.to(dev), b.to(dev), out_dtype=dt)
        res[dev] = (x, h)
    assert torch.equal(res["cuda"][0].cpu(), res["cpu"][0])
    same(res["cuda"][1], res["cpu"][1], dt)
