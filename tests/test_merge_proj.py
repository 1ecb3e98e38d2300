"""Parts of single tokens of a latent layer merged by the product behind them (csrc/kernels/token_attn.hip, token_merge_proj_kernel):
the bits of the two launches, for every count of parts a thread may hold, rows that fill no workgroup and parts without a key."""
import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S
from k8s_llm_rca_amd.ops._lib import lib, ptr, stream_ptr

pytestmark = pytest.mark.gpu
BF, BS = torch.bfloat16, 64


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


def meta(ends):
    n, maxb = len(ends), max(ends) // BS + 1
    return S.SegMeta(n, i32(range(n)), i32(range(n + 1)), i32(ends), i32([0] * n),
                     i32([[i * maxb + (j * 3) % maxb if maxb % 3 else i * maxb + j for j in range(maxb)] for i in range(n)]),
                     list(range(n + 1)), list(ends), [0] * n, n_single=n), n * maxb


@pytest.mark.parametrize("H,R,N,tail", [(16, 256, 128, 64), (5, 256, 64, 0), (16, 128, 128, 32), (3, 128, 192, 0)])
@pytest.mark.parametrize("ends", [[200], [5, 300], [700, 0, 31], [128, 127, 129, 1151, 640], [1100] * 6, [2047, 3], [50] * 7 + [513]])
@pytest.mark.parametrize("extras", [False, True])
def test_bits(monkeypatch, H, R, N, tail, ends, extras):
    n, g = len(ends), torch.Generator().manual_seed(H + R + len(ends))
    pages = meta(ends)[1]
    qa = torch.randn(H, n, R, generator=g).to(BF).cuda().transpose(0, 1)
    qr = torch.randn(n, H, tail, generator=g).to(BF).cuda() if tail else None
    c, ct = torch.randn(pages, BS, R + tail, generator=g).to(BF).cuda(), torch.randn(pages, R, BS, generator=g).to(BF).cuda()
    up = (torch.randn(H, R, N, generator=g) * R ** -0.5).to(BF).cuda()
    gate, sink = (torch.randn(n, H + 3, generator=g).cuda(), torch.randn(H, generator=g).cuda()) if extras else (None, None)
    pos, took, rule = i32(ends), [], S._merge_up
    for fused in (True, False):
        monkeypatch.setattr(S, "_merge_up", lambda *a: fused and took.append(rule(*a)) is None and took[-1])
        out = S.latent_attention_mfma(qa, c, ct, gate, meta(ends)[0], pos, 0.05, qr=qr, window=400 if extras else 0, sink=sink,
                                      head_major=True, up=up)
        assert out.shape == (n, H, N) and torch.isfinite(out).all()
        if fused:
            got = out
    assert took == [max(ends) >= 128 and S._few_heads(n, H, R, N, False)] and torch.equal(got, out)


def test_refused():
    po, pml, items = torch.zeros(4 * 256 * 2, device="cuda"), torch.zeros(4 * 2 * 2, device="cuda"), i32([[0, 0, 1, 0]])
    w, out = torch.zeros(4, 256, 64, device="cuda", dtype=BF), torch.zeros(1, 4, 64, device="cuda", dtype=BF)
    ok = [ptr(po), ptr(pml), 2, ptr(items), 1, 0, 0, 0, ptr(w), ptr(out), 256, 64, 4, 256, 64, stream_ptr(w)]
    assert lib().k8s_latent_merge_proj(*ok) == 0
    for at, bad in ((0, 0), (0, ptr(po) + 4), (1, 0), (2, 1), (2, 17), (3, 0), (8, 0), (8, ptr(w) + 2), (9, 0), (12, 0), (13, 192), (14, 96)):
        assert lib().k8s_latent_merge_proj(*ok[:at], bad, *ok[at + 1:]) != 0, (at, bad)
