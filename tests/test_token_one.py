"""Attention of single tokens whose waves have a block each (csrc/kernels/token_attn.hip, ONE) against the form that walks over
several: the same bits.  The second runs where a step has as many parts as there may be."""
import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
BF, BS = torch.bfloat16, 64
ENDS = [0, 31, 32, 127, 128, 255, 256, 257, 511, 512, 700]


def meta():
    n, maxb = len(ENDS), 11

    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")
    return S.SegMeta(n, i32(range(n)), i32(range(n + 1)), i32(ENDS), i32([0] * n),
                     i32([[i * maxb + (j * 3) % maxb for j in range(maxb)] for i in range(n)]), list(range(n + 1)), list(ENDS),
                     [0] * n, n_single=n), n * maxb


@pytest.mark.parametrize("H,G,D,V", [(16, 2, 128, 128), (40, 2, 64, 128), (6, 3, 128, 64), (20, 1, 96, 96)])
@pytest.mark.parametrize("kw", [dict(), dict(window=300, keep_first=70), dict(chunk=300, softcap=8.0)])
def test_masked(monkeypatch, H, G, D, V, kw):
    g = torch.Generator().manual_seed(H + D)
    _, pages = meta()
    q = torch.randn(len(ENDS), H * D, generator=g).to(BF).cuda()
    kc, vt = torch.randn(pages, BS, G * D, generator=g).to(BF).cuda(), torch.randn(pages, G * V, BS, generator=g).to(BF).cuda()
    parts = S._mask_plan(meta()[0], H, G, D, V, kw.get("chunk", 0), kw.get("window", 0), kw.get("keep_first", 0), 1)[1]
    out = []
    for most in (64, parts):
        monkeypatch.setattr(S, "TOKEN_PARTS", most)
        out.append(S.masked_attention(q, H, G, D, V, kc, None, meta()[0], D ** -0.5, vt=vt, **kw))
    assert 1 < parts < 64 and torch.isfinite(out[0]).all() and torch.equal(*out)


@pytest.mark.parametrize("H,R,tail", [(16, 256, 64), (20, 192, 32), (16, 512, 64), (5, 64, 32)])
@pytest.mark.parametrize("window", [0, 400])
def test_latent(monkeypatch, H, R, tail, window):
    g = torch.Generator().manual_seed(H + R)
    seg, pages = meta()
    qa, qr = torch.randn(len(ENDS), H, R, generator=g).to(BF).cuda(), torch.randn(len(ENDS), H, tail, generator=g).to(BF).cuda()
    c, ct = torch.randn(pages, BS, R + tail, generator=g).to(BF).cuda(), torch.randn(pages, R, BS, generator=g).to(BF).cuda()
    pos = torch.tensor(ENDS, dtype=torch.int32, device="cuda")
    n = [0]
    groups = S._token_groups

    def counted(rows, heads, parts, V):
        n[0] = parts
        return groups(rows, heads, parts, V)
    monkeypatch.setattr(S, "_token_groups", counted)

    def run(most):
        monkeypatch.setattr(S, "TOKEN_PARTS", most)
        return S.latent_attention_mfma(qa, c, ct, None, meta()[0], pos, 0.05, qr=qr, window=window)
    one = run(64)
    parts = n[0]
    assert 1 < parts < 64 and torch.isfinite(one).all() and torch.equal(one, run(parts)) and n[0] == parts
