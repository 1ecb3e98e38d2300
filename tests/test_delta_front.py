"""The front of the delta layer's reply steps against its separate launches, to the bit: the product whose epilogue convolves
(csrc/kernels/gemm_rows.hip) and the state's step that makes its products of low rank (csrc/kernels/state_step.hip)."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops import row_step as R
from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def meta(pos0, slots):
    n = len(pos0)

    def i32(v):
        return torch.tensor(list(v), dtype=torch.int32, device="cuda")
    return S.SegMeta(n, i32(range(n)), i32(range(n + 1)), i32(pos0), i32(slots), i32([0] * n).view(n, 1), list(range(n + 1)),
                     list(pos0), list(slots), n_single=n)


@pytest.mark.parametrize("T", [1, 2, 7, 16])
@pytest.mark.parametrize("C,rest,K,taps", [(2304, 144, 2048, 4), (256, 16, 512, 3), (512, 32, 1536, 2), (160, 48, 1024, 1),
                                           (6144, 2048, 1024, 4)])
def test_convolving_product(T, C, rest, K, taps):
    g = torch.Generator().manual_seed(T + C)
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()      # noqa: E731
    pos0, slots = [i % 5 for i in range(T)], [(3 * i + 1) % (T + 3) if T % 3 else T - i for i in range(T)]
    slots = slots if len(set(slots)) == T else list(range(T, 0, -1))
    x = rnd(T, K + 8)[:, :K].to(BF) if T == 2 else rnd(T, K).to(BF)      # (rows further apart, too)
    w, cw, tail = (rnd(C + rest, K) / K ** 0.5).to(BF), rnd(C, taps), rnd(T + 3, taps - 1, C)
    nf, _ = L.rows_plan(T, C + rest, K)
    if C % (16 * nf):
        pytest.skip("strip across both parts")
    seg, t0, t1 = meta(pos0, slots), tail.clone(), tail.clone()
    out, r = R.conv_proj(x, w, cw, t0, seg)
    want = S.short_conv(L.gemm_rows(x, w[:C], nf), cw, None, t1, seg, act=True)
    assert torch.equal(out, want) and torch.equal(t0, t1)
    assert torch.equal(r, L.gemm_rows(x, w, nf, L.ROWS_F32)[:, C:])


def test_portions_go_the_general_way():
    x, w = torch.randn(3, 512, device="cuda").to(BF), torch.randn(272, 512, device="cuda").to(BF)
    cw, tail = torch.randn(256, 4, device="cuda"), torch.zeros(2, 3, 256, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")      # noqa: E731
    seg = S.SegMeta(2, i32([0, 0, 1]), i32([0, 2, 3]), i32([0, 0]), i32([0, 1]), i32([[0], [0]]), [0, 2, 3], [0, 0], [0, 1])
    t1 = tail.clone()
    out, rest = R.conv_proj(x, w, cw, tail, seg)
    assert torch.equal(out, S.short_conv(L.proj(x, w[:256]), cw, None, t1, seg)) and torch.equal(tail, t1)
    assert torch.equal(rest, L.proj_f32out(x, w[256:]))


@pytest.mark.parametrize("T", [1, 5, 16])
@pytest.mark.parametrize("H,G,D,V,ra,rg", [(16, 2, 64, 128, 64, 64), (4, 4, 64, 64, 32, 128), (6, 3, 128, 128, 128, 32),
                                           (2, 1, 128, 64, 96, 96)])
@pytest.mark.parametrize("wide", [True, False, None])
def test_low_rank(monkeypatch, T, H, G, D, V, ra, rg, wide):
    g = torch.Generator().manual_seed(T + H)
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()      # noqa: E731
    qkv, lr = rnd(T, 2 * G * D + H * V).to(BF), rnd(T, ra + rg + H)
    wa, wg = (rnd(H * D, ra) / ra ** 0.5).to(BF), (rnd(H * V, rg) / rg ** 0.5).to(BF)
    rate, db, st = rnd(H).abs(), rnd(H * D), rnd(T + 2, H, D, V) * 0.3
    w = None if wide is None else rnd(H * V if wide else V)
    monkeypatch.setattr(S, "DELTA_LOW_HEAD", 1 << 30)              # (heads that the rule leaves to two launches, too)
    seg, s1 = meta([i % 3 for i in range(T)], range(T, 0, -1)), st.clone()
    out = S.delta_low_rank(qkv, H, G, D, V, lr, wa, wg, rate, db, st, seg, w, 1e-5, BF)
    dec, gate = S.low_rank_pair(lr, 0, wa, ra, wg, BF)
    want = S.delta_layer(qkv, H, G, D, V, dec, rate, db, lr[:, ra + rg:], s1, seg, gate, w, 1e-5, BF)
    assert torch.isfinite(out).all() and torch.equal(out, want) and torch.equal(st, s1)
