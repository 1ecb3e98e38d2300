"""Attention and matrix memory of single tokens in one launch (csrc/kernels/token_attn.hip, MEM) against the two launches: the same
bits in both results, the caches and the states."""
import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
BF, BS = torch.bfloat16, 64


def meta(pos, maxb):
    n = len(pos)

    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")
    tables = [[i * maxb + (j * 5) % maxb for j in range(maxb)] for i in range(n)]
    slots = i32([tables[i][p // BS] * BS + p % BS for i, p in enumerate(pos)])
    state = list(range(n, 0, -1))
    return S.SegMeta(n, i32(range(n)), i32(range(n + 1)), i32(pos), i32(state), i32(tables), list(range(n + 1)), list(pos),
                     state, n_single=n), slots


@pytest.mark.parametrize("H,G,D,V", [(16, 2, 128, 128), (33, 1, 64, 128), (6, 2, 128, 64), (2, 2, 128, 128), (4, 2, 64, 64)])
@pytest.mark.parametrize("MH,MD,MV", [(16, 64, 128), (3, 64, 64), (5, 128, 64), (2, 128, 128)])
@pytest.mark.parametrize("pos", [[0], [5, 300, 0, 700, 255], [30] * 20])
@pytest.mark.parametrize("kind", ["plain", "window"])
def test_same_bits(monkeypatch, H, G, D, V, MH, MD, MV, pos, kind):
    n, maxb, g = len(pos), 12, torch.Generator().manual_seed(H + MH)
    cols, mcols = (H + G) * D + G * V, 2 * MH * (MD + MV) + 2 * MH

    def rnd(*shape):
        return torch.randn(*shape, generator=g).cuda()
    pad = -(cols + mcols) % 4
    x = rnd(n, cols + mcols + pad)
    k0, v0 = rnd(n * maxb, BS, G * D).to(BF), rnd(n * maxb, G * V, BS).to(BF)
    gb, w = rnd(2 * MH), rnd(MV)
    st0 = [rnd(n + 1, MH, MD, MV) * 0.3, rnd(n + 1, MH, MD), rnd(n + 1, MH)]
    mask = dict(window=200, keep_first=40, sink=rnd(H)) if kind == "window" else {}
    got, made, make = [], [], S._MemoryStep.__init__
    monkeypatch.setattr(S._MemoryStep, "__init__", lambda self, *a: made.append(1) or make(self, *a))
    for one in (True, False):
        seg, slots = meta(pos, maxb)
        kc, vt, st = k0.clone(), v0.clone(), [s.clone() for s in st0]
        memory = (MH, MD, MV, gb, 15.0, *st, seg, w, 1e-5, BF)
        args = (H, G, D, V, seg.seg_pos0, slots, kc, None, vt, seg, BF, D ** -0.5)
        prep = dict(norm=True, eps=1e-5)
        if one:
            o, m = S.attention_and_memory(x[:, :cols], *args, prep, mask, x[:, cols:cols + mcols], *memory)
        else:
            o = S.prep_attention(x[:, :cols], None, *args, prep, mask)
            m = S.memory_layer(x[:, cols:cols + mcols], *memory)
        got.append((o, m, kc, vt, *st))
        assert len(made) == 2 - one                       # one step is prepared, joined or not
    for a, b in zip(*got):
        assert torch.isfinite(a).all() and torch.equal(a, b)


def test_results_of_two_types():
    g = torch.Generator().manual_seed(3)
    seg, slots = meta([40], 4)
    x = torch.randn(1, 20 * 128 + 2 * 4 * 128 + 8, generator=g).cuda()
    xm = x[:, 20 * 128:]
    kc, vt = torch.zeros(4, BS, 256, dtype=BF, device="cuda"), torch.zeros(4, 256, BS, dtype=BF, device="cuda")
    st = [torch.zeros(2, *s, device="cuda") for s in ((4, 64, 64), (4, 64), (4,))]
    memory = (4, 64, 64, torch.zeros(8, device="cuda"), 15.0)
    tail = (seg, None, 1e-5, torch.float32)               # the memory's result stays in fp32
    o, m = S.attention_and_memory(x[:, :20 * 128], 16, 2, 128, 128, seg.seg_pos0, slots, kc, None, vt, seg, BF, 0.1,
                                  dict(norm=True, eps=1e-5), {}, xm, *memory, *(s.clone() for s in st), *tail)
    assert m.dtype == torch.float32 and torch.equal(m, S.memory_layer(xm, *memory, *st, *tail))
