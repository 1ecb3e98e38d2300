"""Attention of single tokens that prepares its rows itself (csrc/kernels/token_attn.hip, PREP) against the pass and the
attention apart: the same bits, in the result and in the caches."""
import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
BF, BS = torch.bfloat16, 64
#: positions: the first, ends of blocks, of pages and of parts
ENDS = [0, 1, 31, 32, 63, 64, 255, 256, 257, 700]


def meta(pos, maxb):
    n = len(pos)

    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")
    tables = [[i * maxb + (j * 5) % maxb for j in range(maxb)] for i in range(n)]      # (5 and maxb have no common factor)
    slots = i32([tables[i][p // BS] * BS + p % BS for i, p in enumerate(pos)])
    return S.SegMeta(n, i32(range(n)), i32(range(n + 1)), i32(pos), i32([0] * n), i32(tables), list(range(n + 1)), list(pos),
                     [0] * n, n_single=n), slots


@pytest.mark.parametrize("H,G,D,V", [(16, 2, 128, 128), (4, 4, 64, 64), (6, 6, 128, 128), (33, 1, 64, 128), (6, 2, 128, 64)])
@pytest.mark.parametrize("planes", [1, 3, 4, 8])
@pytest.mark.parametrize("kind", ["plain", "chunk", "window", "values"])
def test_same_bits(H, G, D, V, planes, kind):
    g = torch.Generator().manual_seed(H + planes)
    n, maxb, cols = len(ENDS), 12, (H + G) * D + G * V

    def rnd(*shape):
        return torch.randn(*shape, generator=g).cuda()
    seg, slots = meta(ENDS, maxb)
    pos = torch.tensor(ENDS, dtype=torch.int32, device="cuda")
    x = rnd(planes, n, cols + 8)[..., :cols]
    x = x if planes > 1 else x[0]
    rope = S.make_rope(D // 2 if kind == "window" else D, 10000.0, "cuda") if kind in ("plain", "window") else None
    bias = rnd(cols) if kind != "window" else None
    prep = dict(norm=kind != "values", eps=1e-5, rope=rope, rope_cs=S.rope_table(pos, rope) if rope else None)
    mask = {"plain": {}, "chunk": dict(chunk=150, softcap=8.0, gate=rnd(n, H + 3)[:, 3:]),
            "window": dict(window=200, keep_first=40, sink=rnd(H)), "values": {}}[kind]
    if kind == "chunk":
        prep.update(q_w=rnd(D), k_w=rnd(D))
    if kind == "values":
        prep.update(lam=0.3, v_other=rnd(n, G * V))
    k0, v0 = rnd(n * maxb, BS, G * D).to(BF), rnd(n * maxb, G * V, BS).to(BF)
    got = []
    for apart in (False, True):
        # (what lies at the row's own place must not matter)
        kc, vt = k0.clone(), v0.clone()
        kc.view(-1, G * D)[slots.long()] = float("nan")
        vt[(slots // BS).long(), :, (slots % BS).long()] = float("nan")
        vc = torch.zeros(n * maxb, BS, G * V, dtype=BF, device="cuda") if kind != "plain" else None
        keep = torch.zeros(n, G * V, device="cuda") if kind in ("chunk", "values") else None
        p = dict(prep, v_keep=keep)
        if apart:
            q = S.attn_prep(x, bias, H, G, D, V, pos, slots, kc, vc, BF, vt=vt, **p)
            o = S.masked_attention(q, H, G, D, V, kc, vc, seg, D ** -0.5, vt=vt, **mask)
        else:
            o = S._prep_tokens(x, bias, H, G, D, V, slots, kc, vc, vt, seg, BF, D ** -0.5, **p, **mask)
            assert o is not None
        got.append((o, kc, vt) + tuple(t for t in (vc, keep) if t is not None))
    for a, b in zip(*got):
        assert torch.isfinite(a).all() and torch.equal(a, b)


def test_rows_of_one_sequence_are_prepared_apart():
    """Two rows of a sequence see each other's keys: the pass has to end first."""
    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")
    seg = S.SegMeta(1, i32([0, 0]), i32([0, 2]), i32([3]), i32([0]), i32([[0]]), [0, 2], [3], [0])
    x = torch.randn(2, 6 * 64, device="cuda")
    kc, vt = (torch.zeros(s, dtype=BF, device="cuda") for s in ((1, BS, 64), (1, 64, BS)))
    args = (x, None, 4, 1, 64, 64, i32([3, 4]), kc, None, vt, seg, BF, 0.125)
    assert S._prep_tokens(*args[:6], args[6], *args[7:]) is None
