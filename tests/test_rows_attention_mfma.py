"""fp32 attention of rows on the matrix units: the same bits as the general kernel, which a workgroup per part of 128 keys is
always made by."""
import pytest
import torch

from k8s_llm_rca_amd.ops._lib import check, lib, ptr, stream_ptr

pytestmark = pytest.mark.gpu
BS, PARTS = 64, 4


def step(segs, g):
    """Block tables, segment of a row, first rows and positions of ``segs`` = (rows, tokens before them), pages in any order."""
    pages = [-(-(n + p) // BS) for n, p in segs]
    table, order, at = torch.zeros(len(segs), max(pages), dtype=torch.int32), torch.randperm(sum(pages), generator=g).int(), 0
    for i, k in enumerate(pages):
        table[i, :k] = order[at:at + k]
        at += k
    rows = [n for n, _ in segs]
    seg = torch.repeat_interleave(torch.arange(len(segs), dtype=torch.int32), torch.tensor(rows))
    row0 = torch.tensor([sum(rows[:i]) for i in range(len(segs) + 1)], dtype=torch.int32)
    pos0 = torch.tensor([p for _, p in segs], dtype=torch.int32)
    return [t.cuda() for t in (table, seg, row0, pos0)] + [sum(pages), sum(rows)]


def both(run, T, H, V):
    """The result of the kernel that walks a row's parts, and of a workgroup per part."""
    out = [torch.full((T, H, V), 7.0, device="cuda") for _ in range(2)]
    po, pml = (torch.empty(T * H * PARTS * n, device="cuda") for n in (V, 2))
    run(out[0], 0, None, None)
    run(out[1], PARTS, po, pml)
    return out


# (rows, tokens before): one key, ends of a tile of 16 and of four, of a part, several parts; a last key of each sort
SEGS = [(1, 0), (3, 14), (1, 62), (2, 63), (3, 126), (1, 128), (40, 220), (1, 500)]


@pytest.mark.parametrize("H,G,D,V,maps", [(16, 2, 128, 128, 1), (4, 1, 16, 64, 1), (15, 3, 80, 192, 1), (17, 1, 64, 256, 1),
                                          (16, 2, 64, 128, 2), (24, 2, 192, 64, 1), (6, 2, 64, 64, 1)])
@pytest.mark.parametrize("mask", [{}, {"window": 90, "keep_first": 3, "sink": True}, {"chunk": 200, "cap": 8.0, "gate": True}])
def test_masked(H, G, D, V, maps, mask):
    g = torch.Generator().manual_seed(H + D)
    table, seg, row0, pos0, pages, T = step(SEGS, g)
    HQ = H * maps
    q, kc, vc = (torch.randn(*s, generator=g).cuda() for s in ((T, HQ * D), (pages * BS, G * maps * D), (pages * BS, G * V)))
    sink = torch.randn(HQ, generator=g).cuda() if "sink" in mask else None
    gate = torch.randn(T, HQ + 1, generator=g).cuda() if "gate" in mask else None
    kc[5], vc[7] = float("-inf"), float("inf")       # (a score and a value of somebody's; NaN where they meet)

    def run(out, parts, po, pml):
        check(lib().k8s_masked_attn_rows(ptr(q), ptr(kc), ptr(vc), ptr(table), table.shape[1], ptr(seg), ptr(row0), ptr(pos0),
                                         ptr(sink), ptr(gate), HQ + 1, ptr(out), T, H, G, D, V, BS, mask.get("chunk", 0),
                                         mask.get("window", 0), mask.get("keep_first", 0), D ** -0.5, mask.get("cap", 0.0), 1,
                                         stream_ptr(q), maps, 0, parts, ptr(po), ptr(pml)), "masked_attn_rows")
    a, b = both(run, T, HQ, V)
    assert torch.equal(a.nan_to_num(123.0), b.nan_to_num(123.0)) and bool(torch.isfinite(a).any())


@pytest.mark.parametrize("H,R,RP", [(16, 256, 64), (4, 64, 16), (20, 128, 32), (5, 512, 0), (16, 192, 64)])
@pytest.mark.parametrize("window", [0, 100])
def test_latent(H, R, RP, window):
    g = torch.Generator().manual_seed(H + R)
    table, seg, row0, pos0, pages, T = step(SEGS, g)
    qa, cache = torch.randn(T, H, R, generator=g).cuda(), torch.randn(pages * BS, R + RP, generator=g).cuda()
    qr = torch.randn(T, H, RP, generator=g).cuda() if RP else None

    def run(out, parts, po, pml):
        check(lib().k8s_latent_attn_rows(ptr(qa), ptr(cache), ptr(table), table.shape[1], ptr(seg), ptr(row0), ptr(pos0), None, 0,
                                         ptr(out), 0, T, H, R, BS, (R + RP) ** -0.5, 1, stream_ptr(qa), H * R, R, ptr(qr), RP,
                                         H * R, R, window, None, parts, ptr(po), ptr(pml)), "latent_attn_rows")
    a, b = both(run, T, H, R)
    assert torch.equal(a, b) and bool(torch.isfinite(a).all())
