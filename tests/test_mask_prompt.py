"""Masked attention of prompt portions on the matrix cores (tiles of 128 token-head rows over 64-key blocks) in a step with
single tokens in front, against 64 bits: every mask, page sizes whose blocks cross pages, odd head counts, score maps."""
import math

import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
LENS, POS0 = [1, 1, 170, 33, 1, 129], [0, 300, 0, 95, 200, 64]      # two single tokens in front, one among the portions


def meta(n_pages, pages):
    row0 = [0]
    for n in LENS:
        row0.append(row0[-1] + n)

    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device="cuda")
    return S.SegMeta(len(LENS), i32([s for s, n in enumerate(LENS) for _ in range(n)]), i32(row0), i32(POS0),
                     i32([0] * len(LENS)), i32([pages] * len(LENS)), row0, list(POS0), [0] * len(LENS))


@pytest.mark.parametrize("H,G,D,V,maps,BS", [(16, 2, 128, 128, 1, 64), (3, 3, 64, 64, 1, 32), (20, 1, 96, 96, 1, 96),
                                             (6, 2, 64, 128, 2, 64), (131, 1, 64, 64, 1, 128), (5, 1, 128, 64, 1, 32)])
@pytest.mark.parametrize("kw", [dict(), dict(window=70, keep_first=20), dict(window=1), dict(window=130, keep_first=70),
                                dict(chunk=50, softcap=6.0), dict(chunk=100, window=33, keep_first=3),
                                dict(scale=-0.05), dict(scale=0.0)])
def test_prompts(H, G, D, V, maps, BS, kw):
    kw = dict(kw)
    n, HQ = 320, H * maps
    g = torch.Generator().manual_seed(D + H)
    scale = kw.pop("scale", D ** -0.5)
    N = -(-n // BS)
    pages = torch.randperm(N, generator=g).tolist()
    k, v = torch.randn(n, G * maps, D, generator=g).to(BF), torch.randn(n, G, V, generator=g).to(BF)
    kc, vt = torch.zeros(N, BS, G * maps * D, dtype=BF), torch.zeros(N, G * V, BS, dtype=BF)
    for i in range(n):
        kc[pages[i // BS], i % BS], vt[pages[i // BS], :, i % BS] = k[i].reshape(-1), v[i].reshape(-1)
    T, m = sum(LENS), meta(N, pages)
    assert [x.shape[0] > 0 for x in m.mask_items(max(1, 128 // (H // G)))[:2]] == [True, True]
    q = (2 * torch.randn(T, HQ, D, generator=g)).to(BF)
    sink, gate = torch.randn(HQ, generator=g), torch.randn(T, HQ + 1, generator=g)
    got = {f32: S.masked_attention(q.view(T, -1).cuda(), H, G, D, V, kc.cuda(), None, m, scale, sink=sink.cuda(),
                                   gate=gate.cuda()[:, 1:], vt=vt.cuda(), maps=maps, out_f32=f32, **kw) for f32 in (0, 1)}
    assert torch.equal(got[1].to(BF), got[0])
    qi = torch.cat([p + torch.arange(x) for p, x in zip(POS0, LENS)])[:, None]
    kp = torch.arange(n)[None]
    vis = kp <= qi
    if "chunk" in kw:
        vis &= qi // kw["chunk"] == kp // kw["chunk"]
    if "window" in kw:
        vis &= (qi - kp < kw["window"]) | (kp < kw.get("keep_first", 0))
    rep = H // G
    kk = k.double().view(n, G, maps, D).repeat_interleave(rep, 1).reshape(n, HQ, D)
    vv = v.double().repeat_interleave(rep, 1).repeat_interleave(maps, 1)
    s = torch.bmm(q.double().transpose(0, 1), kk.permute(1, 2, 0).contiguous()) * scale           # [HQ, T, n]
    if "softcap" in kw:
        s = kw["softcap"] * torch.tanh(s / kw["softcap"])
    s = s.masked_fill(~vis[None], -math.inf)
    p = torch.softmax(torch.cat([s, sink.double()[:, None, None].expand(HQ, T, 1)], -1), -1)[..., :-1]
    want = torch.bmm(p, vv.transpose(0, 1).contiguous()).transpose(0, 1) * torch.sigmoid(gate[:, 1:].double())[..., None]
    # the weights are rounded to bf16 (2^-9 each, of both signs) before they meet the values, the result once more
    assert float((got[1].double().cpu().view(T, HQ, V) - want).abs().max()) < 2.0 ** -7 * float(want.abs().max())


@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("H,G,D,V,BS", [(8, 1, 128, 128, 64), (2, 2, 64, 64, 32), (4, 2, 96, 96, 96)])
@pytest.mark.parametrize("kw", [dict(), dict(window=50, keep_first=7), dict(chunk=40, softcap=9.0)])
@pytest.mark.parametrize("way", ["tiles", "parts"])
def test_values_that_are_not_finite_reach_only_the_rows_that_see_them(H, G, D, V, BS, kw, value, way, monkeypatch):
    """One entry of one key's value, of a key at every place in a block: rows that do not see the key keep their bits, and so
    do all other columns; keys that nobody has written are not read into the sums either."""
    monkeypatch.setattr(S, "MASK_ROW_BYTES", -1)
    monkeypatch.setattr(S, "MASK_TILE_BLOCKS", 1 if way == "parts" else 1000)
    n, lead = 240, 60
    g = torch.Generator().manual_seed(BS)
    N = -(-n // BS)
    kc, v = torch.randn(N, BS, G * D, generator=g).to(BF).cuda(), torch.randn(N * BS, G, V, generator=g).to(BF)
    q, T = torch.randn(n - lead, H * D, generator=g).to(BF).cuda(), n - lead

    def i32(x):
        return torch.tensor(x, dtype=torch.int32, device="cuda")
    m = S.SegMeta(1, i32([0] * T), i32([0, T]), i32([lead]), i32([0]), i32([list(range(N))]), [0, T], [lead], [0])

    def run(keys):
        vx = v.clone()
        vx[n:] = value
        for t in keys:
            vx[t, -1, V - 3] = value
        vt = vx.view(N, BS, G * V).transpose(1, 2).contiguous().cuda()
        return S.masked_attention(q, H, G, D, V, kc, None, m, D ** -0.5, vt=vt, out_f32=True, **kw).view(T, H, V)
    clean = run([])
    assert bool(torch.isfinite(clean).all())
    pos = torch.arange(lead, n, device="cuda")
    for keys in ([3], [70], [127], [128], [191], [239], [64, 160]):
        got, sees = run(keys), torch.zeros(T, dtype=torch.bool, device="cuda")
        for t in keys:
            s = pos >= t
            if "chunk" in kw:
                s &= pos // kw["chunk"] == t // kw["chunk"]
            if "window" in kw:
                s &= (pos - t < kw["window"]) | (t < kw["keep_first"])
            sees |= s
        hit = torch.zeros_like(got, dtype=torch.bool)
        hit[sees, (G - 1) * (H // G):, V - 3] = True
        assert bool((got[~hit] == clean[~hit]).all()) and not bool(torch.isfinite(got[hit]).any())


@pytest.mark.parametrize("H,G,D,V,maps,BS", [(16, 2, 128, 128, 1, 64), (6, 2, 64, 128, 2, 64), (131, 1, 64, 64, 1, 128),
                                             (5, 1, 128, 64, 1, 32)])
@pytest.mark.parametrize("kw", [dict(), dict(window=130, keep_first=70), dict(chunk=100, window=33, keep_first=3),
                                dict(chunk=50, softcap=6.0), dict(scale=0.0)])
def test_tiles_cut_over_their_keys(H, G, D, V, maps, BS, kw, monkeypatch):
    """The same against 64 bits with every 64-key block of a tile in a part of its own."""
    monkeypatch.setattr(S, "MASK_TILE_BLOCKS", 1)
    monkeypatch.setattr(S, "MASK_TILE_FILL", 1 << 20)
    test_prompts(H, G, D, V, maps, BS, kw)


def test_parts_of_a_tile():
    """No block is left out, no part is empty where the list is longest, and a full chip is not cut."""
    for groups in (1, 7, 26, 255, 256, 257, 512, 5000):
        for nblk in (1, 7, 8, 9, 31, 125, 1000):
            n, pb = S._tile_parts(groups, nblk)
            assert n == 1 or (n * pb >= nblk > (n - 1) * pb and pb >= S.MASK_TILE_BLOCKS and n * groups <= S.MASK_TILE_FILL)
    assert S._tile_parts(26, 125)[0] > 8 and S._tile_parts(257, 1000) == (1, 0)


@pytest.mark.parametrize("most", [1 << 30, 40, 5])
def test_keys_that_rows_see(most):
    m = S.SegMeta(3, *[None] * 5, [0, 1, 31, 40], [9, 0, 37], [0] * 3)
    assert [m.keys_behind(f, most) for f in (0, 1, 3)] == [
        sum(min(p + i + 1, most) for p, n in list(zip([9, 0, 37], [1, 30, 9]))[f:] for i in range(n)) for f in (0, 1, 3)]
    assert m.singles() == 1
