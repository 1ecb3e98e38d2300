"""The vector-pipe attention over paged keys: parts of 128 visible keys spread over workgroups against the same parts walked
by one workgroup (the same bits), and against 64 bits, at part borders, odd sizes and more heads than a workgroup has."""
import math

import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
BS = 32


def meta(lens, pos0, pages, dev):
    row0 = [0]
    for n in lens:
        row0.append(row0[-1] + n)

    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device=dev)
    return S.SegMeta(len(lens), i32([s for s, n in enumerate(lens) for _ in range(n)]), i32(row0), i32(pos0),
                     i32([0] * len(lens)), i32([pages] * len(lens)), row0, list(pos0), [0] * len(lens))


def weights(s, vis, sink):
    s = s.masked_fill(~vis, -math.inf)
    if sink is None:
        return torch.softmax(s, -1)
    return torch.softmax(torch.cat([s, sink.double().view(1, -1, 1).expand(s.shape[0], -1, 1)], -1), -1)[..., :-1]


@pytest.mark.parametrize("H,G,D,V,maps,dt", [(16, 2, 128, 128, 1, torch.float32), (3, 1, 7, 5, 1, torch.float32),
                                             (18, 1, 20, 12, 1, torch.float32), (4, 2, 12, 300, 2, torch.float32),
                                             (6, 3, 36, 48, 1, torch.bfloat16)])
@pytest.mark.parametrize("kw", [dict(), dict(window=200, keep_first=9), dict(chunk=150, softcap=8.0)])
def test_masked_rows(H, G, D, V, maps, dt, kw):
    n, dev = 700, torch.device("cuda")
    g = torch.Generator().manual_seed(D)

    def rnd(*shape):
        return torch.randn(*shape, generator=g)
    HQ, pages = H * maps, torch.randperm(22, generator=g).tolist()
    q, k, v = rnd(n, HQ * D).to(dt), rnd(n, G * maps, D).to(dt), rnd(n, G, V).to(dt)
    kc, vc = torch.full((22, BS, G * maps * D), 7.0, dtype=dt), torch.full((22, BS, G * V), 7.0, dtype=dt)
    for i in range(n):
        kc[pages[i // BS], i % BS], vc[pages[i // BS], i % BS] = k[i].reshape(-1), v[i].reshape(-1)
    sink, gate = rnd(HQ), rnd(n, HQ + 1)
    scale = D ** -0.5
    on = dict(kc=kc.to(dev), vc=vc.to(dev), scale=scale, sink=sink.to(dev), maps=maps, **kw)

    def run(a, b):
        return S.masked_attention(q[a:b].to(dev), H, G, D, V, seg=meta([b - a], [a], pages, dev),
                                  gate=gate[a:b, 1:].to(dev), **on)
    full = run(0, n)                                    # rows enough: a workgroup walks its row's parts
    rows = [0, 127, 128, 129, 255, 256, 383, 384, 511, 640, 699]
    for r in rows:                                      # alone: a workgroup per part
        assert torch.equal(run(r, r + 1)[0], full[r])
    for a, b in ((600, 624), (100, 160), (690, 700)):   # workgroups with eight heads of a part, and on both sides of the line
        assert torch.equal(run(a, b), full[a:b])
    qi, kp = torch.arange(n)[:, None], torch.arange(n)[None]
    vis = kp <= qi
    if kw.get("chunk"):
        vis &= qi // kw["chunk"] == kp // kw["chunk"]
    if kw.get("window"):
        vis &= (qi - kp < kw["window"]) | (kp < kw["keep_first"])
    kk = k.double().view(n, G, maps, D).repeat_interleave(H // G, 1).reshape(n, HQ, D)
    vv = v.double().repeat_interleave(HQ // G, 1)
    s = torch.einsum("thd,jhd->thj", q.double().view(n, HQ, D)[rows], kk) * scale
    if kw.get("softcap"):
        s = kw["softcap"] * torch.tanh(s / kw["softcap"])
    p = weights(s, vis[rows][:, None], sink)
    want = torch.einsum("thj,jhv->thv", p, vv) * torch.sigmoid(gate[rows, 1:].double())[..., None]
    # fp32 sums of D and up to 700 terms, weights of scores of a few units; bf16 inputs are exact, the result is rounded
    tol = 2e-5 if dt == torch.float32 else 2.0 ** -8
    assert float((full[rows].double().cpu().view_as(want) - want).abs().max()) < tol * float(want.abs().max())


@pytest.mark.parametrize("H,R,P", [(16, 256, 64), (5, 24, 0), (11, 300, 12), (2, 33, 7)])
@pytest.mark.parametrize("window", [0, 130])
def test_latent_rows(H, R, P, window):
    n, dev = 400, torch.device("cuda")
    g = torch.Generator().manual_seed(R)

    def rnd(*shape):
        return torch.randn(*shape, generator=g)
    pages = torch.randperm(13, generator=g).tolist()
    qa, qr, c = rnd(n, H, R), rnd(n, H, P) if P else None, rnd(n, R + P)
    cache = torch.full((13, BS, R + P), 7.0)
    for i in range(n):
        cache[pages[i // BS], i % BS] = c[i]
    sink, gate, scale, cache = rnd(H), rnd(n, H), (R + P) ** -0.5, cache.to(dev)

    def run(a, b):
        return S.latent_attention(qa[a:b].to(dev), cache, gate[a:b].to(dev), meta([b - a], [a], pages, dev), scale,
                                  torch.float32, qr=qr[a:b].to(dev) if P else None, window=window, sink=sink.to(dev),
                                  head_major=True)
    full = run(0, n)
    rows = [0, 127, 128, 129, 256, 399]
    for r in rows:
        assert torch.equal(run(r, r + 1)[0], full[r])
    for a, b in ((320, 360), (396, 400)):
        assert torch.equal(run(a, b), full[a:b])
    s = torch.einsum("thr,jr->thj", torch.cat([qa, qr], -1).double()[rows] if P else qa.double()[rows], c.double()) * scale
    dist = torch.tensor(rows)[:, None] - torch.arange(n)[None]
    vis = (dist >= 0) & (dist < window) if window else dist >= 0
    p = weights(s, vis[:, None], sink)
    want = torch.einsum("thj,jr->thr", p, c[:, :R].double()) * torch.sigmoid(gate[rows].double())[..., None]
    assert float((full[rows].double().cpu() - want).abs().max()) < 2e-5 * float(want.abs().max())


def test_partial_results_stay_bounded(monkeypatch):
    """Past ROWS_SCRATCH floats of partial results a workgroup walks its row's parts itself: the same bits."""
    n, H, D, dev = 300, 4, 16, torch.device("cuda")
    g = torch.Generator().manual_seed(2)
    q, kc, vc = (torch.randn(*s, generator=g).to(dev) for s in ((3, H * D), (11, BS, D), (11, BS, D)))
    seg = meta([3], [n], [list(range(11))[:10]], dev)
    args = (q, H, 1, D, D, kc, vc, seg, D ** -0.5)
    assert S._rows_parts(seg, 3, H, H, D, dev)[0] == 3
    a = S.masked_attention(*args)
    monkeypatch.setattr(S, "ROWS_SCRATCH", 3 * H * 3 * (D + 2) - 1)
    assert S._rows_parts(seg, 3, H, H, D, dev)[0] == 0
    assert torch.equal(a, S.masked_attention(*args))


@pytest.mark.parametrize("alone", [True, False])
@pytest.mark.parametrize("n", [1, 3, 130, 258])
def test_infinite_keys_and_values(n, alone):
    """An infinite value of the last visible key makes its column infinite, and keys whose scores are all minus infinity weigh
    nothing beside others -- by themselves, in a part of their own or as a whole part in front."""
    H, D, pages, dev = 2, 8, 10, "cuda"
    g = torch.Generator().manual_seed(n)
    q, k, v = (torch.randn(n, H * D, generator=g) for _ in range(3))
    q[:, ::D] = 1.0
    k[:128, ::D] = -math.inf                              # rows up to 127 see nothing else
    v[n - 1, 3] = math.inf
    kc, vc = torch.zeros(pages, BS, H * D), torch.zeros(pages, BS, H * D)
    kc.view(-1, H * D)[:n], vc.view(-1, H * D)[:n] = k, v
    first = n - 1 if alone else 0
    got = S.masked_attention(q[first:].to(dev), H, H, D, D, kc.to(dev), vc.to(dev),
                             meta([n - first], [first], list(range(pages)), dev), 1.0, sink=torch.zeros(H).to(dev))
    s = torch.einsum("thd,nhd->thn", q.double().nan_to_num(0).view(n, H, D), k.double().view(n, H, D).clamp(-1e300, 1e300))
    p = weights(s.masked_fill(s < -1e200, -math.inf), (torch.arange(n)[None] <= torch.arange(n)[:, None])[:, None], torch.zeros(H))
    want = torch.einsum("thn,nhd->thd", p, v.double().nan_to_num(0, 0, 0).view(n, H, D)).reshape(n, -1)
    if n > 128:
        want[n - 1, 3] = math.inf
        assert torch.equal(torch.isinf(got.cpu()), torch.isinf(want[first:]))
    else:                                                 # a weight of zero: the column is not a number, the others are zero
        want[n - 1, 3] = math.nan
        assert torch.equal(torch.isnan(got.cpu()), torch.isnan(want[first:]))
    ok = torch.isfinite(want[first:])
    assert float((got.cpu().double() - want[first:])[ok].abs().max()) < 1e-5


@pytest.mark.parametrize("H", [1, 2, 4, 5, 7])
def test_keys_of_neighbouring_lanes(H):
    """Every count of keys in a part, heads that do not fill the lanes of a key."""
    n, D, dev = 700, 8, torch.device("cuda")
    g = torch.Generator().manual_seed(H)
    q, k, v = (torch.randn(n, h * D, generator=g) for h in (H, 1, 1))
    kc, vc = torch.full((22, BS, D), math.nan), torch.full((22, BS, D), math.nan)      # (slots without a key are not read)
    kc.view(-1, D)[:n], vc.view(-1, D)[:n] = k, v
    seg = meta([n], [0], list(range(22)), dev)
    got = S.masked_attention(q.to(dev), H, 1, D, D, seg=seg, kc=kc.to(dev), vc=vc.to(dev), scale=D ** -0.5)
    rows = torch.arange(0, 270)
    vis = torch.arange(n)[None] <= rows[:, None]
    s = torch.einsum("thd,jd->thj", q.double().view(n, H, D)[rows], k.double()) * D ** -0.5
    want = torch.einsum("thj,jv->thv", weights(s, vis[:, None], None), v.double())
    # fp32 sums of 8 and up to 270 terms
    assert float((got.cpu().double().view(n, H, D)[rows] - want).abs().max()) < 2e-5 * float(want.abs().max())
