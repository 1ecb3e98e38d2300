"""Matrix-core attention of single tokens: heads as matrix rows, a row's keys over waves and parts, against 64 bits; and the
same bits whatever the other rows of the step are."""
import math

import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
BF, BS = torch.bfloat16, 64
ENDS = [0, 1, 31, 32, 33, 127, 128, 129, 255, 256, 257, 513, 700, 1399]   # positions: ends of blocks, waves and parts


def meta(pos, pages, dev="cuda"):
    n = len(pos)

    def i32(v):
        return torch.tensor(v, dtype=torch.int32, device=dev)
    return S.SegMeta(n, i32(range(n)), i32(range(n + 1)), i32(pos), i32([0] * n), i32([pages] * n), list(range(n + 1)),
                     list(pos), [0] * n, n_single=n)


def weights(s, vis, sink):
    s = s.masked_fill(~vis, -math.inf)
    if sink is not None:
        s = torch.cat([s, sink.double().view(1, -1, 1).expand(s.shape[0], -1, 1)], -1)
    p = torch.softmax(s, -1)
    return p if sink is None else p[..., :-1]


def close(got, want):
    # the weights are rounded to bf16 (2^-9 each, of both signs) before they meet the values, the result once more
    assert float((got.double().cpu() - want).abs().max()) < 2.0 ** -7 * float(want.abs().max())


@pytest.mark.parametrize("H,G,D,V", [(16, 2, 128, 128), (4, 4, 64, 64), (20, 1, 96, 96), (33, 1, 64, 128), (6, 2, 128, 64)])
@pytest.mark.parametrize("kw", [dict(), dict(window=200, keep_first=40), dict(window=600), dict(window=1), dict(window=2),
                                dict(chunk=150, softcap=8.0), dict(chunk=513, window=90, keep_first=3)])
@pytest.mark.parametrize("extras", [False, True])
def test_masked(H, G, D, V, kw, extras):
    n, dev = 1400, torch.device("cuda")
    g = torch.Generator().manual_seed(D + H)
    pages = torch.randperm(24, generator=g).tolist()
    k, v = (torch.randn(24 * BS, G, d, generator=g).to(BF) for d in (D, V))
    q = (2 * torch.randn(len(ENDS), H, D, generator=g)).to(BF)
    kc, vt = torch.zeros(24, BS, G * D, dtype=BF), torch.zeros(24, G * V, BS, dtype=BF)
    for i in range(n):
        kc[pages[i // BS], i % BS], vt[pages[i // BS], :, i % BS] = k[i].reshape(-1), v[i].reshape(-1)
    sink, gate = (torch.randn(H, generator=g), torch.randn(len(ENDS), H + 1, generator=g)) if extras else (None, None)
    kc, vt, qd = kc.to(dev), vt.to(dev), q.view(len(ENDS), -1).to(dev)
    gd = gate.to(dev)[:, 1:] if extras else None

    def run(rows, **more):
        return S.masked_attention(qd[rows].contiguous(), H, G, D, V, kc, None, meta([ENDS[r] for r in rows], pages),
                                  D ** -0.5, sink=sink.to(dev) if extras else None, gate=gd[rows] if extras else None, vt=vt,
                                  **kw, **more)
    every = list(range(len(ENDS)))
    got = run(every)
    qi, kp = torch.tensor(ENDS)[:, None], torch.arange(n)[None]
    vis = kp <= qi
    if "chunk" in kw:
        vis &= qi // kw["chunk"] == kp // kw["chunk"]
    if "window" in kw:
        vis &= (qi - kp < kw["window"]) | (kp < kw.get("keep_first", 0))
    s = torch.einsum("thd,jhd->thj", q.double(), k[:n].double().repeat_interleave(H // G, 1)) * D ** -0.5
    if "softcap" in kw:
        s = kw["softcap"] * torch.tanh(s / kw["softcap"])
    want = torch.einsum("thj,jhv->thv", weights(s, vis[:, None], sink), v[:n].double().repeat_interleave(H // G, 1))
    if extras:
        want = want * torch.sigmoid(gate[:, 1:].double())[..., None]
    close(got.view(-1, H, V), want)
    for r in (0, 3, 9, 10, 12):              # alone (fewer parts in the step, or none) and beside a long row: the same bits
        assert torch.equal(run([r])[0], got[r]) and torch.equal(run([r, 13])[0], got[r])
    assert torch.equal(run(every, out_f32=True).to(BF), got)
    assert torch.equal(run(every * 40), got.repeat(40, 1))      # past the workgroups that load by lines: the same bits


@pytest.mark.parametrize("H,R,P", [(16, 256, 64), (5, 32, 0), (20, 64, 32), (16, 512, 64), (3, 384, 0), (33, 128, 32)])
@pytest.mark.parametrize("window", [0, 1, 2, 130, 700])
@pytest.mark.parametrize("extras", [False, True])
def test_latent(H, R, P, window, extras):
    n, dev = 1400, torch.device("cuda")
    g = torch.Generator().manual_seed(R + H)
    pages = torch.randperm(24, generator=g).tolist()
    c, kr = torch.randn(n, R, generator=g).to(BF), torch.randn(n, P, generator=g).to(BF)
    q, qr = (torch.randn(len(ENDS), H, d, generator=g).to(BF) for d in (R, P))
    cache, ct = torch.zeros(24, BS, R + P, dtype=BF), torch.zeros(24, R, BS, dtype=BF)
    for i in range(n):
        cache[pages[i // BS], i % BS], ct[pages[i // BS], :, i % BS] = torch.cat([c[i], kr[i]]), c[i]
    scale = 2.0 * (R + P) ** -0.5
    sink, gate = (torch.randn(H, generator=g), torch.randn(len(ENDS), H + 1, generator=g)) if extras else (None, None)
    cache, ct, qd, rd = cache.to(dev), ct.to(dev), q.to(dev), qr.to(dev)

    def run(rows, head_major=True):
        pos = [ENDS[r] for r in rows]
        return S.latent_attention_mfma(qd[rows], cache, ct, gate.to(dev)[rows, 1:] if extras else None, meta(pos, pages),
                                       torch.tensor(pos, dtype=torch.int32, device=dev), scale, qr=rd[rows] if P else None,
                                       window=window, sink=sink.to(dev) if extras else None, head_major=head_major)
    every = list(range(len(ENDS)))
    got = run(every)
    qi, kp = torch.tensor(ENDS)[:, None], torch.arange(n)[None]
    vis = (kp <= qi) & ((qi - kp < window) if window else (kp >= 0))
    s = (torch.einsum("thd,jd->thj", q.double(), c.double()) + torch.einsum("thd,jd->thj", qr.double(), kr.double())) * scale
    want = torch.einsum("thj,jd->thd", weights(s, vis[:, None], sink), c.double())
    if extras:
        want = want * torch.sigmoid(gate[:, 1:].double())[..., None]
    close(got, want)
    for r in (0, 3, 6, 9, 12):
        assert torch.equal(run([r])[0], got[r]) and torch.equal(run([r, 13], head_major=False)[0], got[r])
    assert torch.equal(run(every * 20), got.repeat(20, 1, 1))


def test_score_maps():
    """Two maps a head: each map against its own key head, both against the head's values."""
    g = torch.Generator().manual_seed(5)
    H, G, D, V, M, n = 6, 2, 64, 128, 2, 640
    k, v = torch.randn(n, G, M, D, generator=g).to(BF), torch.randn(n, G, V, generator=g).to(BF)
    q = torch.randn(3, H, M, D, generator=g).to(BF)
    pos, dev = [0, 257, 639], "cuda"
    kc, vt = k.view(10, BS, -1).to(dev), v.view(10, BS, -1).transpose(1, 2).contiguous().to(dev)
    got = S.masked_attention(q.view(3, -1).to(dev), H, G, D, V, kc, None, meta(pos, list(range(10))), 0.125, vt=vt, maps=M,
                             out_f32=True).view(3, H, M, V)
    for t, p in enumerate(pos):
        s = torch.einsum("hmd,jhmd->hmj", q[t].double(), k[:p + 1].double().repeat_interleave(H // G, 1)) * 0.125
        want = torch.einsum("hmj,jhv->hmv", torch.softmax(s, -1), v[:p + 1].double().repeat_interleave(H // G, 1))
        close(got[t], want)


@pytest.mark.parametrize("most", [1, 3, 5])
def test_rows_of_more_keys_than_parts(most, monkeypatch):
    """Parts grow where the count is bounded; the same result as unbounded."""
    g = torch.Generator().manual_seed(1)
    pages, dev = list(range(24)), "cuda"
    kc, vt = (torch.randn(24, *s, generator=g).to(BF).to(dev) for s in ((BS, 128), (128, BS)))
    q = torch.randn(len(ENDS), 4 * 128, generator=g).to(BF).to(dev)
    cache, ct = torch.randn(24, BS, 64, generator=g).to(BF).to(dev), torch.randn(24, 64, BS, generator=g).to(BF).to(dev)
    qa = torch.randn(len(ENDS), 4, 64, generator=g).to(BF).to(dev)
    pos = torch.tensor(ENDS, dtype=torch.int32, device=dev)

    def run():
        return (S.masked_attention(q, 4, 1, 128, 128, kc, None, meta(ENDS, pages), 0.1, vt=vt),
                S.latent_attention_mfma(qa, cache, ct, None, meta(ENDS, pages), pos, 0.2),
                S.latent_attention_mfma(qa, cache, ct, None, meta(ENDS, pages), pos, 0.2, window=900))
    want = run()
    monkeypatch.setattr(S, "TOKEN_PARTS", most)
    for a, b in zip(run(), want):
        close(a, b.double().cpu())


def test_partial_results_within_a_bound(monkeypatch):
    """A step whose partial results pass the bound takes its rows in groups: the same bits, no allocation past the bound."""
    H, G, D, n = 8, 2, 64, len(ENDS)
    g = torch.Generator().manual_seed(9)
    q, kc, vt = (torch.randn(*s, generator=g).to(BF).cuda() for s in ((n, H * D), (24, BS, G * D), (24, G * D, BS)))
    qa, c, ct = (torch.randn(*s, generator=g).to(BF).cuda() for s in ((n, H, D), (24, BS, D), (24, D, BS)))
    m, sizes, scratch = meta(ENDS, list(range(24))), [], S.scratch
    monkeypatch.setattr(S, "scratch", lambda shape, *a: (sizes.append(shape), scratch(shape, *a))[1])

    def run():
        sizes.clear()
        return (S.masked_attention(q, H, G, D, D, kc, None, m, 0.1, vt=vt),
                S.latent_attention_mfma(qa, c, ct, None, m, m.seg_pos0, 0.1), max(sizes))
    a, b, _ = run()
    for limit in (1, 40000, 10 ** 5, 10 ** 9):
        monkeypatch.setattr(S, "TOKEN_SCRATCH", limit)
        x, y, most = run()
        assert torch.equal(x, a) and torch.equal(y, b) and most <= max(limit, H * 11 * D)


@pytest.mark.parametrize("sink", [False, True])
def test_a_query_that_is_not_a_number(sink):
    """All scores NaN: the row's result is, in one part and in many, and no other row's."""
    H, G, D, n = 4, 2, 64, len(ENDS)
    g = torch.Generator().manual_seed(5)
    q, kc, vt = (torch.randn(*s, generator=g).to(BF).cuda() for s in ((n, H * D), (24, BS, G * D), (24, G * D, BS)))
    qa, c, ct = (torch.randn(*s, generator=g).to(BF).cuda() for s in ((n, H, D), (24, BS, D), (24, D, BS)))
    m, s = meta(ENDS, list(range(24))), torch.zeros(H).cuda() if sink else None

    def run():
        return (S.masked_attention(q, H, G, D, D, kc, None, m, 0.1, vt=vt, sink=s).view(n, H, D),
                S.latent_attention_mfma(qa, c, ct, None, m, m.seg_pos0, 0.1, sink=s))
    clean, bad = run(), [1, 7, 13]
    q[bad, :D], qa[bad, 0, 3] = math.nan, math.nan
    hit = torch.zeros(n, H, dtype=torch.bool, device="cuda")
    hit[bad, 0] = True
    for x, y in zip(run(), clean):
        assert bool(torch.isnan(x[hit]).all()) and torch.equal(x[~hit], y[~hit])
