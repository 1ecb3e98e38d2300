"""The row-streaming product (csrc/kernels/gemm_rows.hip) at the edges of its forms, and the rule that picks it."""
import json
import os

import pytest
import torch

from k8s_llm_rca_amd.ops import attention as A
from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops._lib import lib, ptr, stream_ptr

BF = torch.bfloat16
gpu = pytest.mark.gpu


def operands(m, n, k):
    g = torch.Generator().manual_seed(m * 7 + n + k)
    return torch.randn(m, k, generator=g).to(BF).cuda(), (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()


#: K a wave's one chunk, two, three (odd) and seven; strips: one, and one short of and past what a card runs at once
SHAPES = [(16, 512), (32, 1024), (64, 1536), (4080, 512), (4128, 512), (128, 3584), (256, 2048)]


@gpu
@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("m", [1, 3, 4, 15, 16, 17, 31, 32])
@pytest.mark.parametrize("nf", [1, 2, 4])
def test_forms_against_float64(m, n, k, nf):
    x, w = operands(m, n, k)
    want = x.double() @ w.double().T
    ran = 0
    for ranges in (1, 2, 4):
        if not L.rows_shape_ok(m, n, k, nf, ranges):
            continue
        ran += 1
        buf = torch.full((ranges * m * n + 64,), 7.0, device="cuda")           # nothing is written behind the planes
        y = buf[:ranges * m * n].view(ranges, m, n)
        L.gemm_rows(x, w, nf, L.ROWS_F32, ranges, out=y)
        # fp32 sums of K terms of size K^(-1/2), in chunks, waves and ranges
        assert float((y.double().sum(0) - want).abs().max()) < 4e-6 * k ** 0.5
        assert bool((buf[ranges * m * n:] == 7.0).all())
    if not L.rows_shape_ok(m, n, k, nf, 1):
        assert lib().k8s_gemm_rows(ptr(x), k, ptr(w), ptr(x), n, m, n, k, nf, 1, 0, stream_ptr(x)) != 0
        return
    ldy = n + 24
    wide = torch.full((m, ldy), 7.0, device="cuda", dtype=BF)
    y = L.gemm_rows(x, w, nf, out=wide[:, :n])
    assert bool(((y.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()) and bool((wide[:, n:] == 7.0).all())
    r = L.gemm_rows(x, w, nf, L.ROWS_RELU2)
    assert bool(((r.double() - want.clamp_min(0) ** 2).abs() <= 2.0 ** -8 * want.clamp_min(0) ** 2 + 1e-4).all())
    if n % (16 * nf) == 0 and L.rows_shape_ok(m, n // 2, k, nf, 1, L.ROWS_SILU):
        # the separate pass's rounding of gate and up: the same bits as from the plain form
        g, u = y[:, :n // 2].float(), y[:, n // 2:].float()
        a = L.gemm_rows(x, w, nf, L.ROWS_SILU).float()
        assert torch.allclose(a, torch.nn.functional.silu(g) * u, rtol=2.0 ** -8, atol=1e-6)


@gpu
def test_rows_of_infinities_stay_by_themselves():
    for m, nf in ((5, 1), (16, 2), (20, 4)):
        x, w = operands(m, 256, 1024)
        clean = L.gemm_rows(x, w, nf)
        x[2, 100] = float("inf")
        w2 = w.clone()
        w2[7, 3] = float("nan")
        y = L.gemm_rows(x, w2, nf)
        keep = [i for i in range(m) if i != 2]
        cols = [i for i in range(256) if i != 7]
        assert torch.equal(y[keep][:, cols], clean[keep][:, cols])
        assert bool(torch.isinf(y[2, cols]).all()) and bool(torch.isnan(y[:, 7]).all())


@gpu
@pytest.mark.parametrize("m,nf", [(1, 1), (3, 2), (16, 4), (17, 2), (32, 4)])
@pytest.mark.parametrize("nq,nkv", [(32, 8), (3, 1)])
def test_rotating_form_is_product_and_rope(m, nf, nq, nkv):
    K, BS, NB = 1024, 64, 4
    N = (nq + 2 * nkv) * 128
    x, w = operands(m, N, K)
    cs = A.rope_cos_sin(4096, 500000.0, device="cuda")
    pos = torch.randint(0, 4000, (m,), device="cuda", dtype=torch.int32)
    slots = torch.randperm(NB * BS, device="cuda")[:m].int()
    if m > 1:
        slots[1] = -1
    kc, vc = torch.zeros(NB, nkv, BS, 128, device="cuda", dtype=BF), torch.zeros(NB, nkv, 128, BS, device="cuda", dtype=BF)
    kc2, vc2 = kc.clone(), vc.clone()
    ref = L.gemm_rows(x, w, nf)
    A.rope_kv_write(ref, pos, cs, slots, kc, vc, nq, nkv)
    out = torch.empty_like(ref)
    assert lib().k8s_gemm_rows_rope(ptr(x), K, ptr(w), ptr(out), N, m, N, K, nf, ptr(pos), ptr(cs), ptr(slots), ptr(kc2),
                                    ptr(vc2), nq, nkv, BS, stream_ptr(x)) == 0
    assert torch.equal(out, ref) and torch.equal(kc2, kc) and torch.equal(vc2, vc)


@gpu
@pytest.mark.parametrize("m", [1, 3, 4])
@pytest.mark.parametrize("mode", ["first", "add", "part"])
@pytest.mark.parametrize("H,nf", [(512, 1), (1536, 2), (4096, 4)])
def test_norm_in_front_is_norm_and_product(m, mode, H, nf):
    I, eps, nq, nkv, BS = 512, 1e-5, 6, 1, 64
    g = torch.Generator(device="cuda").manual_seed(m + H)
    res, x = (torch.randn(m, H, device="cuda", generator=g).to(BF) for _ in range(2))
    part = torch.randn(4, m, H, device="cuda", generator=g) * 0.5
    nw = (torch.rand(H, device="cuda", generator=g) + 0.5).to(BF)
    w = (torch.randn(2 * I, H, device="cuda", generator=g) * 0.02).to(BF)
    y, r = torch.empty(m, H, device="cuda", dtype=BF), res.clone()
    s = stream_ptr(x)
    if mode == "part":
        assert lib().k8s_splitk_addnorm(ptr(part), 4, ptr(r), ptr(nw), ptr(y), m, H, H, eps, s) == 0
    else:
        assert lib().k8s_rmsnorm(ptr(x), ptr(r) if mode == "add" else None, ptr(nw), ptr(y), m, H, H, H, eps, s) == 0
    src = (ptr(x) if mode != "part" else None, H, ptr(part) if mode == "part" else None, 4,
           ptr(res) if mode != "first" else None)
    new = torch.full_like(res, float("nan"))
    dst = ptr(new) if mode != "first" else None
    act = torch.empty(m, I, device="cuda", dtype=BF)
    assert lib().k8s_gemm_rows_norm(*src, dst, ptr(nw), eps, ptr(w), ptr(act), I, m, I, H, nf, None, None, None, None, None,
                                    0, 0, 0, s) == 0
    assert torch.equal(act, L.gemm_rows(y, w, nf, L.ROWS_SILU)) and (mode == "first" or torch.equal(new, r))
    N = (nq + 2 * nkv) * 128
    w = (torch.randn(N, H, device="cuda", generator=g) * 0.02).to(BF)
    cs, pos = A.rope_cos_sin(64, 500000.0, device="cuda"), torch.arange(m, device="cuda", dtype=torch.int32)
    pages = [torch.zeros(2, nkv, *d, device="cuda", dtype=BF) for d in ((BS, 128), (128, BS)) for _ in range(2)]
    outs = [torch.empty(m, N, device="cuda", dtype=BF) for _ in range(2)]
    assert lib().k8s_gemm_rows_rope(ptr(y), H, ptr(w), ptr(outs[0]), N, m, N, H, nf, ptr(pos), ptr(cs), ptr(pos),
                                    ptr(pages[0]), ptr(pages[2]), nq, nkv, BS, s) == 0
    assert lib().k8s_gemm_rows_norm(*src, dst, ptr(nw), eps, ptr(w), ptr(outs[1]), N, m, N, H, nf, ptr(pos), ptr(cs), ptr(pos),
                                    ptr(pages[1]), ptr(pages[3]), nq, nkv, BS, s) == 0
    assert torch.equal(*outs) and torch.equal(*pages[:2]) and torch.equal(*pages[2:])


@gpu
@pytest.mark.parametrize("m", [1, 2, 4])
@pytest.mark.parametrize("planes", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("H,nf", [(512, 1), (4096, 4)])
def test_norm_in_front_of_any_count_of_planes(m, planes, H, nf):
    """Up to four planes are asked for in front of the weights (past the last: it again), more are read behind them."""
    I, eps = 512, 1e-5
    g = torch.Generator(device="cuda").manual_seed(m + H + planes)
    res = torch.randn(m, H, device="cuda", generator=g).to(BF)
    buf = torch.full((planes * m * H + 64,), float("nan"), device="cuda")                 # behind the last plane: not read
    part = buf[:planes * m * H].view(planes, m, H)
    part.copy_(torch.randn(planes, m, H, device="cuda", generator=g) * 0.5)
    nw = (torch.rand(H, device="cuda", generator=g) + 0.5).to(BF)
    w = (torch.randn(2 * I, H, device="cuda", generator=g) * 0.02).to(BF)
    y, r = torch.empty(m, H, device="cuda", dtype=BF), res.clone()
    s = stream_ptr(res)
    assert lib().k8s_splitk_addnorm(ptr(part), planes, ptr(r), ptr(nw), ptr(y), m, H, H, eps, s) == 0
    new, act = torch.full_like(res, float("nan")), torch.empty(m, I, device="cuda", dtype=BF)
    assert lib().k8s_gemm_rows_norm(None, H, ptr(part), planes, ptr(res), ptr(new), ptr(nw), eps, ptr(w), ptr(act), I, m, I, H,
                                    nf, None, None, None, None, None, 0, 0, 0, s) == 0
    assert torch.equal(new, r) and torch.equal(act, L.gemm_rows(y, w, nf, L.ROWS_SILU))


def test_rule_gives_what_the_kernel_takes():
    """Every plan fits the kernel; past its rows and sizes there is none."""
    for out in (L.ROWS_BF16, L.ROWS_F32, L.ROWS_SILU, L.ROWS_RELU2):
        for m in (0, 1, 7, 16, 17, 32, 33):
            for n in (8, 16, 100, 128, 264, 1088, 2048, 2576, 5120, 8192, 28672, 128256):
                for k in (256, 512, 768, 1024, 1536, 2048, 4096, 8192, 14336):
                    for planes in ((False, True) if out == L.ROWS_F32 else (False,)):
                        p = L.rows_plan(m, n, k, out, planes)
                        assert p is None or L.rows_shape_ok(m, n, k, p[0], p[1], out), (out, m, n, k, p)
                        if m in (0, 33) or k < 512 or n % 8:
                            assert p is None
    assert L.rows_plan(1, 2048, 2048, L.ROWS_F32, True)[1] > 1 == L.rows_plan(1, 4096, 4096, L.ROWS_F32, True)[1]
    assert L.rows_plan(1, 8192, 8192) is None and L.rows_plan(24, 4096, 4096) is None and L.rows_plan(24, 8192, 2048)


def test_rows_of_weights_on_the_same_channels():
    """A K of 16 KB a row: another kernel is the quicker one until the columns are many; neighbouring K are taken."""
    for out in (L.ROWS_BF16, L.ROWS_F32, L.ROWS_RELU2):
        for m in (17, 24, 32):
            assert L.rows_plan(m, 8192, 8192, out) is None and L.rows_plan(m, 16384, 8192, out) is None
            assert L.rows_plan(m, 28672, 8192, out) and L.rows_plan(m, 16384, 6144, out) and L.rows_plan(m, 16384, 10240, out)
            assert L.rows_plan(m, 28672, 16384, out) is None
        assert L.rows_plan(8, 16384, 8192, out) and L.rows_plan(8, 4096, 8192, out) and L.rows_plan(8, 4096, 16384, out)
        assert L.rows_plan(8, 9216, 8192, out) is None and L.rows_plan(8, 9216, 6144, out)
        assert L.rows_plan(8, 8192, 16384, out) is None and L.rows_plan(16, 28672, 16384, out) is None
    assert L.rows_plan(8, 6144, 8192) is None and L.rows_plan(8, 4608, 8192, L.ROWS_SILU)
    assert L.rows_plan(32, 8192, 8192, L.ROWS_SILU) is None and L.rows_plan(32, 14336, 8192, L.ROWS_SILU)
    assert L.rows_plan(1, 8192, 16384) and L.rows_plan(1, 8192, 16384, L.ROWS_F32) is None
    assert L.rows_plan(24, 57344, 8192) and L.rows_plan(25, 57344, 8192) is None


def test_few_workgroups_are_left_to_other_kernels():
    """Four fragments are all that fits where K is no multiple of 512: taken with columns enough."""
    for k in (768, 1280, 1792, 2816, 3840):
        for m in (1, 4, 16):
            for n in (128, 1088, 2560, 4096):
                assert L.rows_plan(m, n, k) is None and L.rows_plan(m, n, k, L.ROWS_F32, True) is None
                assert L.rows_plan(m, n, k, L.ROWS_RELU2) is None
            assert L.rows_plan(m, 16384, k) and L.rows_plan(m, 2560, k, L.ROWS_SILU)
        assert L.rows_plan(1, 8192, k) is None and L.rows_plan(2, 8192, k)
        assert L.rows_plan(32, 2048, k, L.ROWS_F32, True) is None
    assert L.rows_plan(16, 2560, 1024) and L.rows_plan(32, 2048, 1024, L.ROWS_F32, True)
    assert L.rows_plan(16, 128, 3584, L.ROWS_F32, True) is None and L.rows_plan(8, 128, 3584, L.ROWS_F32, True)
    assert L.rows_plan(32, 8736, 4096) is None and L.rows_plan(32, 8736, 2048) and L.rows_plan(16, 8736, 4096)


def test_tables_take_the_kernel_where_it_was_the_quicker():
    seen = 0
    for name in os.listdir(L.DATA_DIR):
        if not name.startswith("gemm_dispatch_"):
            continue
        with open(os.path.join(L.DATA_DIR, name)) as f:
            shapes = json.load(f)["shapes"]
        for key, rows in shapes.items():
            for r in (r for r in rows if r["kind"] == "rows"):
                n, k = (int(v) for v in key.split(","))
                seen += 1
                assert r["t_us"] < r["lib_us"] and L.rows_shape_ok(r["m"], n, k, r["cfg"], r["splits"]), (name, key, r)
    assert seen


@gpu
def test_operands_the_kernel_cannot_read_go_elsewhere():
    """Rows that do not start on 16 bytes, a transposed weight: the same values as before, by another kernel."""
    x, w = operands(5, 512, 1024)
    want = x.double() @ w.double().T
    odd = torch.empty(5, 1032, device="cuda", dtype=BF)[:, 4:1028]
    odd.copy_(x)
    flat = torch.empty(512 * 1024 + 4, device="cuda", dtype=BF)[4:].view(512, 1024)
    flat.copy_(w)
    for a, b in ((odd, w), (x, flat), (x, w.t().contiguous().t())):
        assert not L.rows_ok(a, b)
        for f in (L.linear, L.proj):
            assert bool(((f(a, b).double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
        assert float((L.proj_planes(a, b).double().sum(0) - want).abs().max()) < 4e-6 * 32


@gpu
def test_gated_operands_the_kernel_cannot_read_go_elsewhere(monkeypatch):
    """The gated form of a table entry, on operands that do not start on 16 bytes; and what the entry points refuse."""
    m, i, k = 5, 256, 1024
    monkeypatch.setitem(L._dispatch, (2 * i, k), [(32, "rows", 2, 1)])
    x, w = operands(m, 2 * i, k)
    assert L.swiglu_choice(m, 2 * i, k) == (L.KIND_ROWS, 2, 1) and L.swiglu_gemm(x, w) is not None
    want = L.glu_proj(x, w)
    odd = torch.empty(m, k + 8, device="cuda", dtype=BF)[:, 4:k + 4]
    odd.copy_(x)
    flat = torch.empty(2 * i * k + 4, device="cuda", dtype=BF)[4:].view(2 * i, k)
    flat.copy_(w)
    for a, b in ((odd, w), (x, flat)):
        assert L.swiglu_gemm(a, b) is None
        # the plain product's sums in another order: a bf16 bit of gate and up
        assert torch.allclose(L.glu_proj(a, b).float(), want.float(), rtol=2.0 ** -6, atol=2.0 ** -9)
    s, y = stream_ptr(x), torch.empty(m, 2 * i, device="cuda", dtype=BF)
    ok = [ptr(x), k, ptr(w), ptr(y), 2 * i, m, 2 * i, k, 2, 1, 0, s]
    assert lib().k8s_gemm_rows(*ok) == 0
    for at, bad in ((0, None), (0, ptr(odd)), (1, k - 8), (1, k + 4), (2, None), (2, ptr(flat)), (3, None), (4, 2 * i - 16)):
        assert lib().k8s_gemm_rows(*ok[:at], bad, *ok[at + 1:]) != 0
    one = ok[:5] + [1] + ok[6:]
    assert lib().k8s_gemm_rows(*one[:1], 0, *one[2:]) == 0                 # one row has no stride


@gpu
@pytest.mark.parametrize("m", [24, 32])
@pytest.mark.parametrize("ld,first", [(512, 0), (519, 0), (520, 0), (520, 4)])
def test_sums_of_ranges_only_where_they_can_be_stored(m, ld, first, monkeypatch):
    """A table's K ranges end in 16-byte stores: a result with other rows or another start is left to another kernel."""
    n, k = 512, 1024
    monkeypatch.setitem(L._dispatch, (n, k), [(32, "rows", 2, 2)])
    x, w = operands(m, n, k)
    want = x.double() @ w.double().T
    buf = torch.full((m * ld + 16,), 7.0, device="cuda", dtype=BF)
    out = buf[first:first + m * ld].view(m, ld)[:, :n]
    ranges = ld % 8 == 0 == first % 8
    assert (L.select_gemm(m, n, k, True, True, True, ranges) == (L.KIND_ROWS, 2, 2)) == ranges
    L.linear(x, w, out=out)
    assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
    kept = torch.ones_like(buf, dtype=torch.bool)
    kept[first:first + m * ld].view(m, ld)[:, :n] = False
    assert bool((buf[kept] == 7.0).all())
    part = torch.zeros(2, m, n, device="cuda")
    s = stream_ptr(x)
    assert (lib().k8s_gemm_stream_reduce(ptr(part), 2, ptr(out), ld, m, n, s) == 0) == ranges


@gpu
def test_prompts_do_not_pay_for_the_rule(monkeypatch):
    """Past the kernel's rows neither the operands nor the rule are looked at: a small prompt's step is host time."""
    def asked(*a, **k):
        raise AssertionError("asked")
    x, w = operands(L.ROWS_MAX_M + 1, 512, 1024)
    monkeypatch.setattr(L, "rows_ok", asked)
    monkeypatch.setattr(L, "row_cut", asked)
    for f in (L.linear, L.linear_f32out, L.proj_f32out, L.proj_planes, L.relu_sq_proj, L.glu_proj):
        f(x, w)


@gpu
def test_executor_with_the_norms_in_front_of_both_products():
    """One and two rows: the norm in front of the rotated and the gated product, the latter on the widest strips (whatever the
    table says); three and four: apart.  The same bits as all apart, and as without the executor."""
    from k8s_llm_rca_amd.models.config import get_config
    from k8s_llm_rca_amd.models.llama import LlamaModel
    from k8s_llm_rca_amd.ops import layer_exec as LX
    from tests.test_tp_gpu import _prefill_inputs
    keys = [(1536, 512), (2048, 512), (512, 1024)]
    saved, fuse0 = {k: L._dispatch.get(k) for k in keys}, LX._norm_fuse
    try:
        L._dispatch[(1536, 512)] = L._dispatch[(2048, 512)] = [(16, "rows", 1, 1)]
        L._dispatch[(512, 1024)] = [(16, "rows", 1, 2)]
        m = LlamaModel(get_config("tiny-llama", n_layers=2, init_std=0.08), "cuda:0", BF, None, seed=4)
        for T in (1, 2, 3, 4):
            got = {}
            for mode in ("fused", "apart", "python"):
                LX._norm_fuse = mode == "fused"
                LX.set_enabled(mode != "python")
                inp, kc, vc = _prefill_inputs(m, T, seed=T)
                got[mode] = m.forward(inp, kc, vc).float().cpu(), kc.float().cpu()
                if mode == "fused":
                    assert m._exec.st.norm_fuse == (3 if T <= LX.NORM_FUSE_ROWS_T else 0)
                    assert m._exec.st.sel[2].cfg == (4 if T <= LX.NORM_FUSE_ROWS_T else 1)
            for a, b in zip(got["fused"], got["apart"]):
                assert torch.equal(a, b)
            for a, b in zip(got["fused"], got["python"]):
                assert torch.equal(a, b)
    finally:
        LX._norm_fuse = fuse0
        LX.set_enabled(True)
        for k, v in saved.items():
            L._dispatch.pop(k, None)
            if v is not None:
                L._dispatch[k] = v
