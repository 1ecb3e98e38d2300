"""Products of 17 to 64 rows (csrc/kernels/gemm_batch.hip): every count of row fragments and chunks, strips that begin within the one
before, K ranges; and what the rule (ops/linear.py: batch_plan) gives to it."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops._lib import lib, ptr, stream_ptr

BF = torch.bfloat16
OUTS = (L.ROWS_BF16, L.ROWS_F32, L.ROWS_SILU, L.ROWS_RELU2)


def test_rule():
    assert L.batch_plan(64, 8192, 2048, L.ROWS_SILU) == (4, 1) and L.batch_plan(17, 4096, 2048, L.ROWS_SILU) == (2, 1)
    assert L.batch_plan(64, 8192, 2048, L.ROWS_RELU2) == (2, 1) and L.batch_plan(48, 8736, 2048, L.ROWS_F32) == (4, 1)
    assert L.batch_plan(17, 2048, 8192, L.ROWS_F32, True) == (2, 4) and L.batch_plan(48, 2048, 2048, L.ROWS_F32, True) == (2, 4)
    assert L.batch_plan(64, 2560, 2048, L.ROWS_F32, True) == (2, 2)
    for m, n, k, out, planes in ((16, 8192, 2048, 0, False), (65, 8192, 2048, 0, False), (64, 8200, 2048, 0, False),
                                 (64, 8192, 2112, 0, False), (64, 8192, 1024, 2, False), (64, 8736, 2048, 1, False),
                                 (64, 2048, 8192, 1, True), (64, 2048, 2048, 1, True), (64, 32768, 2048, 1, False), (40, 4096, 4096, 0, False)):
        assert L.batch_plan(m, n, k, out, planes) is None
    for m in (17, 32, 33, 64):                  # whatever the rule gives away fits the kernel
        for n in range(16, 20000, 368):
            for k in (512, 768, 1024, 1280, 2048, 3840, 4096, 8192):
                for out, planes in [(o, False) for o in OUTS] + [(L.ROWS_F32, True)]:
                    plan = L.batch_plan(m, n, k, out, planes)
                    if plan is not None:
                        strip = (8 if out == L.ROWS_SILU else 16) * plan[0]
                        assert n >= strip and k % (256 * plan[1]) == 0 and (out != L.ROWS_SILU or n % strip == 0)


def test_planes_rule():
    """Which planes it takes turns on how far K is cut and on the rows, and on both sides of a line for a range of widths."""
    def took(n, k, m):
        return L.batch_plan(m, n, k, L.ROWS_F32, True) is not None
    for n in (512, 640, 768, 896, 1024):                    # eight ranges: at every number of rows
        assert all(took(n, k, m) for k in (2048, 4096, 6144, 8192) for m in (17, 32, 33, 48, 49, 64))
    for n in (1040, 1280, 1536, 2048):                      # four: up to 48 rows
        assert all(took(n, k, m) == (m <= 48) for k in (2048, 3072, 4096, 5120, 8192) for m in (17, 32, 33, 48, 49, 64))
    for n in (512, 1024, 1536, 2048):                       # two, of K that no more divide
        for k, most in ((1536, 32), (2560, 24), (3584, 24), (4608, 0), (5632, 0), (7680, 0)):
            assert all(took(n, k, m) == (m <= most) for m in (17, 24, 25, 32, 33, 48, 64))
    for n in (2064, 2304, 3072, 4096):                      # two that fill the units
        for k, most in ((1024, 32), (2048, 64), (2560, 64), (3584, 64), (4096, 32), (8192, 32)):
            assert all(took(n, k, m) == (m <= most) for m in (17, 32, 33, 48, 64))


def test_long_k_over_few_strips():
    def took(big, k, m):
        return L.batch_plan(m, big // 2, k, L.ROWS_SILU) is not None
    for k, least in ((4096, (0, 0, 0)), (4864, (0, 0, 0)), (5120, (0, 2560, 4096)), (5632, (2048, 2560, 4096)), (8192, (2048, 2560, 4096))):
        for big in (512, 1024, 2048, 2112, 2560, 2624, 4096, 4160, 8192):
            for m, line in ((17, least[0]), (32, least[0]), (33, least[1]), (48, least[1]), (49, least[2]), (64, least[2])):
                assert took(big, k, m) == (big > line), (big, k, m)


def test_more_than_a_wave_of_few_rows():
    """Up to 24 rows the row-streaming kernel keeps what it takes with two fragments; where it has four, or nothing, this one goes on."""
    for out in (L.ROWS_SILU, L.ROWS_RELU2):
        for big in (16384, 16640, 18432, 20480, 24576, 28672, 32768):
            for k in (512, 768, 1024, 1536, 2048, 3072, 4096):
                for m in (17, 24, 25, 32):
                    n = big // 2 if out == L.ROWS_SILU else big
                    left = m <= 24 and 16384 < big <= 24576 and k not in (1536, 3072)
                    assert (L.batch_plan(m, n, k, out) is None) == left, (out, big, k, m)


def check_one(m, n, k, nf, ranges, out, pad=8):
    g = torch.Generator().manual_seed(m + n + k)
    rows = n * (2 if out == L.ROWS_SILU else 1)
    x = torch.randn(m, k + pad, generator=g).to(BF).cuda()[:, :k]
    w = (torch.randn(rows, k, generator=g) / k ** 0.5).to(BF).cuda()
    f32 = out == L.ROWS_F32
    y = torch.full((ranges * m + 1, n), float("nan"), device="cuda", dtype=torch.float32 if f32 else BF)
    assert lib().k8s_gemm_batch(ptr(x), x.stride(0), ptr(w), ptr(y), n, m, n, k, nf, ranges, out, stream_ptr(x)) == 0
    assert bool(torch.isnan(y[ranges * m]).all())                       # nothing behind the last row
    y = y[:ranges * m].view(ranges, m, n).double().sum(0)
    full = x.double() @ w.double().T
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)    # exact products, k fp32 additions
    if out == L.ROWS_SILU:      # gate and up rounded to bf16, the result again; the gate's slope is at most 1.1
        a, u = full[:, :n], full[:, n:]
        want = torch.nn.functional.silu(a) * u
        half = 2.0 ** -8
        tol = (1.1 * (half * a.abs() + bound[:, :n]) * u.abs() + torch.nn.functional.silu(a).abs() * (half * u.abs() + bound[:, n:]))
        tol = 1.01 * tol + half * want.abs() + 1e-6
    elif out == L.ROWS_RELU2:
        want = full.clamp_min(0).square()
        tol = 2.1 * full.abs() * bound + bound * bound + 2.0 ** -8 * want * 1.01
    else:
        want = full
        tol = bound + (0 if f32 else 2.0 ** -8 * full.abs() * 1.01)
    assert bool(((y - want).abs() <= tol).all()), (m, n, k, nf, ranges, out, float((y - want).abs().max()))


@pytest.mark.gpu
@pytest.mark.parametrize("out", OUTS)
@pytest.mark.parametrize("nf", [2, 4])
@pytest.mark.parametrize("m", [1, 17, 32, 33, 48, 49, 64])
def test_against_64_bits(m, nf, out):
    for n, k in ((64, 256), (128, 512), (192, 768), (64, 1024), (128, 1280)):
        check_one(m, n, k, nf, 1, out)
    if out != L.ROWS_SILU:
        check_one(m, 64 + 48, 768, nf, 1, out, pad=0)


@pytest.mark.gpu
@pytest.mark.parametrize("ranges", [2, 4, 8])
@pytest.mark.parametrize("m", [17, 64])
def test_planes(m, ranges):
    check_one(m, 160, 256 * ranges, 2, ranges, L.ROWS_F32)
    check_one(m, 80, 768 * ranges, 4, ranges, L.ROWS_F32)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [17, 40, 64])
def test_entry_points(m):
    """The products that the rule gives to it, against the same rows apart (kernels of up to 16 rows and others)."""
    g = torch.Generator().manual_seed(m)
    x = torch.randn(m, 2048, generator=g).to(BF).cuda()
    w = (torch.randn(8192, 2048, generator=g) / 45).to(BF).cuda()
    for f, out in ((L.glu_proj, L.ROWS_SILU), (L.relu_sq_proj, L.ROWS_RELU2), (L.proj, L.ROWS_BF16), (L.proj_f32out, L.ROWS_F32),
                   (L.linear_f32out, L.ROWS_F32)):
        assert L.batch_plan(m, 8192 // (2 if out == L.ROWS_SILU else 1), 2048, out)
        got, want = f(x, w).float(), torch.cat([f(x[i:i + 16], w) for i in range(0, m, 16)]).float()
        # fp32 sums in another order (1e-5 of entries of size 1), rounded to bf16 up to three times
        assert float((got - want).abs().max()) <= (1e-4 if out == L.ROWS_F32 else 2.0 ** -6 * float(want.abs().max()))
    got, want = L.proj_planes(x, w[:2048]).sum(0), L.proj_f32out(x[:16], w[:2048])
    assert float((got[:16] - want).abs().max()) <= 1e-4


@pytest.mark.gpu
def test_refused():
    x, w, y = (torch.zeros(*s, device="cuda", dtype=BF) for s in ((64, 1024), (128, 1024), (64, 256)))
    ok = [ptr(x), 1024, ptr(w), ptr(y), 128, 64, 128, 1024, 2, 1, 0, stream_ptr(x)]
    assert lib().k8s_gemm_batch(*ok) == 0
    for at, bad in ((0, 0), (0, ptr(x) + 2), (1, 1020), (1, 512), (2, 0), (3, 0), (4, 64), (5, 0), (5, 65), (6, 120), (6, 16), (7, 1088),
                    (8, 1), (8, 3), (9, 0), (9, 2), (9, 8), (10, 4), (10, -1)):
        assert lib().k8s_gemm_batch(*ok[:at], bad, *ok[at + 1:]) != 0, (at, bad)
