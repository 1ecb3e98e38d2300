"""Library products of which whole waves of tiles go into a launch of their own (ops/linear.py: row_cut), and those that
gemm_big adds to the residual."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L

BF = torch.bfloat16


def test_cut_is_whole_waves_of_tiles():
    for n, k in [(2048, 2048), (2048, 8192), (8192, 2048), (2560, 2048), (8736, 2048), (3072, 768), (384, 384), (100, 64),
                 (65536, 512), (70000, 512)]:
        nt = -(-n // 256)
        for m in list(range(1, 700, 37)) + [1024, 2047, 2049, 4123, 8192, 8193, 16500, 24576, 24730, 32768]:
            cut = L.row_cut(m, n, k)
            assert 0 <= cut < m and cut % 256 == 0
            assert cut // 256 * nt <= -(-m // 256) * nt // 256 * 256          # no more tiles than the whole waves hold
            parts = L._row_parts(m, n, k)
            assert parts[0][0] == 0 and parts[-1][1] == m and all(a < b for a, b in parts)
    assert L.row_cut(24730, 2048, 2048) == 24576 and L.row_cut(20000, 2048, 2048) == 0
    assert L.row_cut(540, 32768, 4096) == L.row_cut(1061, 32768, 4096) == 0 and L.row_cut(1600, 32768, 4096) == 1536
    assert L.row_cut(19744, 8192, 512) == 0 and L.row_cut(19744, 8192, 2048) and L.row_cut(2100, 8192, 512) == 2048
    for m, n, k in ((1704, 28672, 256), (11027, 8736, 4096), (14181, 1088, 512)):
        assert L.row_cut(m, n, k) == 0
    assert L.row_cut(27000, 2560, 2048) and L.row_cut(6341, 2576, 2048)
    assert L.row_cut(20000, 2048, 8192) == 16384 and L.row_cut(16384, 2048, 8192) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(2049, 8192, 512), (4100, 4096, 256), (8450, 2048, 384)])
def test_cut_products_against_float64(m, n, k):
    assert L.row_cut(m, n, k)
    g = torch.Generator().manual_seed(m)
    wide = torch.randn(m, k + 64, generator=g).to(BF).cuda()
    x, w = wide[:, :k], (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()      # rows apart
    want = x.double() @ w.double().T
    buf = torch.full((m + 1, n), 7.0, device="cuda")
    y = L.linear_f32out(x, w)
    assert float((y.double() - want).abs().max()) < 4e-6 * k ** 0.5                       # fp32 sums of K terms of K^(-1/2)
    r = buf[:m]
    old, L.ADD_ROWS = L.ADD_ROWS, 0
    try:
        assert L.proj_add(r, x, w, 0.5) is None
    finally:
        L.ADD_ROWS = old
    assert float((r.double() - 7.0 - 0.5 * want).abs().max()) < 4e-6 * k ** 0.5 and bool((buf[m] == 7.0).all())
    out = torch.full((m, n + 16), 3.0, device="cuda", dtype=BF)
    b = L.lib_gemm(x, w, out[:, :n])
    assert bool(((b.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()) and bool((out[:, n:] == 3.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,lda", [(6200, 2048, 2048, 2048), (6144, 2304, 2048, 2112), (50100, 256, 2048, 2048),
                                       (8191, 2048, 2048, 2056), (200, 512, 256, 256), (1, 256, 128, 128)])
def test_gemm_big_adds_to_the_residual(m, n, k, lda):
    g = torch.Generator().manual_seed(m + n)
    x = torch.randn(m, lda, generator=g).to(BF).cuda()[:, :k]
    w = (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()
    want = x.double() @ w.double().T
    buf = torch.randn(m + 1, n, generator=g).cuda()
    before = buf.clone()
    L.check(L.lib().k8s_gemm_big_add(L.ptr(x), lda, L.ptr(w), L.ptr(buf), n, m, n, k, 0.5, L.stream_ptr(x)), "add")
    assert float((buf[:m].double() - before[:m].double() - 0.5 * want).abs().max()) < 4e-6 * k ** 0.5
    assert torch.equal(buf[m], before[m])
    if m >= L.ADD_ROWS and k >= 2048:
        assert L.big_add_pays(m, n, k)
        r = before[:m].clone()
        assert L.proj_add(r, x, w, 0.5) is None and torch.equal(r, buf[:m])
    assert L.lib().k8s_gemm_big_add(L.ptr(x), lda, L.ptr(w), L.ptr(buf), n, m, n - 128, k, 0.5, L.stream_ptr(x)) != 0


def test_fused_epilogues_count_rows_not_tiles():
    """Past the general line a fused epilogue wants the rows to fill the waves, not tiles that end early."""
    for silu, n in ((True, 8192), (False, 16384)):
        assert not L.big_tiles_fill(274, n, silu, 1024) and L.big_tiles_fill(512, n, silu, 1024)
        assert not L.big_tiles_fill(537, 2 * n, silu, 2048) and L.big_tiles_fill(768, 2 * n, silu, 2048)
        assert L.big_tiles_fill(1, 4 * n, silu, 1024)                        # whole waves of tiles, as ever
        assert not L.big_tiles_fill(768, 2 * n, silu, 4096)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(4300, 4096, 2048), (200, 4096, 2048), (1540, 4096, 8192), (1, 256, 8192)])
def test_gemm_big_adds_tiles_that_are_split(m, n, k):
    """A last wave in slices of K: the last to arrive adds the sum of all to the residual, once."""
    g = torch.Generator().manual_seed(m + k)
    x = torch.randn(m, k + 8, generator=g).to(BF).cuda()[:, :k]
    w = (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()
    want = x.double() @ w.double().T
    before = torch.randn(m + 1, n, generator=g).cuda()

    def add():
        r = before.clone()
        L.check(L.lib().k8s_gemm_big_add(L.ptr(x), k + 8, L.ptr(w), L.ptr(r), n, m, n, k, 0.5, L.stream_ptr(x)), "add")
        return r

    dev = torch.device("cuda", torch.cuda.current_device())
    try:
        L.reserve_big_ws(dev, enable=False)
        whole = add()
        L.reserve_big_ws(dev, enable=True)              # (the next launch claims the slices' memory for its stream)
        split = [add() for _ in range(3)]
    finally:
        L.reserve_big_ws(dev)
    assert all(torch.equal(s, split[0]) for s in split) and not torch.equal(split[0], whole)
    for r in (whole, split[0]):
        assert float((r[:m].double() - before[:m].double() - 0.5 * want).abs().max()) < 4e-6 * k ** 0.5
        assert torch.equal(r[m], before[m])
