"""The sizes past the first line at which a product takes the residual's pass (ops/row_step.py: into_long), and A and W turned in
the waves' LDS (csrc/kernels/gemm_step.hip): every count of loads with the slots they share, rows up to and past eight."""
import pytest
import torch

from k8s_llm_rca_amd.ops import row_step as R
from k8s_llm_rca_amd.ops._lib import check, lib, ptr, stream_ptr

BF = torch.bfloat16


def test_rule():
    yes = ((9, 2048, 8192), (16, 2048, 8192), (16, 4096, 4096), (16, 6144, 4096), (9, 4096, 8192), (8, 1024, 8192), (16, 512, 4096))
    no = ((12, 4096, 8192), (9, 6144, 8192), (9, 1024, 8192), (8, 512, 8192), (16, 8192, 2048), (17, 2048, 8192), (1, 2048, 16384))
    for m, n, k in yes:
        assert R.into_long(m, n, k) and not R.into_ok(m, n, k)
    for m, n, k in no:
        assert not R.into_long(m, n, k) and not R.into_ok(m, n, k)
    assert R.into_long(16, 2048, 4096, True) and not R.into_long(16, 2048, 2048, True) and not R.into_long(1, 2048, 2048)


@pytest.mark.gpu
@pytest.mark.parametrize("loads", [1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16])
@pytest.mark.parametrize("m", [1, 2, 7, 8, 9, 15, 16])
def test_loads(loads, m):
    n, k = 72, 512 * loads
    g = torch.Generator().manual_seed(loads * 17 + m)
    a, w = torch.randn(m, k + 8, generator=g).to(BF).cuda()[:, :k], (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()
    x0, nw, nb = (torch.randn(*s, generator=g).cuda() for s in ((m, n), (n,), (n,)))
    for rms in (True, False):
        x, h, part = x0.clone(), torch.empty(m, n, device="cuda", dtype=BF), torch.empty(m, n // 8, device="cuda")
        if rms:
            check(lib().k8s_gemm_step_rms(ptr(a), k + 8, ptr(w), ptr(x), 0, 0, 1.0, 0.0, 0, 0, 0.0, ptr(nw), ptr(h), ptr(part), m, n, k,
                                          stream_ptr(x)), "rms")
        else:
            check(lib().k8s_gemm_step_dyt(ptr(a), k + 8, ptr(w), 0.5, 0, 0, 0, 0.0, ptr(x), 0.7, ptr(nw), ptr(nb), ptr(h), m, n, k,
                                          stream_ptr(x)), "dyt")
        want = x0.double() + (1.0 if rms else 0.5) * (a.double() @ w.double().T)
        bound = 4e-6 * (k ** 0.5 + 1)               # fp32 sums of k products of size k^(-1/2) each
        assert float((x.double() - want).abs().max()) < bound
        hw = want * nw.double() if rms else torch.tanh(0.7 * want) * nw.double() + nb.double()
        assert bool(((h.double() - hw).abs() <= 2.0 ** -8 * hw.abs() + 4 * bound).all())       # (weights of up to four)
        if rms:
            sums = (want * want).view(m, n // 8, 8).sum(2)
            assert float((part.double() - sums).abs().max()) < 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,two", [(9, 2048, 8192, False), (16, 2048, 8192, False), (8, 1024, 8192, False), (16, 2048, 4096, True)])
def test_past_the_line(m, n, k, two):
    g = torch.Generator().manual_seed(m + k)
    a, w, a2, w2 = ((torch.randn(*s, generator=g) * f).to(BF).cuda() for s, f in (((m, k), 1), ((n, k), k ** -0.5)) * 2)
    x0, nw, nb = (torch.randn(*s, generator=g).cuda() for s in ((m, n), (n,), (n,)))
    assert R.into_long(m, n, k, two)
    x = x0.clone()
    h = R.dyt_product(x, a, w, 0.75, a2 if two else None, w2 if two else None, 0.5, 0.7, nw, nb, BF)
    want = x0.double() + 0.75 * (a.double() @ w.double().T) + (0.5 * (a2.double() @ w2.double().T) if two else 0)
    bound = 4e-6 * (2 * k ** 0.5 + 1)
    assert float((x.double() - want).abs().max()) < bound
    ref = torch.tanh(0.7 * want) * nw.double() + nb.double()
    assert bool(((h.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 4 * bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,stride", [(3, 64, 3072, 8), (16, 64, 4096, 0), (12, 64, 4096, 2048), (1, 64, 4096, 0)])
def test_rows_that_overlap(m, n, k, stride):
    """Rows of X that share memory go where they went: the kernel takes rows that lie apart, and any single one."""
    assert R.into_long(m, n, k) or R.into_ok(m, n, k)
    g = torch.Generator().manual_seed(m + stride)
    a = torch.randn(m * stride + k, generator=g).to(BF).cuda().as_strided((m, k), (stride, 1))
    w = (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()
    x0, nw, nb = (torch.randn(*s, generator=g).cuda() for s in ((m, n), (n,), (n,)))
    x = x0.clone()
    h = R.dyt_product(x, a, w, 0.5, None, None, 1.0, 0.7, nw, nb, BF)
    want = x0.double() + 0.5 * (a.double() @ w.double().T)
    bound = 4e-6 * (k ** 0.5 + 1)
    ref = torch.tanh(0.7 * want) * nw.double() + nb.double()
    if isinstance(h, R.RowStep):
        h = h.read()
    assert bool(((h.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 4 * bound).all())
