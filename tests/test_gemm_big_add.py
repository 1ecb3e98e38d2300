"""Products added to an fp32 residual in the tile's epilogue (csrc/kernels/gemm_big.hip, MODE 4): rows that end within a tile, a
wave's rows and half a tile; a residual of wider rows; the split last wave; and when it is taken."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops._lib import check, lib, ptr, stream_ptr

BF = torch.bfloat16


def test_rule():
    assert L.big_add_pays(16384, 2048, 2048) and L.big_add_pays(24576, 2048, 2048) and L.big_add_pays(8192, 2048, 8192)
    assert L.big_add_pays(13817, 2048, 2048) and not L.big_add_pays(12025, 2048, 2048) and L.big_add_pays(12025, 2048, 8192)
    assert L.big_add_pays(20473, 2048, 2048) and not L.big_add_pays(17145, 2048, 2048) and not L.big_add_pays(4096, 2048, 2048)
    assert not L.big_add_pays(16384, 2000, 2048) and not L.big_add_pays(16384, 2048, 1024)


@pytest.mark.gpu
@pytest.mark.parametrize("m", [1, 15, 127, 128, 129, 255, 256, 257, 391, 512])
@pytest.mark.parametrize("n,k,wide", [(256, 128, 0), (512, 2048, 0), (256, 256, 24)])
@pytest.mark.parametrize("scale", [1.0, 0.3])
def test_add(m, n, k, wide, scale):
    g = torch.Generator().manual_seed(m + n)
    x, w = torch.randn(m, k, generator=g).to(BF).cuda(), (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()
    r0 = torch.randn(m + 3, n + wide, generator=g).cuda()
    r = r0.clone()
    L.reserve_big_ws(torch.device("cuda", 0))
    check(lib().k8s_gemm_big_add(ptr(x), k, ptr(w), ptr(r), n + wide, m, n, k, scale, stream_ptr(x)), "gemm_big_add")
    want = r0[:m, :n].double() + scale * (x.double() @ w.double().T)
    # fp32 sums of k products of size k^(-1/2) each
    assert float((r[:m, :n].double() - want).abs().max()) < 4e-6 * k ** 0.5 + 1e-6
    assert torch.equal(r[m:], r0[m:]) and torch.equal(r[:, n:], r0[:, n:])      # nothing beside them is written
