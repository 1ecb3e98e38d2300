"""fp32 results of 17 to 64 rows on the stream kernel (csrc/kernels/gemm_stream.hip, act 2), columns that are no whole number of
strips included; and what its rule leaves to the library."""
import pytest
import torch

from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops._lib import check, lib, ptr, stream_ptr

BF = torch.bfloat16


def test_rule():
    assert L.stream_f32_cfg(40, 2576, 2048) == 34 and L.stream_f32_cfg(17, 8192, 1024) == 34
    assert L.stream_f32_cfg(64, 8736, 2048) == 14 and L.stream_f32_cfg(33, 32768, 2048) == 14
    for m, n, k in ((16, 4096, 2048), (65, 4096, 2048), (40, 2288, 2048), (40, 4104, 2048), (40, 4096, 2080), (40, 4096, 4096),
                    (40, 4096, 960), (40, 24576, 2048), (40, 50256, 2048)):
        assert L.stream_f32_cfg(m, n, k) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("M", [17, 32, 33, 64])
@pytest.mark.parametrize("N,K", [(2576, 2048), (2304, 1024), (8192, 1088), (8208, 1024), (16384, 1024), (32768, 1024)])
def test_against_64_bits(M, N, K):
    g = torch.Generator().manual_seed(M + N)
    x = torch.randn(M, K + 8, generator=g).to(BF).cuda()[:, :K]
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(BF).cuda()
    assert L.stream_f32_cfg(M, N, K)
    out = torch.full((M + 1, N), float("nan"), device="cuda")
    check(lib().k8s_gemm_stream_f32(ptr(x), x.stride(0), ptr(w), ptr(out), M, N, K, L.stream_f32_cfg(M, N, K), stream_ptr(x)), "f32")
    assert bool(torch.isnan(out[M]).all())                  # nothing behind the last row
    want = x.double() @ w.double().T
    # exact products of bf16, K fp32 additions of partly cancelling terms
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((out[:M].double() - want).abs() <= bound).all())
    got = L.proj_f32out(x, w)
    assert got.shape == (M, N) and bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.gpu
def test_no_result_is_refused():
    x, w = torch.zeros(20, 1024, device="cuda").to(BF), torch.zeros(2304, 1024, device="cuda").to(BF)
    for out, n in ((None, 2304), (x, 24), (x, 2312)):
        assert lib().k8s_gemm_stream_f32(ptr(x), 1024, ptr(w), ptr(out), 20, n, 1024, 34, stream_ptr(x)) != 0
    assert lib().k8s_gemm_stream_part(ptr(x), 1024, ptr(w), None, 2304, 20, 2304, 1024, 34, 1, ptr(x), stream_ptr(x)) != 0
