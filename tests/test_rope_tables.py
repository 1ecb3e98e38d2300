"""cos | sin of a step's positions made beside the embedding (csrc/kernels/rope_rows.h): the bits of the launch that makes one
table alone, and the embedding's own results as without them."""
import pytest
import torch

from k8s_llm_rca_amd.ops import norm as N
from k8s_llm_rca_amd.ops import seq_ops as S


@pytest.mark.parametrize("dev", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
@pytest.mark.parametrize("T,W", [(1, 2048), (7, 64), (300, 1024), (3, 250)])      # (250: rows by single entries)
@pytest.mark.parametrize("dims", [(), (64,), (128, 30), (2, 64, 96)])
def test_beside_the_embedding(dev, T, W, dims):
    g = torch.Generator().manual_seed(T + W)
    pos = torch.randint(0, 100000, (T,), generator=g, dtype=torch.int32).to(dev)
    ids = torch.randint(0, 50, (T,), generator=g, dtype=torch.int32).to(dev)
    embed, w = torch.randn(50, W, generator=g).to(torch.bfloat16).to(dev), torch.randn(W, generator=g).to(dev)
    ropes = [S.make_rope(d, 10000.0 + d, dev) for d in dims]
    one = torch.ones(1, device=dev)

    def rms(x, tables):
        return N.hyper_embed(ids, embed, 2.0, x.view(T, 1, W), one, w, 1e-5, torch.bfloat16, tables=tables)

    def dyt(x, tables):
        return N.embed_scale_dyt(ids, embed, 2.0, x, 0.5, w, w, torch.bfloat16, tables=tables)
    for embedding in (rms, dyt):
        x0, x1, tables = torch.empty(T, W, device=dev), torch.empty(T, W, device=dev), S.RopeTables(pos, ropes)
        assert torch.equal(embedding(x0, tables), embedding(x1, None)) and torch.equal(x0, x1)
        for r in ropes:
            assert torch.equal(tables.of(r), S.rope_table(pos, r))
    assert S.RopeTables(pos, ropes).of(None) is None
