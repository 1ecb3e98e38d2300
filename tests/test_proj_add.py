"""Output projections that add to the residual themselves: the product against 64 bits, and whole models with every step, no
step and single prompts on that path."""
import pytest
import torch

from k8s_llm_rca_amd.engine.engine import EngineConfig, LLMEngine
from k8s_llm_rca_amd.ops import linear as L

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (129, 256, 512), (300, 100, 72), (6144, 128, 256), (6143, 128, 256)])
@pytest.mark.parametrize("scale", [1.0, 0.25])
@pytest.mark.parametrize("rows", [1, L.ADD_ROWS])
def test_product(m, n, k, scale, rows, monkeypatch):
    monkeypatch.setattr(L, "ADD_ROWS", rows)
    g = torch.Generator().manual_seed(m + n + k)
    x, w = torch.randn(m, k, generator=g).to(BF), (torch.randn(n, k, generator=g) * k ** -0.5).to(BF)
    r = torch.randn(m, n, generator=g)
    on = r.clone().cuda()
    y = L.proj_add(on, x.cuda(), w.cuda(), scale)
    p = x.double() @ w.double().T
    bound = 4e-6 * k ** 0.5 + 1e-6
    if m >= rows:
        assert y is None
        assert float((on.double().cpu() - (r.double() + scale * p)).abs().max()) < bound
    else:
        assert torch.equal(on.cpu(), r) and float((y.double().sum(0).cpu() - p).abs().max()) < bound
    # an operand that the sum does not take (rows of odd pitch) leaves the residual alone
    odd = torch.randn(m, k + 1, generator=g).to(BF).cuda()[:, :k]
    assert L.proj_add(on, odd, w.cuda(), scale) is not None


@pytest.mark.parametrize("model", ["tiny-fikerax", "tiny-lizesun"])
def test_models(model, monkeypatch):
    def logits(rows):
        monkeypatch.setattr(L, "ADD_ROWS", rows)
        eng = LLMEngine(EngineConfig(model=model, device="cuda", dtype=BF, num_blocks=96, block_size=64, max_context=2048,
                                     state_slots=6, use_graphs=False, prefix_sharing=False, temperature=0.0, seed=3))
        g = torch.Generator().manual_seed(2)
        ids = [eng.new_sequence() for _ in range(3)]
        out = []
        for lens in ((200, 31, 70), (1, 1, 1), (150, 1, 9)):
            out.append(eng.feed([(i, torch.randint(0, eng.mc.vocab_size, (n,), generator=g).tolist(), [n - 1])
                                 for i, n in zip(ids, lens)]).float())
        return torch.cat(out)
    want = logits(1 << 30)
    for rows in (1, 100):
        got = logits(rows)
        # bf16 activations whose roundings fall apart where the fp32 sums differ in their last bits
        assert float((got - want).norm() / want.norm()) < 0.02
