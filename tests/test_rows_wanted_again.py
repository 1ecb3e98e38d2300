"""More rows wanted than the step has: the products behind a :class:`Scaled` of repeated rows."""
import pytest
import torch

from k8s_llm_rca_amd.engine.engine import EngineConfig, LLMEngine
from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops import row_step as R

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("dt,m,most", [(BF, 16, R.INTO_ROWS), (BF, 2, R.INTO_ROWS), (torch.float32, 4, R.INTO_F32_ROWS),
                                       (torch.float32, 1, R.INTO_F32_ROWS)])
@pytest.mark.parametrize("cols", [8192, 32768])
def test_products(dt, m, most, cols):
    g = torch.Generator().manual_seed(m + cols)

    def rnd(*s, dtype=dt):
        return torch.randn(*s, generator=g).to(dtype).cuda()
    n, one = 2048, torch.ones(1, device="cuda")
    x = rnd(m, 1, n, dtype=torch.float32)
    h = R.add_product(x, rnd(m, 512), rnd(n, 512) * 0.04, one, one.view(1, 1), rnd(n, dtype=torch.float32), 1e-5, dt)
    assert isinstance(h, R.Scaled)
    w = rnd(cols, n) * 0.02
    for rows in (most, most + 1, 2 * most, 2 * most + 1, 40):
        some = R.rows(h, torch.arange(rows, device="cuda") * 3 % m)
        for mine, plain in ((R.proj_f32out, L.proj_f32out), (R.proj, L.proj), (R.glu_proj, L.glu_proj), (R.proj_planes, L.proj_planes)):
            got, want = mine(some, w), plain(some.read(), w)
            if mine is R.proj_planes:
                got, want = got.sum(0), want.sum(0)
            assert got.shape == want.shape
            # bf16 rows rounded in front of the norm's factor or behind it: 2^-8 of each term, of a row's 2-norm
            assert float((got.double() - want.double()).norm() / want.double().norm()) < (6e-3 if dt == BF else 1e-6)
            if rows > most:
                assert torch.equal(got, want)


@pytest.mark.parametrize("dt,tokens,wanted", [(BF, 16, 17), (BF, 16, 32), (BF, 3, 24), (BF, 5, 33), (torch.float32, 4, 5),
                                              (torch.float32, 3, 9), (torch.float32, 2, 17)])
def test_feed(dt, tokens, wanted):
    eng = LLMEngine(EngineConfig(model="fikerax-1b", device="cuda", dtype=dt, seed=3, num_blocks=16, block_size=64, max_context=256,
                                 state_slots=2))
    toks, out = [5 + 7 * i for i in range(tokens)], []
    for offs in ([i % tokens for i in range(wanted)], list(range(tokens))):
        out.append(eng.feed([(eng.new_sequence(), toks, offs)]))
    got, want = out[0], out[1][[i % tokens for i in range(wanted)]]
    # (the head's product of other numbers of rows is another kernel's sum)
    assert float((got.double() - want.double()).norm() / want.double().norm()) < (6e-3 if dt == BF else 2e-6)
