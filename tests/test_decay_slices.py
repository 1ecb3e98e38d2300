"""The decaying attention's reply steps with several workgroups a head (csrc/kernels/state_step.hip): the states to the bit, results
and sums of squares as with one."""
import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu


def meta(n):
    def i32(v):
        return torch.tensor(list(v), dtype=torch.int32, device="cuda")
    pos0, slots = [i % 3 for i in range(n)], list(range(n, 0, -1))
    return S.SegMeta(n, i32(range(n)), i32(range(n + 1)), i32(pos0), i32(slots), i32([0] * n).view(n, 1), list(range(n + 1)),
                     pos0, slots, n_single=n)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("T,H", [(1, 16), (8, 16), (9, 16), (5, 3), (2, 17)])
def test_slices(monkeypatch, T, H, D, dt):
    V, g = 128, torch.Generator().manual_seed(T + H)
    x = torch.randn(T, H * (2 * D + 2 * V), generator=g).to(dt).cuda()
    dec, w = torch.linspace(0.5, 0.99, H).cuda(), torch.randn(H * V, generator=g).cuda()
    st0 = (torch.randn(T + 1, H, D, V, generator=g) * 0.3).cuda()
    assert S.decay_slices(T, H, V) == (4 if T * H <= 128 and H <= 16 else 1) and S.decay_slices(1, 1, 64) == 1
    res = []
    for n in (S.decay_slices(T, H, V), 1, 2):
        monkeypatch.setattr(S, "decay_slices", lambda *a, n=n: n)
        st = st0.clone()
        y, (ss, width, eps) = S.decay_layer(x, H, D, V, dec, st, meta(T), x[:, -H * V:], w, 1e-5, dt)
        assert ss.shape == (T, H * n) and width == H * V
        res.append((y, ss.sum(1), st))
    for y, ss, st in res:
        assert torch.equal(st, res[1][2])
        # D products of fp32 in another order, before one rounding; the sums of the squares of these
        tol = 2.0 ** -8 if dt == torch.bfloat16 else 64 * 2.0 ** -24
        big = float(res[1][0].double().abs().max())
        assert float((y.double() - res[1][0].double()).abs().max()) <= tol * big
        assert torch.allclose(ss, res[1][1], rtol=1e-5, atol=0)
