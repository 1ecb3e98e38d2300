"""One token per sequence through the matrix states with norm and gate in one launch, against the CPU forms and against the
token-by-token kernels: outputs and states, fresh sequences, slots in any order, every size the launch takes."""
import pytest
import torch

from k8s_llm_rca_amd.ops import norm as N
from k8s_llm_rca_amd.ops import seq_ops as S

pytestmark = pytest.mark.gpu
TYPES = [torch.bfloat16, torch.float32]


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed + sum(shape)))


def meta(pos0, slots, dev):
    n = len(pos0)

    def i32(v):
        return torch.tensor(list(v), dtype=torch.int32, device=dev)
    return S.SegMeta(n, i32(range(n)), i32(range(n + 1)), i32(pos0), i32(slots), i32([0] * n).view(n, 1), list(range(n + 1)),
                     list(pos0), list(slots), n_single=n)


def close(a, b, dt):
    """fp32 sums of up to 256 terms in another order; activations of ``dt`` one rounding apart (bf16: of the row's scale, the
    norms divide sums that cancel)."""
    a, b = a.double().cpu(), b.double().cpu()
    tol = 2.0 ** -7 if dt == torch.bfloat16 else 2e-5
    assert float((a - b).abs().max()) < tol * float(b.abs().max()), float((a - b).abs().max() / b.abs().max())


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("H,G,D,V", [(4, 2, 128, 128), (3, 1, 64, 64), (2, 2, 128, 64), (6, 3, 64, 128)])
@pytest.mark.parametrize("pos0", [[0], [7, 0, 1], [3] * 9])
@pytest.mark.parametrize("wide", [True, False, None])
def test_delta(H, G, D, V, pos0, wide, dt):
    T = len(pos0)
    slots = list(range(T, 0, -1))
    qkv, a, rate, db = rnd(T, 2 * G * D + H * V).to(dt), rnd(T, H * D), rnd(H).abs(), rnd(H * D)
    beta, gate = rnd(T, H + 3), rnd(T, H * V + 4, seed=1)
    w = None if wide is None else rnd(H * V if wide else V)

    def on(dev, fused):
        st = (rnd(T + 2, H, D, V) * 0.3).to(dev)
        args = (qkv.to(dev), H, G, D, V, a.to(dev), rate.to(dev), db.to(dev), beta.to(dev)[:, 2:], st, meta(pos0, slots, dev))
        g, wd = gate.to(dev), None if w is None else w.to(dev)
        if fused:
            return S.delta_layer(*args, g, wd, 1e-5, dt), st
        return S.head_norm_gate(S.gated_delta(*args), g, wd, H, V, 1e-5, dt), st
    got = on("cuda", True)
    for want in (on("cpu", True), on("cuda", False)):
        close(got[0], want[0], dt)
        close(got[1], want[1], torch.float32)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("H,D,V", [(4, 128, 128), (3, 64, 64), (2, 128, 64), (5, 64, 128)])
@pytest.mark.parametrize("pos0", [[0], [7, 0, 1], [3] * 9])
@pytest.mark.parametrize("wide", [True, False])
def test_memory(H, D, V, pos0, wide, dt):
    T = len(pos0)
    slots = [(5 * i + 2) % (T + 2) if T == 1 else T - i for i in range(T)]
    pad = 4                                                  # a column slice of a wider projection, rows of 16 bytes
    x = rnd(T, pad + 2 * H * (D + V) + 2 * H + (-2 * H) % 4)
    gb, w = rnd(2 * H), rnd(H * V if wide else V)
    states = [rnd(T + 2, H, D, V) * 0.3, rnd(T + 2, H, D), rnd(T + 2, H)]
    width = 2 * H * (D + V) + 2 * H

    def fn(dev, st, off):
        xs = x.to(dev)[:, pad:pad + width]
        return S.memory_layer(xs, H, D, V, gb.to(dev), 15.0, *st, meta(pos0, slots, dev), w.to(dev), 1e-5, dt)
    cpu, one, parts = ([s.clone().to(d) for s in states] for d in ("cpu", "cuda", "cuda"))
    a, b = fn("cpu", cpu, 0), fn("cuda", one, 0)
    xs = x.cuda()[:, pad:pad + width]
    o, mul = S.matrix_memory(xs, H, D, V, gb.cuda(), 15.0, *parts, meta(pos0, slots, "cuda"), defer_scale=True)
    c = S.head_norm_gate(o, xs[:, 2 * H * D + H * V:2 * H * (D + V)], w.cuda(), H, V, 1e-5, dt, mul=mul)
    for want, st in ((a, cpu), (c, parts)):
        close(b, want, dt)
        for p, q in zip(one, st):
            close(p, q, torch.float32)


@pytest.mark.parametrize("dt", TYPES)
@pytest.mark.parametrize("H,D,V", [(4, 128, 128), (3, 64, 64), (2, 128, 64), (5, 64, 128)])
@pytest.mark.parametrize("pos0", [[0], [7, 0, 1], [3] * 9])
def test_decay(H, D, V, pos0, dt):
    """With the division by the row's root mean square made up for behind a product."""
    T, HV, W = len(pos0), H * V, 64
    slots = list(range(T, 0, -1))
    x, dec, w = rnd(T, H * (2 * D + V) + HV).to(dt), torch.linspace(0.5, 0.99, H), rnd(HV)
    wo, res0, one = (rnd(W, HV) * HV ** -0.5).to(dt), rnd(T, 1, W), torch.ones(1)
    out = {}
    for name, dev in (("cpu", "cpu"), ("cuda", "cuda")):
        st = (rnd(T + 2, H, D, V) * 0.3).to(dev)
        xd, r = x.to(dev), res0.clone().to(dev)
        y, rms = S.decay_layer(xd, H, D, V, dec.to(dev), st, meta(pos0, slots, dev), xd[:, x.shape[1] - HV:], w.to(dev), 1e-5,
                               dt)
        assert (rms is not None) == (dev == "cuda") and y.dtype == dt
        N.hyper_step(r, y.float() @ wo.float().to(dev).T, one.to(dev), one.view(1, 1).to(dev), rms=rms)
        out[name] = (r, st)
    # sums of 512 products of activations, each rounded once
    close(out["cuda"][0] - res0.cuda(), out["cpu"][0] - res0, dt)
    close(out["cuda"][1], out["cpu"][1], torch.float32)


def test_other_steps_take_the_other_kernels():
    """A step with a longer portion, other sizes, unaligned gates: accepted, and without a factor left over."""
    H, D, V, dt = 2, 64, 64, torch.bfloat16
    x, dec, w = rnd(3, H * (2 * D + V) + H * V).to(dt).cuda(), torch.rand(H).cuda(), rnd(H * V).cuda()
    st = rnd(4, H, D, V).cuda()
    m = S.SegMeta(2, *(torch.tensor(v, dtype=torch.int32).cuda() for v in ([0, 0, 1], [0, 2, 3], [1, 4], [0, 1], [[0], [0]])),
                  [0, 2, 3], [1, 4], [0, 1])
    assert S.decay_layer(x, H, D, V, dec, st, m, x[:, -H * V:], w, 1e-5, dt)[1] is None
    one = meta([1, 2, 3], [0, 1, 2], "cuda")
    assert S.decay_layer(x, H, D, V, dec, st, one, x[:, -H * V:], w, 1e-5, dt)[1] is not None
    assert S.decay_layer(x, H, D, V, dec, st, one, x[:, -H * V - 1:-1], w, 1e-5, dt)[1] is None
    xs = rnd(1, 3 * (2 * 32 + 32) + 96).to(dt).cuda()
    assert S.decay_layer(xs, 3, 32, 32, torch.rand(3).cuda(), rnd(2, 3, 32, 32).cuda(), meta([1], [0], "cuda"), xs[:, -96:],
                         rnd(96).cuda(), 1e-5, dt)[1] is None
