"""One row's product with the residual's pass in front (csrc/kernels/gemm_row_step.hip, ops/row_step.py)."""
import pytest
import torch

from k8s_llm_rca_amd.engine.engine import EngineConfig, LLMEngine
from k8s_llm_rca_amd.models.registry import get_any_config
from k8s_llm_rca_amd.ops import linear as L
from k8s_llm_rca_amd.ops import norm as N
from k8s_llm_rca_amd.ops import row_step as R
from k8s_llm_rca_amd.ops import seq_ops as S

BF = torch.bfloat16
gpu = pytest.mark.gpu
#: columns, K: a strip of one wave's least rows, one and several load instructions of K, odd counts of strips and of K
SHAPES = [(128, 512), (2560, 2048), (1088, 2048), (4112, 1536), (640, 1024), (8736, 2048)]


def test_plan_and_what_is_refused():
    for n, k in SHAPES:
        for kind in (L.ROWS_BF16, L.ROWS_F32, L.ROWS_SILU, L.ROWS_RELU2):
            for planes in (False, True)[:1 + (kind == L.ROWS_F32)]:
                p = R.plan(n, k, kind, planes)
                if p is not None:
                    assert n % ((8 if kind == L.ROWS_SILU else 16) * p[0]) == 0 and k % (R.COLS * p[1]) == 0 and p[0] <= 2
    assert R.plan(8192, 2048, L.ROWS_SILU) is not None
    assert R.plan(8192, 4096, L.ROWS_BF16) is None and R.plan(8200, 2048, L.ROWS_BF16) is None
    x, y, w, b = torch.ones(1, 512), torch.ones(1, 512), torch.ones(512), torch.zeros(512)
    h = R.dyt_step(x, y, 1.0, None, 1.0, 0.5, w, b, torch.float32)      # on the CPU: the separate pass
    assert isinstance(h, torch.Tensor) and bool((x == 2.0).all())


def _weights(n, k, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(n, k, generator=g) * k ** -0.5).to(BF).cuda()


def _products(n, k, h, again):
    """(name, result) of every product of the activations' maker ``again()``."""
    w = _weights(n, k, n + k)
    yield "f32", R.proj_f32out(again(), w), (h.double() @ w.double().T)
    planes = R.proj_planes(again(), w)
    yield "planes", planes.sum(0), (h.double() @ w.double().T)
    yield "bf16", R.proj(again(), w), (h.double() @ w.double().T)
    w2 = _weights(2 * n, k, n)
    g, u = (h.double() @ w2.double().T).split(n, 1)
    yield "silu", R.glu_proj(again(), w2), torch.nn.functional.silu(g) * u
    yield "relu2", R.relu_sq_proj(again(), w), (h.double() @ w.double().T).clamp_min(0) ** 2


def _check(name, got, want, k):
    # fp32 sums of K terms of size K^(-1/2);  results, gate and up rounded to bf16 once each
    if name in ("f32", "planes"):
        assert float((got.double() - want).abs().max()) < 4e-6 * k ** 0.5, name
    else:
        tol = 2.0 ** -8 if name == "bf16" else 2.0 ** -6
        assert bool(((got.double() - want).abs() <= tol * want.abs() + 2e-3).all()), name


@gpu
@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("planes,rn,add", [(1, 0, False), (4, 16, False), (3, 64, True), (2, 0, True), (8, 0, False)])
def test_rms_pass_in_front(n, k, planes, rn, add):
    g = torch.Generator().manual_seed(k + planes)
    x0 = (torch.randn(1, 1, k, generator=g) * 3).cuda()
    y = torch.randn(planes, 1, k, generator=g).cuda()
    nw = (1 + 0.1 * torch.randn(k, generator=g)).cuda()
    one = torch.ones(1, device="cuda")
    ss = (torch.rand(1, rn, generator=g) * 100).cuda() if rn else None
    again = None
    if add:
        again = torch.tensor([3], dtype=torch.int32, device="cuda"), torch.randn(5, k, generator=g).to(BF).cuda(), 4.5
    kw = dict(again=again, rms=(ss, 2048.0, 1e-5) if rn else None)
    x1 = x0.clone()
    h = N.hyper_step(x1, y, one, one.view(1, 1), inn=one, nw=nw, eps=1e-5, out_dtype=BF, **kw)
    seen = []

    def make():
        x = x0.clone()
        seen.append((x, R.step(x, y, one, one.view(1, 1), nw, 1e-5, BF, **kw)))
        return seen[-1][1]

    for name, got, want in _products(n, k, h, make):
        x, s = seen[-1]
        _check(name, got, want, k)
        assert isinstance(s, R.RowStep) == (planes <= R.PLANES)
        assert torch.equal(R.residual(s, x), x1), name                 # the pass's own bits
        if isinstance(s, R.RowStep) and s.x.data_ptr() != x.data_ptr():
            assert torch.equal(x, x0)                                  # made elsewhere: the old row is left alone
            with pytest.raises(RuntimeError):
                s.read()
    s = make()
    if isinstance(s, R.RowStep):                                       # a product that the kernel does not take
        assert torch.equal(s.product(_weights(40, k, 1), L.ROWS_F32, L.proj_f32out), L.proj_f32out(h, _weights(40, k, 1)))
        assert torch.equal(s.h, h) and torch.equal(R.residual(s, x1), x1)


@gpu
@pytest.mark.parametrize("n,k", SHAPES)
@pytest.mark.parametrize("planes,planes2", [(1, 0), (4, 2), (3, 4), (4, 0)])
def test_dyt_pass_in_front(n, k, planes, planes2):
    g = torch.Generator().manual_seed(k + planes)
    x0 = torch.randn(1, k, generator=g).cuda()
    y = torch.randn(planes, 1, k, generator=g).cuda()
    y2 = torch.randn(planes2, 1, k, generator=g).cuda() if planes2 else None
    w, b = (torch.randn(k, generator=g).cuda() for _ in range(2))
    x1 = x0.clone()
    h = N.add_dyt(x1, y, 0.75, y2, 0.5, 0.7, w, b, out_dtype=BF)
    seen = []

    def make():
        x = x0.clone()
        seen.append((x, R.dyt_step(x, y, 0.75, y2, 0.5, 0.7, w, b, BF)))
        return seen[-1][1]

    for name, got, want in _products(n, k, h, make):
        x, s = seen[-1]
        _check(name, got, want, k)
        assert torch.equal(R.residual(s, x), x1), name
    s = make()
    a = R.proj(s, _weights(n, k, 1), keep=True)
    assert torch.equal(s.read(), h)                                    # kept for the layer's second product
    _check("bf16", a, h.double() @ _weights(n, k, 1).double().T, k)
    assert torch.equal(R.proj_f32out(s, _weights(160, k, 2)), L.proj_f32out(h, _weights(160, k, 2)))


@gpu
def test_values_that_are_not_finite_stay_where_they_are():
    k, n = 2048, 256
    x, y = torch.zeros(1, k, device="cuda"), torch.randn(1, k, device="cuda")
    w, wn = _weights(n, k, 3), torch.ones(k, device="cuda")
    w[7, 3] = float("nan")
    w[9, 100] = float("inf")
    h = N.add_dyt(x.clone(), y, 1.0, None, 1.0, 1.0, wn, wn, out_dtype=BF)
    got = R.proj_f32out(R.dyt_step(x, y, 1.0, None, 1.0, 1.0, wn, wn, BF), w)
    want = L.proj_f32out(h, w)
    assert torch.equal(torch.isfinite(got), torch.isfinite(want)) and int((~torch.isfinite(got)).sum()) == 2


@gpu
def test_captured_and_repeated():
    k, n = 2048, 2560
    x0, y = torch.randn(1, 1, k, device="cuda"), torch.randn(4, 1, k, device="cuda")
    one, nw, w = torch.ones(1, device="cuda"), torch.rand(k, device="cuda"), _weights(n, k, 5)

    def f():
        s = R.step(x0, y, one, one.view(1, 1), nw, 1e-5, BF)
        return R.proj_planes(s, w), s.x

    eager = [t.clone() for t in f()]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = f()
    for _ in range(3):
        for t in out:
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, eager))


def test_the_only_row_is_every_row():
    def rows(t, idx):
        ids = torch.zeros(t, dtype=torch.int32)
        return S.wanted_rows(S.SegStepInputs(ids, ids, ids, None, idx))

    some = torch.tensor([0])
    assert rows(1, some) is None and rows(1, None) is None and rows(2, None) is None
    assert rows(2, some) is some and rows(1, some[:0]) is not None and rows(1, some.repeat(2)).numel() == 2


@gpu
@pytest.mark.parametrize("model", ["fikerax-1b", "lizesun-1b"])
def test_one_row_has_the_same_bits_captured_and_not(model):
    """At widths that the kernel takes: the head behind the last pass, and behind the row picked from the residual."""
    over = {"layers": get_any_config(model).layers[:3]} if model == "lizesun-1b" else {}

    def logits(graphs):
        eng = LLMEngine(EngineConfig(model=model, model_overrides=over, device="cuda", dtype=BF, num_blocks=16, block_size=64,
                                     max_context=512, state_slots=2, use_graphs=graphs, prefix_sharing=False, seed=3))
        sid = eng.new_sequence()
        out = [eng.feed([(sid, [5, 6, 7], [2])])] + [eng.feed([(sid, [11 * i], [0])]).clone() for i in range(8)]
        torch.cuda.synchronize()
        return out, eng.stats["graph_steps"]

    (want, none), (got, some) = logits(False), logits(True)
    assert not none and some >= 4
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_more_rows_do_not_pay_for_the_rule(monkeypatch):
    """From two rows on neither operand is looked at: a small prompt's step is host time."""
    def asked(*a, **k):
        raise AssertionError("asked")
    monkeypatch.setattr(R, "_one_row", asked)
    monkeypatch.setattr(R, "use_hip", asked)
    monkeypatch.setattr(N, "hyper_step", lambda *a, **k: "apart")
    monkeypatch.setattr(N, "add_dyt", lambda *a, **k: "apart")
    x, y, w = torch.randn(2, 1, 512), torch.randn(2, 512), torch.ones(512)
    assert R.step(x, y, w, w, w, 1e-6, BF) == "apart"
    assert R.dyt_step(x[:, 0], y, 1.0, None, 1.0, 0.5, w, w, BF) == "apart"
