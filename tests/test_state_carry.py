"""What passes between the parts of a prompt: the states of ranges (csrc/kernels/state_carry.h), more of them than are asked for at
once and entries that do not come in fours, and the matrix memory's gates (csrc/kernels/matrix_mem.hip) over rounds of waves."""
import pytest
import torch

from k8s_llm_rca_amd.ops._lib import check, lib, ptr, stream_ptr

pytestmark = pytest.mark.gpu


def i32(v):
    return torch.tensor(v, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("ranges", [[1], [8], [9, 0, 1], [17, 8, 3]])
@pytest.mark.parametrize("D,V,bf16", [(64, 32, True), (128, 128, True), (6, 5, False), (16, 48, False)])
def test_ranges_carry_the_state(ranges, D, V, bf16):
    """Portions cut into ranges against the same portions in one, in 64 bits where the cut may round otherwise."""
    H, L, n = 3, 16, len(ranges)
    g = torch.Generator().manual_seed(D + len(ranges))
    rows = [max(1, L * k - 5) if k else 1 for k in ranges]
    T = sum(rows)
    x = torch.randn(T, H * (2 * D + V), generator=g).cuda() * 0.3
    x = x.bfloat16() if bf16 else x
    decay = torch.tensor([0.9, 0.99, 0.5], device="cuda")
    row0 = [sum(rows[:i]) for i in range(n + 1)]
    pos0 = [0 if i % 2 == 0 else 7 for i in range(n)]
    start = torch.randn(n, H, D, V, generator=g).cuda()
    items, item0 = [], [0]
    for i, m in enumerate(rows):
        items += [[i, row0[i] + a, min(L, m - a), 0] for a in range(0, m, L)]
        item0.append(len(items))
    out, r0, p0, sl = [], i32(row0), i32(pos0), i32(list(range(n)))
    for cut in (True, False):
        st, o = start.clone(), torch.full((T, H * V), float("nan"), device="cuda")
        cs = torch.full((len(items), H, D, V), float("nan"), device="cuda") if cut else None
        it, i0 = (i32(items), i32(item0)) if cut else (None, None)
        if bf16:
            check(lib().k8s_decay_attn_mfma(ptr(x), x.stride(0), 0, ptr(decay), ptr(st), ptr(r0), ptr(p0),
                                            ptr(sl), ptr(o), n, H, D, V, stream_ptr(x), ptr(it),
                                            len(items) if cut else 0, ptr(i0), ptr(cs), 0), "decay")
        else:
            check(lib().k8s_decay_attn(ptr(x), x.stride(0), 1, 0, ptr(decay), ptr(st), ptr(r0), ptr(p0),
                                       ptr(sl), ptr(o), n, H, D, V, stream_ptr(x), ptr(it),
                                       len(items) if cut else 0, ptr(i0), ptr(cs)), "decay")
        out.append((st, o))
    (s1, o1), (s0, o0) = out
    # fp32 sums of up to 16 decayed products of size 0.1 (of two bf16 parts: 2^-16 of them) on states of size 1, in another order
    assert float((s1 - s0).abs().max()) < 1e-4 and float((o1 - o0).abs().max()) < 1e-3


@pytest.mark.parametrize("rows", [[1], [63, 64, 65], [512, 513], [1, 1100, 700, 0, 300]])
def test_gates(rows):
    H, D, V, cap, n = 2, 8, 4, 15.0, len(rows)
    T, g = sum(rows), torch.Generator().manual_seed(len(rows))
    x = torch.randn(T, 2 * H * D + 2 * H * V + 2 * H, generator=g).cuda()
    bias, ms = torch.randn(2 * H, generator=g).cuda(), torch.rand(n, H, generator=g).cuda()
    pos0 = [0 if i % 2 == 0 else 5 for i in range(n)]
    row0 = [sum(rows[:i]) for i in range(n + 1)]
    r0, p0, sl = i32(row0), i32(pos0), i32(list(range(n)))
    st, ns, start = torch.zeros(n, H, D, V, device="cuda"), torch.zeros(n, H, D, device="cuda"), ms.clone()
    ab, nq, mul, out = (torch.empty(T, H, *s, device="cuda") for s in ((3,), (), (), (V,)))
    check(lib().k8s_matrix_memory(ptr(x), x.stride(0), ptr(bias), cap, ptr(st), ptr(ns), ptr(ms), ptr(r0), ptr(p0),
                                  ptr(sl), ptr(ab), ptr(nq), ptr(mul), ptr(out), n, T, H, D, V, 1e-6, 0,
                                  stream_ptr(x), 0, 0, 0, 0, 0, 0, 0), "memory")
    gi = cap * torch.tanh((x[:, -2 * H:-H].double() + bias[:H].double()) / cap)
    gf = torch.nn.functional.logsigmoid(cap * torch.tanh((x[:, -H:].double() + bias[H:].double()) / cap))
    for i in range(n):
        m = start[i].double() if pos0[i] else torch.zeros(H, dtype=torch.float64, device="cuda")
        for t in range(row0[i], row0[i + 1]):
            new = torch.maximum(gf[t] + m, gi[t])
            want = torch.stack([torch.exp(gf[t] + m - new), torch.exp(gi[t] - new), new], -1)
            # sums of up to 64 log gates in fp32 (2^-24 of some 100), and m carried over the waves in front
            assert float((ab[t].double() - want).abs().max()) < 1e-4 * (1 + float(new.abs().max())), (i, t)
            m = new
        assert float((ms[i].double() - m).abs().max()) < 1e-4 * (1 + float(m.abs().max()))


@pytest.mark.parametrize("rows", [[10, 1, 30, 19], [70, 0, 0, 0, 0, 0, 0, 0], [64, 1, 129], [64] * 3 + [1] * 9])
def test_gates_of_short_sequences(rows):
    """Sequences that one wave has alone, among themselves and beside a longer one, and one wave for more rows than it has lanes."""
    test_gates(rows)
