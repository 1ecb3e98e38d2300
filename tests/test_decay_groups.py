"""Linear attention with a fixed decay in more than 256 workgroups (csrc/kernels/linear_attn.hip: two of them a compute unit)
against a recurrence in 64 bits, and the rule that cuts portions into ranges."""
import pytest
import torch

from k8s_llm_rca_amd.ops import seq_ops as S


def test_ranges():
    assert S._lin_rows(16384, 16, 16, 128, 128) == 0                  # 256 workgroups as they are
    assert S._lin_rows(16384, 8, 16, 128, 128) == 512 and S._lin_rows(16384, 2, 16, 128, 128) == 1024
    assert S._lin_rows(16384, 8, 16, 64, 64) == 1024                  # the smaller heads: a workgroup a unit
    assert S._lin_rows(100, 1, 16, 128, 128) == S.LIN_CHUNK
    for n_seg in (1, 3, 4, 9):
        for H in (1, 5, 300):
            assert S._lin_rows(5000, n_seg, H, 128, 200) % 64 == 0


def test_ranges_follow_the_lengths():
    """However many short portions are beside it, a long one is cut as it is alone."""
    def rows(lens, H=16):
        return S._lin_rows(sum(lens), len(lens), H, 128, 128, lens)

    assert rows([4000]) == rows([1] * 15 + [4000]) == rows([1] * 63 + [4000]) == 256
    assert rows([4000] + [40] * 15) == 320 and rows([1] * 3 + [4000]) == 256
    assert 0 < rows([512] * 63 + [4096]) < 4096 and 0 < rows([512] * 31 + [2048]) < 2048
    assert rows([1024] * 16) == rows([512] * 15 + [1024]) == rows([1] * 32 + [300]) == 0      # nothing to wait for
    assert rows([1000] * 4) == 256 and rows([1000] * 5) == 192                               # two workgroups a unit
    assert rows([1024] * 16, 4) == 256 and rows([2000] * 5, 4) == 192 and rows([2048] * 8) == 512
    assert rows([1] * 15 + [512], 64) == 0 and rows([1] * 15 + [768], 64) == 256


def test_two_workgroups_a_unit():
    assert S._lin_two([1024] * 17, 0, 16, 128) and not S._lin_two([1024] * 16, 0, 16, 128)
    assert S._lin_two([1] * 15 + [4000], 256, 16, 128) and not S._lin_two([4000], 256, 16, 128)
    assert not S._lin_two([1] * 48 + [1000] * 16, 256, 4, 128) and S._lin_two([1000] * 17, 256, 4, 128)   # single rows
    assert not S._lin_two([64] * 100, 0, 4, 128) and S._lin_two([65] * 100, 0, 4, 128)


@pytest.mark.gpu
@pytest.mark.parametrize("lens,V,silu", [([70] * 18, 128, False), ([64, 1, 130, 65] * 5, 128, True), ([300] * 6, 128, False),
                                         ([129] * 9, 144, True), ([600] * 5, 128, True), ([1] * 15 + [900], 128, True)])
def test_more_than_a_workgroup_a_unit(lens, V, silu):
    H, D, dev = 16, 128, "cuda"
    g = torch.Generator().manual_seed(sum(lens) + V)
    T, n = sum(lens), len(lens)
    x = torch.randn(T, H * (2 * D + V) + 8, generator=g).to(torch.bfloat16)
    decay = torch.linspace(0.5, 0.9995, H)
    start = torch.randn(n, H, D, V, generator=g)
    row0 = [0]
    for k in lens:
        row0.append(row0[-1] + k)
    pos0 = [0 if s % 2 else 7 for s in range(n)]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=dev)  # noqa: E731
    seg = S.SegMeta(n, i32([s for s, k in enumerate(lens) for _ in range(k)]), i32(row0), i32(pos0), i32(list(range(n))),
                    i32([[0]] * n), row0, pos0, list(range(n)))
    rows = S._lin_rows(T, n, H, D, V, lens)
    groups = (sum(-(-k // rows) for k in lens) if rows and max(lens) > rows else n) * H * -(-V // 128)
    assert groups > 256 and S._lin_two(lens, rows if rows and max(lens) > rows else 0, H, V)
    state = start.to(dev)
    xd = x.to(dev)
    got = S.decay_attention(xd, H, D, V, decay.to(dev), state, seg, silu=silu)
    a = xd[:, :H * (2 * D + V)].double()
    if silu:
        a = (a * torch.sigmoid(a)).to(torch.bfloat16).double()
    q, k, v = (z.reshape(T, H, -1) for z in a.split([H * D, H * D, H * V], 1))
    want, last = torch.zeros(T, H, V, dtype=torch.float64, device=dev), torch.zeros(n, H, D, V, dtype=torch.float64, device=dev)
    dec = decay.double().to(dev)[:, None, None]
    for s in range(n):
        M = start[s].double().to(dev) if pos0[s] else torch.zeros(H, D, V, dtype=torch.float64, device=dev)
        for r in range(row0[s], row0[s + 1]):
            M = M * dec + k[r][:, :, None] * v[r][:, None, :]
            want[r] = (q[r][:, None, :] @ M)[:, 0]
        last[s] = M
    # operands of 16 bits and more (2^-16), sums in 32; silu's own rounding can flip a bf16 bit of q, k or v (2^-9 of one term)
    tol = 2e-3 if silu else 1e-4
    assert float((got.double().view(T, H, V) - want).norm() / want.norm()) < tol
    assert float((state.double() - last).norm() / last.norm()) < tol
