"""The waits of csrc/kernels/gemm_split_f32.hip, read from the assembly that its source gives: where the kernel's waves meet, no
wave's loads into LDS are still on their way, whatever path it came by."""
import re
import shutil
import subprocess

import pytest

from k8s_llm_rca_amd import _build

NONE = 1 << 30      # no load into LDS on its way


def _blocks(lines):
    """(instructions, successors) of every basic block of a function, the entry first."""
    at, blocks = {}, [[]]
    for line in lines:
        text = line.split(";")[0].strip()
        label = re.match(r"(\.LBB\w+):", text)
        if label:
            blocks.append([])
            at[label.group(1)] = len(blocks) - 1
        elif text and not text.startswith("."):
            blocks[-1].append(text)
            if text.startswith(("s_cbranch", "s_branch", "s_endpgm")):
                blocks.append([])
    out = []
    for i, b in enumerate(blocks):
        last = b[-1].split() if b else [""]
        nxt = [at[last[1]]] if last[0].startswith(("s_cbranch", "s_branch")) else []
        if last[0] not in ("s_branch", "s_endpgm") and i + 1 < len(blocks):
            nxt.append(i + 1)
        out.append((b, nxt))
    return out


def unwaited(lines):
    """Barriers (block, index) that may be reached with a load into LDS on its way.  Followed through the function: the least
    number of memory instructions issued behind the last such load; a wait for that many or fewer ends it."""
    return _follow(lines)[0]


def overlap(lines):
    """The waits that end such loads, with the least number of matrix instructions issued between the two."""
    return _follow(lines)[1]


def _follow(lines):
    blocks = _blocks(lines)
    state, todo, bad, between = {0: (NONE, 0)}, [0], set(), {}
    while todo:
        i = todo.pop()
        behind, matrix = state[i]                  # memory and matrix instructions since the last load into LDS
        for k, text in enumerate(blocks[i][0]):
            op = text.split()[0]
            wait = re.search(r"vmcnt\((\d+)\)", text)
            if "load_lds" in op or (op.startswith("buffer_load") and " lds" in text):
                behind, matrix = 0, 0
            elif op.startswith(("global_", "buffer_", "flat_", "scratch_")) and behind != NONE:
                behind += 1
            elif op.startswith("v_mfma") and behind != NONE:
                matrix += 1
            elif op == "s_waitcnt" and wait and int(wait.group(1)) <= behind:
                if behind != NONE:
                    between[i, k] = text, min(matrix, between.get((i, k), (text, matrix))[1])
                behind = NONE
            elif op in ("s_barrier", "s_endpgm") and behind != NONE:
                bad.add((i, k))
        for j in blocks[i][1]:
            old = state.get(j, (NONE + 1, NONE))
            new = (min(behind, old[0]), min(matrix if behind != NONE else NONE, old[1]))
            if new != old:
                state[j] = new
                todo.append(j)
    return bad, list(between.values())


def test_reading():
    """The reading itself, on a few lines."""
    def f(s):
        return unwaited(s.split("\n"))
    load, dma = "global_load_dwordx4 v[0:3], v4, s[0:1]", "global_load_lds_dwordx4 v4, s[0:1]"
    end = "s_waitcnt vmcnt(0)\ns_endpgm"
    assert not f(f"{dma}\n{load}\ns_waitcnt vmcnt(1)\ns_barrier\n{end}")
    assert f(f"{load}\n{dma}\ns_waitcnt vmcnt(1)\ns_barrier\n{end}") and f(f"{dma}\ns_endpgm")
    loop = "{0}\n.LBB0_1:\ns_waitcnt vmcnt({1})\ns_barrier\n{2}\ns_cbranch_scc1 .LBB0_1\n" + end
    assert not f(loop.format(f"{dma}\n{load}", 1, f"{dma}\n{load}"))
    assert f(loop.format(f"{dma}\n{load}", 1, f"{load}\n{dma}"))          # by the way back only
    mfma = "v_mfma_f32 v0\n" * 2
    assert overlap(loop.format(dma, 1, f"{mfma}{dma}").split("\n")) == [("s_waitcnt vmcnt(0)", 0)]
    assert overlap(loop.format(dma, 0, f"{dma}\n{mfma}").split("\n")) == [("s_waitcnt vmcnt(0)", 0), ("s_waitcnt vmcnt(0)", 2)]
    assert f(f"{dma}\ns_cbranch_scc0 .LBB0_1\n{load}\n.LBB0_1:\ns_waitcnt vmcnt(1)\ns_barrier\n{end}")


@pytest.mark.skipif(shutil.which(_build.HIPCC) is None, reason="needs the compiler")
def test_waits_cover_the_loads(tmp_path):
    src, out = _build.CSRC + "/kernels/gemm_split_f32.hip", tmp_path / "split.s"
    subprocess.run([_build.HIPCC, *_build.hip_flags(), "-S", "--cuda-device-only", src, "-o", str(out)], check=True,
                   capture_output=True)
    kernels = re.findall(r"^(_ZN3k8s21gemm_split_f32_kernel\w+):(.*?)^\.Lfunc_end", out.read_text(), re.S | re.M)
    assert len(kernels) == 10                                              # five tiles, plain and gated
    bad = {name: found for name, body in kernels if (found := unwaited(body.split("\n")))}
    assert not bad
    for name, body in kernels:
        # a step's matrix instructions (two columns, six products a fragment) stand between its loads and their wait
        ended = [n for text, n in overlap(body.split("\n")) if "vmcnt(4)" in text]
        assert ended and set(ended) == {12 * int(re.search(r"ILi(\d+)E", name).group(1))}
        assert "global_load_lds" in body and body.count("s_barrier") >= 2
