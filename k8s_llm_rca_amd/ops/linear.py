"""Projection GEMMs: hand-written skinny MFMA GEMM for decode shapes, hipBLASLt otherwise."""
from __future__ import annotations

import functools
import json
import math
import os
from typing import Dict, List, Tuple

import torch
import torch.nn.functional as F

from ..knobs import KNOBS
from ._lib import check, lib, ptr, scratch, stream_ptr, unwatched
from .moe import glu_clamp
from .norm import relu_sq

SKINNY_MAX_M = KNOBS.skinny_max_m
# measured on MI355X (tools/bench_kernels.py): the skinny kernel beats hipBLASLt
# ~2x on the small-N decode projections (o_proj / QKV) for M <= 16 and ties or
# loses on the wide ones; beyond M = 16 its L2-read X operand is the bottleneck.
SKINNY_MAX_NK = 8192 * 4096
_enabled = KNOBS.skinny


def set_skinny(enabled: bool) -> None:
    global _enabled
    _enabled = enabled


KIND_LIB, KIND_SKINNY, KIND_MID, KIND_GRP, KIND_STREAM, KIND_BIG, KIND_ROWS = 0, 1, 2, 3, 4, 5, 6

# -------------------------------------------------- products of up to 32 rows (csrc/kernels/gemm_rows.hip)
ROWS_MAX_M = 32
ROWS_BF16, ROWS_F32, ROWS_SILU, ROWS_RELU2 = 0, 1, 2, 3


def _rows_channels(M: int, big: int, K: int, out: int, planes: bool) -> bool:
    """Whether rows of W that are a multiple of 16 KB apart make another kernel the quicker one.  They, and no others, cost up
    to a third of the rate until there are columns enough (they likely fall on few of the memory's channels).  us before /
    with the row-streaming kernel, bf16:  one row of 16384 x 7168, 8192, 8704 48.6 / 38.5, 52.1 / 57.9, 62.3 / 46.0;  8 rows
    of 6144 x 8192 1.06, 9216 x 8192 1.12, 15360 x 8192 1.05 of the time before, but 4096 x 8192 0.87, 16384 x 8192 0.83, and
    gated 0.9 at all columns;  8192 x 16384 56.5 / 61.4;  32 rows of 8192 x 8192 31.4 / 35.2, 16384 x 8192 54.7 / 67.5, 28672
    x 8192 115 / 100, 16384 x 16384 96.7 / 119.6, 28672 x 16384 167 / 175."""
    if K % 8192:
        return False
    if M == 1 and out != ROWS_F32:
        return K == 8192                 # (16384 and more: 0.72 to 0.88 of the skinny kernel's time)
    if M > 16 or K % 16384 == 0:
        return 8192 <= big < 3 * K
    return out != ROWS_SILU and (8192 if planes or out == ROWS_RELU2 else 5119) < big < 2 * K


def rows_shape_ok(M: int, N: int, K: int, nf: int, ranges: int, out: int = ROWS_F32) -> bool:
    """What csrc/kernels/gemm_rows.hip accepts; ``N``: result columns."""
    return (0 < M <= ROWS_MAX_M and nf in ((1, 2, 4) if M <= 16 else (2, 4)) and N > 0 and K > 0
            and N % ((8 if out == ROWS_SILU else 16) * nf) == 0 and ranges >= 1 and (ranges == 1 or out == ROWS_F32)
            and K % (4 * ranges * (64 if nf == 4 or M > 16 else 128)) == 0)


@functools.lru_cache(maxsize=4096)
def rows_plan(M: int, N: int, K: int, out: int = ROWS_BF16, planes: bool = False):
    """(16-row fragments of a workgroup, K ranges) with which the row-streaming kernel takes a product, or None: another
    kernel is the quicker one or the shape does not fit.  ``N``: result columns; ``planes``: K ranges may stay apart.

    Up to 16 rows it is the quickest at sizes from 128 x 512 to 128256 x 4096, at 0.53 to 0.97 of the time before with cold
    weights.  Up to 32 rows X is half of what it reads: from 8192 columns on (us at 32 rows before / this: 8192 x 2048
    10.3 / 9.0, 16384 x 4096 42.0 / 26.9; 4096 x 2048 9.2 / 10.0 in fp32, 4096 x 8192 20.8 / 26.8), and of these where K is
    up to 1024 or a multiple of 2048 (1280 to 3584 0.61 to 1.07 of the time before, by shape); planes up to a K of 2048
    (2048 x 2048 with the pass behind 0.93, 2560 x 4096 1.10, 1088 x 8192 1.06 of the time before); and not past 40960
    columns of a K from 8192 on with 25 rows or more, where X is most of it (57344 x 8192 188 / 202, gated 57344 x 12288
    280 / 299).

    Where K is no multiple of 512, only four fragments with loads of 128 bytes fit up to 16 rows, and few workgroups are left:
    us before / this at 2560 x 1280 and 1 row 4.2 / 6.2, 2048 x 3840 and 4 rows 9.0 / 13.9, 128 x 768 and 16 rows 3.0 / 4.8,
    but 8192 x 1280 0.9 to 1.0 (one row 1.02 to 1.08), 16384 x 1280 0.6 to 0.8 of the time before, gated from 2048 columns on
    0.7 to 1.04.  Planes that cannot be cut lose to those that can: 2048 x 768 at 32 rows 1.14, 128 x 3584 at 16 rows 1.12.
    Little more columns than a wave of workgroups has: 8736 x 4096 at 32 rows 1.15, 9216 x 12288 at 16 1.10, 4112 x 12288 1.14.

    The fragments and ranges are those of the least work on the busiest compute unit: a workgroup streams 16 nf x K / ranges
    weights and X of M rows (2.5 % of a fragment's time each row), and 256 of them run at once.  Four fragments, whose loads
    cover 128 bytes of a row instead of 256, cost a tenth more.  Over the measured sizes this is within 0.6 % of the best
    choice on average.  K is cut only where one fragment a workgroup would leave more than a quarter of the compute units
    idle, and not for a K of up to 1024 (2048 x 1024 whole / cut 5.1 / 5.0 us with the pass behind)."""
    big = N * (2 if out == ROWS_SILU else 1)
    if not 0 < M <= ROWS_MAX_M or big < 128 or K < 512:
        return None
    if M > 16 and not ((K <= 1024 or K % 2048 == 0) and (K <= 2048 if planes else big >= 8192)):
        return None
    if M <= 16 and K % 512 and big < (4096 if out == ROWS_SILU else 8192 + (M == 1)):
        return None
    if planes and (M > 16 and K % 512 or M > 8 and K > 2048 and K % 1024 and big < 1024):
        return None
    if _rows_channels(M, big, K, out, planes):
        return None
    if out != ROWS_SILU and (8192 < big <= 10240 and (M > 8 and K > 6144 or M > 16 and K > 2048 and big < 9216)
                             or 4096 < big < 4608 and M > 8 and K >= 8192):
        return None
    if M > 24 and K >= 8192 and big > 40960:
        return None
    strips = -(-big // (16 if M <= 16 else 32))
    cut = planes and (K > 1024 or M > 16) and 4 * strips < 3 * 256 * -(-strips // 256)
    best = None
    for nf in (1, 2, 4):
        for ranges in (1, 2, 4, 8) if cut else (1,):
            if not rows_shape_ok(M, N, K, nf, ranges, out):
                continue
            wgs = big // (16 * nf) * ranges
            waves = -(-wgs // 256) if wgs <= 6 * 256 else wgs / 256
            cost = (waves * (nf * K / ranges * (1 + 0.025 * M / nf) * (1.1 if nf == 4 else 1) + 50)
                    + (ranges * M * N / 512 if planes else 0))
            if best is None or cost < best[0]:
                best = cost, nf, ranges
    return best and best[1:]


def rows_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """Layout and alignment the row-streaming kernel needs (16-byte loads of both)."""
    return (x.is_cuda and x.dtype == torch.bfloat16 == w.dtype and x.shape[1] == w.shape[1] and x.stride(1) == 1
            and x.stride(0) % 8 == 0 and w.is_contiguous() and x.data_ptr() % 16 == 0 == w.data_ptr() % 16)


def _rows_choice(x: torch.Tensor, w: torch.Tensor, M: int, N: int, K: int, out: int):
    """:func:`rows_plan` of operands that lie as the kernel needs them (asked last: prompts pay for one comparison)."""
    return rows_plan(M, N, K, out) if 0 < M <= ROWS_MAX_M and rows_ok(x, w) else None


def gemm_rows(x: torch.Tensor, w: torch.Tensor, nf: int, out_kind: int = ROWS_BF16, ranges: int = 1,
              out: torch.Tensor = None) -> torch.Tensor:
    """``x @ w.T`` of up to 32 rows on the row-streaming kernel: bf16, fp32 (with ``ranges`` as planes [ranges, M, N]),
    SwiGLU (w = [Wg; Wu]) or squared relu."""
    M, K = x.shape
    N = w.shape[0] // (2 if out_kind == ROWS_SILU else 1)
    if out is None:
        out = torch.empty((ranges, M, N) if ranges > 1 else (M, N), device=x.device,
                          dtype=torch.float32 if out_kind == ROWS_F32 else x.dtype)
    check(lib().k8s_gemm_rows(ptr(x), x.stride(0), ptr(w), ptr(out), out.stride(-2), M, N, K, nf, ranges, out_kind,
                              stream_ptr(x)), "gemm_rows")
    return out

# ------------------------------------------------- products of 17 to 64 rows (csrc/kernels/gemm_batch.hip)
BATCH_ROWS = 16, 64     # more than, up to


@functools.lru_cache(maxsize=4096)
def batch_plan(M: int, N: int, K: int, out: int = ROWS_BF16, planes: bool = False):
    """(16-row fragments of a workgroup, K ranges) with which that kernel takes a product of ``N`` result columns, or None; ``planes``: K
    ranges may stay apart.

    Two fragments while their strips are one wave of 256 workgroups, else four.  What it costs grows with the rows (every workgroup
    reads them all), the other kernels' cost by steps at 32 rows.  Time over that of the stream kernel, of the row-streaming kernel
    up to 32 rows, or of the library, by whichever had it, at 24, 32 | 40, 48, 56, 64 rows:
    SwiGLU 8192 x 2048 0.96, 0.95 | 0.81, 0.81, 0.89, 0.92;  4096 x 2048 0.92, 0.88 | 0.82, 0.80, 0.91, 0.92;  6144 x 2048 (0.75 waves of
    four fragments) 0.86, 0.93 | 0.91, 0.93, 0.99, 1.02;  16384 x 2048 0.98, 0.96 | 0.82, 0.84, 0.86, 0.92;  8192 x 4096 0.93, 0.96 |
    0.77, 0.65, 0.82, 0.87;  3072 x 1024 0.78, 0.76 | 0.86, 0.91, 0.95, 0.98;  8192 x 1024 0.94, 0.93 | 1.07, 1.05, 1.15, 1.17;  1024 x
    512 0.82, 0.87 | 1.06 - 1.14;  4096 x 8192 0.96, 0.97 | 0.92 - 0.97.  A long
    K over few strips is the library's, which cuts it (weights out of memory, at 17, 28 | 40, 48 | 56 rows): 512 x 5632 0.99, 1.07 | 1.26,
    1.33 | 1.41, x 8192 1.10, 1.20 | 1.36, 1.39 | 1.47;  1024 x 5120 0.67, 0.72 | 0.99, 1.08 | 1.18, x 6144 0.98, 1.04 | 0.92, 0.97 | 1.07, x 8192
    1.00, 1.08 | 1.27, 1.21 | 1.36;  1408 x 6144 0.70, 0.76 | 0.86, 0.91 | 0.98, x 8192 0.96, 0.99 | 0.91, 0.93 | 1.05;  2304 x 8192 0.71,
    0.80 | 0.57, 0.58 | 0.86.  More than a wave of four
    fragments (8256, 10240, 12288 | 14336 at 17, 20, 24 rows), x 768 1.04, 1.02, 0.98, 1.04, 1.02, 0.97, 1.10, 1.07, 1.02 | 0.97, 0.98, 0.96, x 2048
    1.03, 1.01, 0.99, 1.01, 1.00, 0.99, 1.05, 1.05, 1.01 | 0.97, 0.97, 0.98: up to there the row-streaming kernel has two of them.  Squared relu 8192 x 2048 0.88, 0.86 | 0.81, 0.84, 0.90, 0.91, x
    4096 0.84, 0.86 | 0.71 - 0.83;  16384 x 2048 0.89, 0.95 | 0.69 - 0.77;  4096 x 512 0.77, 0.82 | 1.03 - 1.09.  bf16 2560 x 2048 0.70,
    0.75 | 0.79 - 0.92;  1024 x 2048 0.76, 0.80 | 0.91, 0.97, 1.04, 1.09;  4096 x 4096 0.82, 0.90 | 0.97, 1.02, 1.12, 1.06;  8192 x 1024
    0.89, 0.87 | 0.87 - 0.97;  2048 x 1024 0.75, 0.78 | 0.95, 0.97, 1.04, 1.07.  fp32 2576 x 2048 0.92, 0.88 | 0.80 - 0.92;  8736 x
    2048 0.83, 0.77 | 0.92, 0.95, 1.01, 1.03;  32768 x 2048 0.99, 0.99 | 0.95, 0.96, 1.03, 1.05;  50256 x 4096 0.94, 0.96 | 1.01 - 1.13.
    Planes with the pass behind, by K ranges, over 512 to 4096 columns, weights out of memory: eight 0.80 - 0.99 at every number of rows;
    four 0.80 - 0.98 up to 32 rows (2048 x 8192 0.93), 0.91 - 1.01 up to 48, past that 0.93 - 1.05 (8192 entries of K 1.00 - 1.05);  two, which
    is all that 2560, 3584, 4608 and 7680 allow, leave up to 2048 columns on few units: at 17, 24, 32 | 48 rows 1024 x 2560 0.96, 1.00,
    1.02 | 1.12, x 3584 0.94, 0.97, 0.99 | 1.10, x 4608 1.02, 1.05, 1.08 | 1.18, x 7680 1.10, 1.20, 1.25 | 1.37 (but x 1536 0.94 - 0.97);  two
    of more than 2048 columns, whose strips fill the units, 0.74 - 0.99 up to 32 rows, 0.84 - 0.99 past them with K up to 3584, from
    4096 on 0.94 - 1.10."""
    big = N * (2 if out == ROWS_SILU else 1)
    if not BATCH_ROWS[0] < M <= BATCH_ROWS[1] or N % 16 or big < 512 or K % 256 or not 512 <= K <= 8192:
        return None
    few = M <= 32
    if planes:
        if N > 4096 or K < (1024 if few else 2048):
            return None
        ranges = 8
        while ranges > 1 and (-(-N // 32) * ranges > 256 or K % (256 * ranges)):
            ranges //= 2
        if ranges == 1:
            return None
        if ranges == 4 and M > 48:                   # (more planes to read than gain)
            return None
        if ranges == 2 and N <= 2048 and (not few or K > 2048 and (M > 24 or K >= 4096)):      # K that more ranges do not divide
            return None
        if ranges == 2 and not few and K >= 4096:
            return None
        return 2, ranges
    if K > 4096 and out != ROWS_SILU:
        return None
    nf = 2 if big <= 8192 else 4
    if out == ROWS_SILU and N % (8 * nf):
        return None
    if K >= 5120 and big <= (4096 if M > 48 else 2560 if not few else 2048 if K > 5120 else 0):
        return None                                  # a long K over few strips, which the library cuts
    if few:
        if M <= 24 and big > 16384 and (out < ROWS_SILU and K <= 2048
                                        or out >= ROWS_SILU and big <= 24576 and rows_plan(M, N, K, out) == (2, 1)):
            return None                              # up to one and a half waves of strips: the row-streaming kernel's two fragments
        return nf, 1
    if K < 2048:
        return (nf, 1) if K >= 1024 and 6144 <= big <= 8192 else None
    if out >= ROWS_SILU:
        return (nf, 1) if M <= 48 or not 8192 < big < 15360 or out == ROWS_RELU2 else None
    if K > 2048 or M > 48 and (big < 2048 or 8192 < big < 15360 or big > 16384):
        return None
    return nf, 1


def _batch(x: torch.Tensor, w: torch.Tensor, out: int, planes: bool = False):
    """That product (planes [ranges, M, N]), or None."""
    M, K = x.shape
    if not BATCH_ROWS[0] < M <= BATCH_ROWS[1] or K != w.shape[1] or not planes and (w.shape[0], K) in _dispatch:
        return None
    if not (_few_ok(x, w) and K <= x.stride(0) <= 1 << 24) or out == ROWS_SILU and w.shape[0] % 2:
        return None
    N = w.shape[0] // (2 if out == ROWS_SILU else 1)
    plan = batch_plan(M, N, K, out, planes)
    if plan is None:
        return None
    f32 = out == ROWS_F32
    y = torch.empty((plan[1], M, N) if planes else (M, N), dtype=torch.float32 if f32 else x.dtype, device=x.device)
    check(lib().k8s_gemm_batch(ptr(x), x.stride(0), ptr(w), ptr(y), N, M, N, K, plan[0], plan[1], out, stream_ptr(x)), "gemm_batch")
    return y


def select_gemm(M: int, N: int, K: int, x_ok_layout: bool = True, out_contig: bool = True,
                rows: bool = True, out_wide: bool = True) -> Tuple[int, int, int]:
    """(kind, cfg, splits) :func:`linear` runs for a contiguous bf16 ``x`` [M, K]
    and ``w`` [N, K] on the GPU -- the measured dispatch table first, then the
    row-streaming kernel and the skinny kernel's default range, else hipBLASLt.  Also used by the native
    layer executor (ops/layer_exec.py) so both paths pick the same kernel.
    ``rows``: x and w lie as the row-streaming kernel needs them; ``out_wide``: the result can be stored by 16 bytes, as the
    sum of K ranges is."""
    forced_skinny = False
    rows = rows and x_ok_layout
    if _dispatch and M <= DISPATCH_MAX_M:
        ent = _lookup(N, K, M)
        if ent is not None:
            kind, cfg, splits = ent
            if kind == "mid" and x_ok_layout and _mid_shape_ok(M, N, K, cfg, splits):
                return KIND_MID, cfg, splits
            if kind == "grp" and x_ok_layout and out_contig and N % 128 == 0 and K % (64 * splits) == 0:
                return KIND_GRP, 0, splits
            if kind == "stream" and x_ok_layout and out_contig and stream_shape_ok(M, N, K, cfg, splits):
                return KIND_STREAM, cfg, splits
            if kind == "rows" and rows and (splits == 1 or out_wide) and rows_shape_ok(M, N, K, cfg, splits):
                return KIND_ROWS, cfg, splits
            if kind == "lib":
                return KIND_LIB, 0, 1
            forced_skinny = kind == "skinny" and M <= 128
    if M > DISPATCH_MAX_M and x_ok_layout:
        big_splits = _big_pick(M, N, K)
        if big_splits:
            return KIND_BIG, BIG_PIPE, big_splits
    if rows and not forced_skinny:
        plan = rows_plan(M, N, K)
        if plan is not None:
            return KIND_ROWS, plan[0], 1
    if (_enabled and (M == 1 or forced_skinny or (M <= SKINNY_MAX_M and N * K <= SKINNY_MAX_NK))
            and x_ok_layout and K % 256 == 0 and N % 16 == 0):
        return KIND_SKINNY, 0, 1
    return KIND_LIB, 0, 1


# fp32 products of a few rows (csrc/kernels/few_rows_f32.hip).  Up to 8 rows, for wide weights up to 5: each row is read by
# every workgroup, so past that a wide weight is no faster.  us, library / this at 1, 2, 4, 8 rows: 2048 x 2048 12.0 / 4.9,
# 12.1 / 5.2, 12.1 / 5.8, 12.2 / 7.1;  2048 x 8192 22.9 / 12.5, 23.3 / 12.7, 22.9 / 13.5, 23.3 / 17.2;  3072 x 768 7.2 / 3.8,
# 8.4 / 4.1, 8.3 / 4.4, 7.3 / 5.3;  16384 x 2048 31.7 / 20.7, 32.0 / 20.7, 31.8 / 24.1, 32.2 / 30.8;  8192 x 2048 at 5, 6, 8
# rows 16.2 / 14.9, 16.2 / 16.2, 16.4 / 17.5.  (16384 x 2048 at 20.7 is 6.5 TB/s: part of the weights stays in the caches.)
FEW_F32_ROWS = 8
FEW_F32_WIDE = 8192, 5


def _few_f32_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    (M, K), N = x.shape, w.shape[0]
    return (x.is_cuda and w.is_cuda and x.dtype == torch.float32 == w.dtype
            and 0 < M <= (FEW_F32_WIDE[1] if N >= FEW_F32_WIDE[0] else FEW_F32_ROWS) and N > 0 and K > 0 and K % 4 == 0
            and w.dim() == 2 and w.shape[1] == K and unwatched(x, w) and w.is_contiguous() and w.data_ptr() % 16 == 0
            and x.stride(1) == 1 and x.stride(0) % 4 == 0 and x.stride(0) >= K and x.data_ptr() % 16 == 0
            and x.stride(0) < 2 ** 31)


# fp32 products of many rows as bf16 ones (csrc/kernels/gemm_split_f32.hip)
SPLIT_ROWS = 128, 4096
SPLIT_TILES = (4, 6, 8, 10, 12)      # 16-row fragments of a tile


@functools.lru_cache(maxsize=4096)
def split_plan(M: int, N: int, K: int, planes: bool = False, glu: bool = False):
    """(16-row fragments of a tile, K ranges) with which an fp32 product of many rows is quicker as products of bf16 parts than
    on the library, or None.  ``N``: rows of the weight; ``planes``: K ranges may stay apart.

    A step of a workgroup (K 32) takes some 0.5 us and 0.13 a fragment, less the fewer of them a compute unit has at once; the
    rows' split is a pass of 4 us and their bytes, each range writes and reads the result once more; and the library takes its
    operations at 120 TFLOP/s and a start.  us library / the split and this:  16384 x 2048 at 333, 622, 1024 rows 210 / 150,
    380 / 231, 515 / 341, at 166 104 / 99;  8192 x 2048 at the same 103 / 93, 183 / 131, 257 / 182, 59 / 84;  2048 x 8192 (eight
    ranges, without the bytes of their sums) 107 / 87, 176 / 124, 246 / 207;  2048 x 2048 31 / 31, 46 / 43, 65 / 60;  2560 x
    2048 at 1024 93 / 74.  Over 54 sizes that it takes, with what stands behind, 0.74 of the time before, none past 1.02."""
    if not SPLIT_ROWS[0] <= M <= SPLIT_ROWS[1] or N < 512 or K < 512 or K % 32 or N % (128 if glu else 4):
        return None
    best = None
    for mt in SPLIT_TILES:
        for ranges in (1, 2, 4, 8) if planes else (1,):
            if K % (32 * ranges) or K // ranges < 256:
                continue
            load = -(-M // (16 * mt)) * -(-N // 128) * ranges / 256
            cost = K / 32 / ranges * (0.5 + 0.13 * mt) * max(1.15 + 0.2 * load, 0.55 + 0.7 * load, 0.95 * load)
            if ranges > 1:
                cost += ranges * M * N * 8 / 5e6
            if best is None or cost < best[0]:
                best = cost, mt, ranges
    cost = best[0] + 4 + M * K * 10 / 5e6
    return best[1:] if cost < 0.93 * (2 * M * N * K / 120e6 + 5) else None


def _split_f32(x: torch.Tensor, w: torch.Tensor, planes: bool = False, glu: bool = False):
    """The product as [ranges, M, N] (``glu``: [M, N / 2]), or None: another kernel is the quicker one or has to take it."""
    M = x.shape[0]
    if not SPLIT_ROWS[0] <= M <= SPLIT_ROWS[1] or w.dim() != 2 or x.shape[1] != w.shape[1]:
        return None
    N, K = w.shape
    plan = split_plan(M, N, K, planes, glu) if x.is_cuda and x.dtype == torch.float32 == w.dtype and w.is_cuda else None
    if plan is None or not unwatched(x, w) or not (
            w.is_contiguous() and w.data_ptr() % 16 == 0 == x.data_ptr() % 16 and x.stride(1) == 1 and x.stride(0) % 4 == 0
            and K <= x.stride(0) < 2 ** 31 and w.device == x.device):
        return None
    parts = torch.empty(3 * M * K + 2 * M, dtype=torch.bfloat16, device=x.device)      # and an fp32 factor a row
    p, f = ptr(parts), ptr(parts) + 6 * M * K
    check(lib().k8s_split_rows_f32(ptr(x), x.stride(0), p, f, M, K, stream_ptr(x)), "split_rows_f32")
    if glu:
        out = torch.empty(M, N // 2, dtype=torch.float32, device=x.device)
        check(lib().k8s_gemm_split_glu_f32(p, f, ptr(w), ptr(out), M, N // 2, K, plan[0], stream_ptr(x)), "gemm_split_glu_f32")
        return out
    out = torch.empty(plan[1], M, N, dtype=torch.float32, device=x.device)
    check(lib().k8s_gemm_split_f32(p, f, ptr(w), ptr(out), M, N, K, *plan, stream_ptr(x)), "gemm_split_f32")
    return out


def linear(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor = None) -> torch.Tensor:
    """``x @ w.T`` for ``x`` [M, K] and ``w`` [N, K]."""
    M, K = x.shape
    N = w.shape[0]
    if not (x.is_cuda and x.dtype == torch.bfloat16):
        if out is None and _few_f32_ok(x, w):
            out = torch.empty((M, N), dtype=torch.float32, device=x.device)
            check(lib().k8s_few_rows_f32(ptr(x), x.stride(0), ptr(w), ptr(out), M, N, K, stream_ptr(x)), "few_rows_f32")
            return out
        if out is None:
            y = _split_f32(x, w)
            if y is not None:
                return y[0]
        return lib_gemm(x, w, out)
    layout = x.stride(1) == 1 and x.stride(0) % 8 == 0 and w.is_contiguous()
    rows = M <= ROWS_MAX_M and rows_ok(x, w) and (out is None or out.stride(1) == 1)
    wide = out is None or out.stride(0) % 8 == 0 == out.data_ptr() % 16
    kind, cfg, splits = select_gemm(M, N, K, layout, out is None or out.is_contiguous(), rows, wide)
    if kind == KIND_ROWS:
        if splits == 1:
            return gemm_rows(x, w, cfg, out=out)
        part = _scratch(x.device, splits * M * N)
        check(lib().k8s_gemm_rows(ptr(x), x.stride(0), ptr(w), ptr(part), N, M, N, K, cfg, splits, ROWS_F32, stream_ptr(x)),
              "gemm_rows")
        if out is None:
            out = torch.empty((M, N), dtype=x.dtype, device=x.device)
        check(lib().k8s_gemm_stream_reduce(ptr(part), splits, ptr(out), out.stride(0), M, N, stream_ptr(x)), "gemm_reduce")
        return out
    if kind == KIND_MID:
        return gemm_mid(x, w, cfg, splits, out)
    if kind == KIND_GRP:
        return gemm_grp(x, w, splits, out)
    if kind == KIND_STREAM:
        return gemm_stream(x, w, cfg, splits, out)
    if kind == KIND_BIG:
        return gemm_big(x, w, out, pipe=cfg, splits=splits)
    if kind == KIND_SKINNY:
        if out is None:
            out = torch.empty((M, N), dtype=x.dtype, device=x.device)
        check(lib().k8s_gemm_skinny(ptr(x), x.stride(0), ptr(w), ptr(out), out.stride(0), M, N, K,
                                    stream_ptr(x)), "gemm_skinny")
        return out
    return lib_gemm(x, w, out)


# ------------------------------------------------------------ library GEMM
# Native hipBLASLt front end (csrc/kernels/blaslt.hip): descriptors and the
# heuristic's algorithm cached per shape, so a call costs a hash lookup plus
# hipblasLtMatmul instead of F.linear's ~28 us of host time.
BLASLT_WS_BYTES = 64 << 20
_blaslt_ws = {}
_native_lib_gemm = KNOBS.native_blaslt


_lib_tuned: Dict[Tuple[int, int], List[Tuple[int, int]]] = {}    # rows (from, to) of weights with a measured solution


def row_cut(M: int, N: int, K: int, tuned: bool = False) -> int:
    """Rows of a library product that go into a launch of their own because their 256 x 256 tiles are whole waves of the 256
    compute units (the rest follows in a second one), or 0.  For some tiles more than whole waves the library takes a wave
    more, or smaller tiles for all of them.  us whole / cut:  2048 x 2048 added to fp32 at 17000 rows (2.09 waves) 172 / 150,
    24730 (3.03) 246 / 218;  2048 x 8192 at 16500 641 / 434, 24730 743 / 639, but 20000 (2.47) 726 / 542 and 22000 (2.69)
    765 / 579;  8192 x 2048 in bf16 at 2100 (1.12) 85 / 64, 12000 (5.88) 389 / 295, 24730 629 / 592, 3300 (1.62) 94 / 95;
    2560 x 2048 at 27000 (4.14) 313 / 261, 22000 (3.36) 218 / 246;  4096 x 14336 at 4123 (1.06) 730 / 367.  So up to 0.15 of
    a wave where the columns are up to 24 tiles that they nearly fill (past that the tiles of a row leave too little to gain:
    28672 x 256 at 1704 43 / 67, 8736 x 4096 at 11027 685 / 778, 1088 x 512 at 14181 35 / 43) or divide a wave;  further where
    they divide it and are many or K is long, past two waves (three of tiles of which a wave is two rows) and with a K from
    1024 on (32768 x 4096 at 540, 1.5 waves, 150 / 177, x 1024 at 1109, 2.5, 95 / 110, 8192 x 512 at 19744 186 / 207).  What
    the library takes for a size is not to be foreseen: over 452 random sizes that this cuts 0.89 of the time, 32 of them past
    1.02 (8192 x 384 at 2284 30 / 37, 2560 x 14336 at 19632 1128 / 1350).  ``tuned``: a call that takes measured solutions,
    which stay with the rows they were measured for."""
    nt = -(-N // 256)
    full, over = divmod(-(-M // 256) * nt, 256)
    if full < 1 or not over or tuned and any(lo <= M <= hi for lo, hi in _lib_tuned.get((N, K), ())):
        return 0
    most = 0.15
    if 256 % nt == 0 and N % 256 == 0:
        most = 1.0 if full > 1 + (nt > 64) and K >= 1024 and (nt >= 32 or K >= 4096) else most
    elif nt > 24 or 10 * N < 9 * 256 * nt:
        return 0
    return full * 256 // nt * 256 if over <= most * 256 else 0


def _row_parts(M: int, N: int, K: int, tuned: bool = False) -> Tuple[Tuple[int, int], ...]:
    if M * N < 256 << 16:                # less than a wave
        return ((0, M),)
    cut = row_cut(M, N, K, tuned)
    return ((0, cut), (cut, M)) if 0 < cut < M else ((0, M),)


def lib_gemm(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor = None) -> torch.Tensor:
    """``x @ w.T`` on hipBLASLt (bf16, fp32 accumulate)."""
    if (_native_lib_gemm and x.is_cuda and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
            and x.stride(1) == 1 and w.is_contiguous() and (out is None or out.stride(1) == 1)):
        M, K = x.shape
        N = w.shape[0]
        if out is None:
            out = torch.empty((M, N), dtype=x.dtype, device=x.device)
        if M == 0:
            return out
        ws = _blaslt_ws.get(x.device)
        if ws is None:
            ws = _blaslt_ws[x.device] = torch.empty(BLASLT_WS_BYTES, dtype=torch.uint8, device=x.device)
        ldx, ldo = x.stride(0), out.stride(0)
        for a, b in _row_parts(M, N, K, True):
            check(lib().k8s_blaslt_gemm(ptr(x) + 2 * a * ldx, ldx, ptr(w), ptr(out) + 2 * a * ldo, ldo, b - a, N, K, ptr(ws),
                                        BLASLT_WS_BYTES, stream_ptr(x)), "blaslt_gemm")
        return out
    if out is None:
        return F.linear(x, w)
    return torch.matmul(x, w.t(), out=out)


def linear_f32out(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``x @ w.T`` with fp32 output (bf16 operands, fp32 accumulate): the
    lm_head, whose logits the sampler reads in fp32."""
    if x.is_cuda and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.stride(1) == 1 \
            and w.is_contiguous():
        M, K = x.shape
        N = w.shape[0]
        y = _batch(x, w, ROWS_F32)
        if y is not None:
            return y
        plan = _rows_choice(x, w, M, N, K, ROWS_F32)
        if plan is not None:
            return gemm_rows(x, w, plan[0], ROWS_F32)
        out = torch.empty((M, N), dtype=torch.float32, device=x.device)
        if M == 0:  # a step whose chunks all end mid-prompt samples no row
            return out
        ws = _blaslt_ws.get(x.device)
        if ws is None:
            ws = _blaslt_ws[x.device] = torch.empty(BLASLT_WS_BYTES, dtype=torch.uint8, device=x.device)
        ldx = x.stride(0)
        for a, b in _row_parts(M, N, K):
            check(lib().k8s_blaslt_gemm2(ptr(x) + 2 * a * ldx, ldx, ptr(w), ptr(out) + 4 * a * N, N, b - a, N, K, ptr(ws),
                                         BLASLT_WS_BYTES, stream_ptr(x), 1, 1.0), "blaslt_gemm_f32out")
        return out
    return x.float() @ w.float().t()


SKINNY_F32_MAX_M = 32
# rows x columns of the skinny kernel's fp32 form: every 16-column workgroup reads all rows again, so a wide weight leaves it
# at fewer rows (us, hipBLASLt / skinny: 8192 x 2048 at 16 rows 13.0 / 10.9, at 32 12.9 / 15.4; 8736 x 2048 at 7 / 16 / 32
# 14.2 / 12.2, 14.2 / 14.4, 14.3 / 21.2; 2560 x 2048 at 32 9.8 / 8.0)
SKINNY_F32_MAX_MN = 144 * 1024
# ... where K is long; the rows of a short one are little to read (8192 x 1024 at 32 rows 11.9 / 9.3, x 512 at 24 9.4 / 6.7)
SKINNY_F32_SHORT_K, SKINNY_F32_SHORT_MN = 1024, 256 * 1024


def _skinny_f32(M: int, N: int, K: int) -> bool:
    return (_enabled and 0 < M <= SKINNY_F32_MAX_M and N * K <= SKINNY_MAX_NK and K % 256 == 0 and N % 16 == 0
            and M * N <= (SKINNY_F32_SHORT_MN if K <= SKINNY_F32_SHORT_K else SKINNY_F32_MAX_MN))


STREAM_F32_MAX_M = 64


def stream_f32_cfg(M: int, N: int, K: int) -> int:
    """The stream kernel's form for a product of 17 to 64 rows with an fp32 result that neither :func:`batch_plan` nor the
    row-streaming nor the skinny kernel takes, or 0: the library.  Strips of 32 columns within one wave of workgroups, then of 64 where they fill their waves.
    us of the library / this at 33, 64 rows:  2304 x 2048 8.8 / 8.6, 9.2 / 8.6;  2576 x 2048 9.0 / 8.7, 9.3 / 8.8;  2304 x 1024 8.6 /
    5.7, 8.9 / 5.8;  6144 x 2048 10.1 / 8.8, 10.0 / 8.9;  8192 x 2048 12.8 / 10.9, 13.2 / 11.4;  8736 x 2048 14.7 / 12.7, 14.9 / 13.3;
    12288 x 1024 9.9 / 7.6, 9.7 / 7.9;  16384 x 2048 18.2 / 17.7, 18.4 / 17.8;  32768 x 2048 36 / 31, 36 / 32;  65536 x 1024 32 / 28, 36 /
    32;  at 17 rows 5136 x 2048 12.0 / 8.7, 12304 x 2048 16.7 / 13.8.  Not: 1088 x 2048 8.6 / 8.6, 576 x 2048 5.7 / 8.4, 2048 x 4096 9.5 /
    14.1, 20480 x 1536 (1.25 waves) 18.0 / 19.1, 24576 x 2048 (1.5) 26.2 / 26.4, 50256 x 2048 (3.07) 50.6 / 52.3;  2576 x 2048 at
    97 rows 9.8 / 10.9.  And the library's front end takes 12 us more of the host a call."""
    if not (16 < M <= STREAM_F32_MAX_M and N >= 2304 and N % 16 == 0 and 1024 <= K <= 2048 and K % 64 == 0):
        return 0
    if N <= 32 * NARROW_WGS:
        return 34
    strips = -(-N // 64)
    return 14 if strips <= 256 or 20 * strips >= 19 * 256 * -(-strips // 256) else 0


def proj_f32out(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``x @ w.T`` with an fp32 result: bf16 operands with fp32 accumulation (the weight-streaming kernels for up to 64
    rows, hipBLASLt otherwise), or fp32 throughout."""
    if not x.is_cuda or x.dtype != torch.bfloat16:
        return linear(x, w)
    M, K = x.shape
    N = w.shape[0]
    y = _batch(x, w, ROWS_F32)
    if y is not None:
        return y
    plan = _rows_choice(x, w, M, N, K, ROWS_F32)
    if plan is not None:
        return gemm_rows(x, w, plan[0], ROWS_F32)
    if (_skinny_f32(M, N, K) and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and w.dtype == torch.bfloat16 and w.is_contiguous()):
        out = torch.empty((M, N), dtype=torch.float32, device=x.device)
        check(lib().k8s_gemm_skinny_f32(ptr(x), x.stride(0), ptr(w), ptr(out), N, M, N, K, stream_ptr(x)),
              "gemm_skinny_f32")
        return out
    cfg = stream_f32_cfg(M, N, K) if 16 < M <= STREAM_F32_MAX_M else 0
    if cfg and (N, K) not in _dispatch and K == w.shape[1] and _few_ok(x, w):
        out = torch.empty((M, N), dtype=torch.float32, device=x.device)
        check(lib().k8s_gemm_stream_f32(ptr(x), x.stride(0), ptr(w), ptr(out), M, N, K, cfg, stream_ptr(x)), "gemm_stream_f32")
        return out
    return linear_f32out(x, w)


# -------------------------------------------------- products of a few rows by their shape
# The stream kernel on 32-column strips (csrc/kernels/gemm_stream.hip): twice the workgroups of the 64-column form, so a
# weight of 2k..8k rows puts one on each of the 256 compute units without cutting K.
NARROW_WGS = 256        # strips one wave of workgroups holds; more of them lose to the wider strips
NARROW_MAX_M = 128      # two 16-row fragments per wave


def _narrow_cfg(M: int) -> int:
    """Stages of the 32-column form: 6 up to 32 rows, 4 above (us at 8192 x 2048, 6 / 4 stages: 1 row 10.0 / 10.4, 32 rows
    10.2 / 10.6, 64 rows 11.4 / 11.1, 128 rows 14.7 / 13.7)."""
    return 36 if M <= 32 else 34


def plane_plan(M: int, N: int, K: int):
    """(stream configuration, K ranges) of :func:`proj_planes`, (ROWS_CFG + fragments, K ranges) where the row-streaming kernel
    takes it, (BATCH_CFG + fragments, K ranges) :func:`batch_plan`'s; one range: the product is not cut.  The other forms: 2048 columns are 32 or
    64 strips for 256 compute units, so K is cut until each has a workgroup: four ranges of 32-column strips where K is
    short, eight of 64-column strips from 4096 on.  us with cold weights at 1 / 16 / 64 / 128 rows: 2048 x 2048 hipBLASLt
    8.1 / 8.3 / 8.9 / 8.8, the skinny kernel 4.9 / 6.2 / 11.7 / --, 64-column planes 4.2 / 4.5 / 5.5 / 7.2, 32-column
    planes 4.1 / 4.4 / 4.8 / 6.6 and half as many to read;  2560 x 2048 32-column planes 5.0 / 5.3 / 6.8 / 10.0 against
    10.5 / 11.7 / 12.5 / 15.9;  2048 x 8192 12.4 / 12.5 / 21.8 / 20.8, 12.6 / 17.5 / 38 / --, 64-column 8.7 / 9.2 / 10.0 /
    12.8, 32-column 9.9 / 10.0 / 11.5 / 15.6.

    Up to 16 rows the skinny kernel leaves the planes only where K is long for the columns, up to 32 where it is more than a
    strip or two.  us with the pass behind, skinny / planes:  1024 x 512 at 1 / 16 rows 4.8 / 5.6, 5.5 / 6.1, x 1536 6.6 /
    6.4, 7.7 / 6.8;  2048 x 1024 5.7 / 6.1, 6.8 / 6.4;  4096 x 1024 6.2 / 7.6, 7.3 / 7.9, x 3072 10.6 / 13.3, 12.0 / 12.5, x
    6144 16.0 / 15.3, 18.6 / 15.5, x 8192 18.8 / 22.7, 22.1 / 22.5;  5120 x 1024 7.2 / 8.5, 9.2 / 9.0, x 2048 10.5 / 10.9,
    13.3 / 11.7;  2048 x 256 at 24 rows 5.6 / 6.1."""
    plan = batch_plan(M, N, K, ROWS_F32, True)
    if plan is not None:
        return BATCH_CFG + plan[0], plan[1]
    plan = rows_plan(M, N, K, ROWS_F32, True) if M <= ROWS_MAX_M else None
    if plan is not None:
        return ROWS_CFG + plan[0], plan[1]
    return _plane_plan(M, N, K, _enabled) if 0 < M <= NARROW_MAX_M else _more_rows_plan(M, N, K)


ROWS_CFG = 100      # past every stream configuration
BATCH_CFG = 200     # past those


@functools.lru_cache(maxsize=4096)      # (asked for every product of a step; 1.2 us of the host worked out, 0.2 looked up)
def _plane_plan(M: int, N: int, K: int, skinny: bool):
    if skinny and _skinny_f32(M, N, K):
        long_k = (1024 if M > 8 else 1536) if N <= 2048 else 1536 if N > 4096 else 3072 if M > 8 else 4096
        if K <= 256 if M > 16 else K < long_k or N * K >= 1 << 25:
            return 14, 1
    cfg, bn, s, most = (34, 32, 4, 320) if K < 4096 else (14, 64, 8, 256)
    while s > 1 and (-(-N // bn) * s > most or K < 128 * s or not stream_shape_ok(M, N, K, cfg, s)):
        s //= 2
    return cfg, s


def _more_rows_plan(M: int, N: int, K: int):
    """The same for 129 to 256 rows: a long K over few columns, which the library does not cut.  us of the library / of 64-column planes
    at 129, 192, 256 rows:  2048 x 8192 26.6 / 14.8, 26.6 / 16.5, 28.8 / 19.7;  4096 x 4096 22.4 / 14.8, 33.0 / 16.2, 22.8 / 19.5;  4096 x 14336
    65.6 / 38.0, 104 / 43, 69.6 / 50.4.  Not 2048 x 2048 9.3 / 7.3, 9.4 / 8.1, 9.9 / 10.5 and 1024 x 2048 8.4 / 6.6, 8.5 / 6.9, 8.9 / 8.9: the
    pass behind has eight planes to read.  Nor few columns, which the library does cut, of a long K or past 192 rows (three stages of
    the ring; one strip is the same either way), with that pass at 129, 192, 193, 256 rows:  64 x 4096 13.8 / 11.7, 13.7 / 12.3, 13.8 / 14.0,
    13.8 / 14.1;  256 x 4096 14.0 / 11.8, 13.8 / 12.6, 13.9 / 14.4, 13.9 / 14.6, x 8192 14.4 / 15.6, 14.1 / 16.9, 14.2 / 19.6, 14.2 / 19.9;  512 x
    8192 16.2 / 16.9, 17.4 / 17.7, 16.6 / 20.0, 17.1 / 20.8;  768 x 8192 16.6 / 16.9, 23.5 / 18.4, 23.4 / 20.7, 22.6 / 21.7;  1024 x 4096 15.8 /
    13.9, 16.0 / 15.4, 15.9 / 17.1, 16.0 / 18.2;  1280 x 4096 16.1 / 14.6, 16.3 / 16.4, 17.9 / 17.9, 19.4 / 18.0."""
    strips = -(-N // 64)
    if (not NARROW_MAX_M < M <= DISPATCH_MAX_M or K < 4096 or N > 4096 or strips < 8 and K > 5120
            or M > 192 and 1 < strips < (20 if K <= 5120 else 12)):
        return 14, 1
    cfg, s = 14 if M <= 192 else 13, 8
    while s > 1 and (-(-N // 64) * s > 256 or K < 512 * s or not stream_shape_ok(M, N, K, cfg, s)):
        s //= 2
    return cfg, s


def proj_planes(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``x @ w.T`` in fp32 as planes [S, M, N] whose sum over S is the product (bf16 operands, fp32 accumulation): for
    consumers that read it once and add the planes on the way in.  S = 1 wherever the planes do not pay."""
    M, K = x.shape
    N = w.shape[0]
    if _few_ok(x, w):
        cfg, S = plane_plan(M, N, K)
        if cfg > BATCH_CFG:
            y = _batch(x, w, ROWS_F32, True)
            if y is not None:
                return y
            cfg, S = _plane_plan(M, N, K, _enabled)
        if cfg > ROWS_CFG and K == w.shape[1]:
            return gemm_rows(x, w, cfg - ROWS_CFG, ROWS_F32, S).view(S, M, N)
        if cfg > ROWS_CFG:
            cfg, S = _plane_plan(M, N, K, _enabled)
        if S > 1:
            out = torch.empty((S, M, N), dtype=torch.float32, device=x.device)
            check(lib().k8s_gemm_stream_part(ptr(x), x.stride(0), ptr(w), None, N, M, N, K, cfg, S, ptr(out),
                                             stream_ptr(x)), "gemm_stream_part")
            return out
    y = _split_f32(x, w, planes=True)
    return y if y is not None else proj_f32out(x, w)[None]


def _few_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    return (x.is_cuda and x.dtype == torch.bfloat16 == w.dtype and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and w.is_contiguous() and x.data_ptr() % 16 == 0 == w.data_ptr() % 16)


# Rows from which an output projection is added to the residual by the product itself, so that the norm behind it reads one
# fp32 row instead of two and writes none.  us, product + residual and norm apart / together: K 8192 at 5000 rows 164 / 170,
# 8102 246 / 231, 16384 509 / 465, 24730 856 / 800;  K 2048 at 2000 35 / 33, 8102 100 / 91, 16384 194 / 169, 24730 357 / 313
# (2048 columns; at 256 to 5120 columns and 6200 to 32000 rows nothing is slower together).
ADD_ROWS = 6144


def big_add_pays(M: int, N: int, K: int) -> bool:
    """Whether gemm_big adds a product to an fp32 residual quicker than the library, by how far its 256-row tiles fill their
    last wave of 256: whole waves, or a last one of two thirds, from the third on two fifths, with a K from 8192 on a fifth.
    us library / gemm_big, the residual out of memory, at waves of tiles:  2048 x 2048 at 0.50 53 / 59, 0.88 77 / 71, 1.28 112 /
    116, 1.47 119 / 120, 1.69 141 / 128, 2.00 154 / 144, 2.50 201 / 186, 3.00 220 / 204, 4.00 286 / 268;  2048 x 8192 at 0.69
    165 / 175, 0.88 210 / 194, 1.28 313 / 299, 1.47 341 / 327, 2.00 418 / 397, 3.00 620 / 589, 3.50 752 / 712;  4096 x 4096 at
    0.50 80 / 95, 0.88 119 / 110, 1.25 168 / 185, 1.44 190 / 199, 1.69 217 / 204, 2.50 427 / 302, 3.00 355 / 336, 4.00 462 / 462;
    4096 x 14336 at 0.75 286 / 310, 0.88 330 / 322, 1.25 488 / 459, 2.00 689 / 670;  1024 x 4096 at 1.47 197 / 210, 1.69 225 /
    215;  5120 x 2048 at 1.09 104 / 110, 1.64 141 / 127, 2.89 220 / 200."""
    if N % 256 or K % 128 or K < 2048:
        return False
    tiles = -(-M // 256) * (N // 256)
    if tiles <= 256:
        return tiles >= 196
    full, over = divmod(tiles, 256)
    return not over or over >= (51 if K >= 8192 else 102 if full >= 2 else 166)


def proj_add(r: torch.Tensor, x: torch.Tensor, w: torch.Tensor, scale: float = 1.0):
    """``r += scale * (x @ w.T)`` on an fp32 residual ``r`` [M, N] where that pays (the result is then None), else the
    product as :func:`proj_planes` leaves it, which the caller's next pass adds."""
    M, K = x.shape
    N = w.shape[0]
    if M < ADD_ROWS or not (_few_ok(x, w) and r.dtype == torch.float32 and r.is_contiguous()):
        return proj_planes(x, w)
    assert r.shape == (M, N)
    ws = _blaslt_ws.get(x.device)
    if ws is None:
        ws = _blaslt_ws[x.device] = torch.empty(BLASLT_WS_BYTES, dtype=torch.uint8, device=x.device)
    ldx = x.stride(0)
    for a, b in _row_parts(M, N, K):
        xa, ra = ptr(x) + 2 * a * ldx, ptr(r) + 4 * a * N
        if big_add_pays(b - a, N, K) and ra % 16 == 0:
            check(lib().k8s_gemm_big_add(xa, ldx, ptr(w), ra, N, b - a, N, K, float(scale), stream_ptr(x)), "gemm_big_add")
            continue
        check(lib().k8s_blaslt_gemm2(xa, ldx, ptr(w), ra, N, b - a, N, K, ptr(ws), BLASLT_WS_BYTES, stream_ptr(x), 2,
                                     float(scale)), "blaslt_gemm_add")
    return None


# -------------------- a prompt's products added to the residual, with what reads it next (csrc/kernels/gemm_add.hip)
THEN_NOTHING, THEN_DYT, THEN_SCALED = 0, 1, 2
# us of a wave of 256 tiles by rows of a tile / 32: at no K, and more for each entry of K (2048 columns at K 1024, 2048, 8192: 25,
# 38, 121 with 128 rows, 29, 45, 136 with 160, 32, 53, 160 with 192, 43, 70, 193 with 256)
ADD_WAVES = {4: (11.5, 0.01318), 5: (14.5, 0.0147), 6: (15.5, 0.0174), 8: (21.0, 0.0206)}
ADD_MIN_ROWS, ADD_MAX_N = 512, 5120


def _waves_time(waves: dict, M: int, N: int, K: int, f: int) -> float:
    full, over = divmod(-(-M // (32 * f)) * -(-N // 256), 256)
    t = waves[f][0] + waves[f][1] * K
    return full * t + ((0.75 + 0.25 * over / 256) * t if over else 0.0)


# us of a second launch: its own, and a chip that the first one leaves to drain.  (But whole waves of 256-row tiles with tanh go in
# two: inside an engine's prompts of 16000 and 16384 rows of 2048 columns, two launches / one 12.55 / 12.62 and 12.84 / 12.89 ms, 13.45 / 13.57 on
# another card, though one of them after the other takes 176 / 172 us.  With the norm left, with smaller tiles and from three waves on one is
# as quick or quicker: 19.10 / 19.06, 8.54 / 8.50, 19.04 / 19.04.)
CUT_US = 5.0


def _add_time(M: int, N: int, K: int, f: int) -> float:
    """With 4096 columns the 32 tiles an XCD has at a time are half of four row tiles' columns, and in every XCD the same half where
    their ranges begin with a group: half of the memory's channels.  us of one launch / of two that do not, with tanh: K 1024 at 16384 rows
    272 / 235, 2048 at 8192 165 / 154, at 16384 351 / 319, 4096 505 / 479, 8192 829 / 808."""
    t = _waves_time(ADD_WAVES, M, N, K, f)
    return t * 1.05 if N == 4096 and -(-M // (32 * f)) % 32 == 0 else t


@functools.lru_cache(maxsize=4096)
def add_plan(M: int, N: int, K: int, then: int):
    """Row ranges (from, to, rows of a tile / 32) in which :func:`gemm_add` makes a product of ``M`` rows, or None: the product and
    the pass behind it are the quicker.  Tiles that leave the least of their last wave of 256 idle, or whole waves of them and, where that
    is worth a second launch, other tiles, or (0) a product and a pass of its own, for the rest.  us of two launches of the same tiles / of
    one, with tanh:  12288 x 2048, K 1024 90 / 85, 10000 x 2048, K 2048 109 / 105, 8192 285 / 276, 16384 x 5120, K 2048 419 / 391;  of others:
    12288 x 2048, K 2048 123 / 116, 24576 x 1024 123 / 116, but 20000 x 2048, K 8192 542 / 574, 8192 x 3072 335 / 358.

    Taken by what the same work takes in whole waves of 256-row tiles, over what it takes so.  Time of product and pass over this,
    at 0.40 of the whole waves' rate 0.86 (with tanh) and 0.98 (scaled), 0.48 1.00 and 1.17, 0.55 0.98 - 1.08 and 1.00 - 1.14, 0.66
    1.13 - 1.18 and 1.25, 0.80 1.05 - 1.27 and 1.11 - 1.37, 1.00 1.01 - 1.19 and 1.01 - 1.27, over 1024 to 5120 columns and a K of
    1024 to 14336.  Without a norm there is the pass that reads it left (with its time, product and pass over both: at 0.55 0.95 -
    1.00, 0.66 1.01 - 1.06, 0.80 0.99 - 1.17, 0.85 1.00 - 1.20).  With a longer K the library has a wave that is not full the quicker; over
    product and pass with tanh, K 6144 at 0.52 0.96, 0.54 1.01, 0.59 1.06;  8192 at 0.52 0.92, 0.54 1.02, 0.55 1.08 (2048 columns) and 1.12
    (4096), 0.58 0.98, 0.59 1.05, 0.65 1.10;  11008 at
    0.52 - 0.57 0.90 - 0.99, 0.63 0.93, 0.65 1.11, 0.67 1.13 - 1.25;  14336 at 0.51 - 0.59 0.83 - 0.98, 0.63 0.94, 0.65 1.06, 0.67 1.12 and more.
    Without a norm, from ADD_ROWS on, there is the product that adds itself (0.82 0.90, 0.86 0.98 - 1.17, 1.00 0.96 - 1.08: it stays)."""
    if N % 256 or N > ADD_MAX_N or K % 64 or not 1024 <= K <= 16384 or M < ADD_MIN_ROWS or then == THEN_NOTHING and M >= ADD_ROWS:
        return None
    nt = N // 256
    best = min((_add_time(M, N, K, f), ((0, M, f),)) for f in ADD_WAVES)
    took = best[0]                                   # (of that or a cut, the second launch left out)
    for f in ADD_WAVES:
        for waves in range(1, -(-M // (32 * f)) * nt // 256 + 1):
            cut = 256 * waves // nt * 32 * f
            rest = M - cut
            if rest <= 0:
                break
            c, g = min((_add_time(rest, N, K, g), g) for g in ADD_WAVES)
            own = 10.0 + rest * N * K / 3.5e8 + rest * N / 2e5
            if rest < 512 and own < c:
                c, g = own, 0
            c += _add_time(cut, N, K, f)
            took = min(took, c)
            charge = -1.0 if then == THEN_DYT and f == g == 8 and 256 % nt == 0 else CUT_US
            best = min(best, (c + charge, ((0, cut, f), (cut, M, g))))
    whole = M * N / 2.0 ** 24 * (ADD_WAVES[8][0] + ADD_WAVES[8][1] * K)
    least = 0.5 + min(0.14, (0.0115 * max(0, min(K, 8192) - 4096) + 0.032 * max(0, K - 8192)) / 1024)
    return best[1] if whole >= (max(0.6, least) if then == THEN_NOTHING else least) * took else None


# The same of gemm_prep.hip (K 2048: 39 us with 128 rows, 48 with 160, 54 with 192, 65 with 256)
PREP_WAVES = {4: (12.5, 0.01318), 5: (16.5, 0.0147), 6: (18.0, 0.0174), 8: (22.0, 0.0206)}
PREP_MIN_ROWS = 1280


@functools.lru_cache(maxsize=4096)
def prep_plan(M: int, N: int, K: int, n: int = 0):
    """Rows of a tile / 32 with which csrc/kernels/gemm_prep.hip makes an attention's input product of ``M`` rows and ``N`` columns, of
    which the first ``n`` (0: all) are rotated, normed or paged, or None: product and pass apart are the quicker.  The tiles that leave the least of their last wave of 256 idle.  us apart / so, 16
    heads over 2 of 128 and K 2048, 2560 columns (rotated), 2576 (values mixed), 8736:  512 rows 23 / 39, 23 / 40, 36 / 49;  1024 31 / 36, 31 /
    37, 53 / 48;  1280 42 / 37, 43 / 38, 70 / 55;  2048 48 / 38, 49 / 39, 98 / 84;  3517 60 / 46, 63 / 48, 139 / 123;  4096 65 / 52, 71 / 54, 190 / 147;
    4850 74 / 62, 81 / 64, 207 / 164;  8192 112 / 95, 128 / 95, 332 / 275;  16384 237 / 176, 248 / 176, 614 / 515;  24730 345 / 239, 405 / 259, 940 /
    765.  K 1024 and 4096 at 1280 rows 36 / 27, 35 / 28, 54 / 39 and 58 / 56, 55 / 56, 110 / 87, at 4096 51 / 38, 56 / 39, 133 / 96 and 98 / 83, 104 /
    90, 378 / 274.  Whole waves with one size and the rest with another, in two launches, gain up to 3 % and lose up to 8.

    Taken by what the same work takes in whole waves of 256-row tiles, over what it takes so: the longer K, the better the library has a
    wave that is not full, and the fewer columns the pass has, the less there is to save.  us apart / so at 1280, 1536, 1800, 2048, 2600 rows
    (0.37, 0.43, 0.49, 0.55, 0.66 of the whole waves' rate):  2576 columns, K 3072 46 / 46, 48 / 47, 53 / 48, 57 / 49, 66 / 52;  4096 53 / 55, 55 / 56,
    61 / 58, 68 / 59, 77 / 63;  6144 66 / 74, 69 / 74, 77 / 76, 84 / 79, 105 / 86;  8192 77 / 89, 82 / 89, 93 / 97, 104 / 97, 123 / 106;  2560 with K 8192
    80 / 89, 83 / 89, 96 / 97, 101 / 100, 120 / 102.  2048 columns with 1536 for the pass (0.31, 0.36, 0.41, 0.46, 0.56): K 2048 34 / 36, 35 / 36, 37 / 37,
    37 / 36, 42 / 38;  4096 44 / 52, 45 / 54, 49 / 55, 51 / 55, 60 / 56;  8192 66 / 87, 68 / 87, 77 / 90, 80 / 91, 101 / 95."""
    if M < PREP_MIN_ROWS or K % 64 or not 1024 <= K <= 8192:
        return None
    t, f = min((_waves_time(PREP_WAVES, M, N, K, f), f) for f in PREP_WAVES)
    whole = M * N / 2.0 ** 24 * (PREP_WAVES[8][0] + PREP_WAVES[8][1] * K)
    least = 0.33 + (0.06 * max(0, min(K, 4096) - 2048) + 0.02 * max(0, K - 4096)) / 1024
    if K >= 2048 and n:
        least += min(0.1, 0.4 * (1 - n / N))
    return f if whole >= least * t else None


def gemm_add(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor, scale: float, plan, then: int, alpha: float = 0.0, nw=None,
             nb=None, rms=None, again=None):
    """``x += scale * (a @ w.T)`` on the fp32 residual ``x`` [M, N] by :func:`add_plan`; ``then`` the activations behind it:
    ``tanh(alpha x) nw + nb``, or ``x nw`` and the sums of squares of the rows in parts [M, N / 256].  ``rms = (ss, width, eps)``: the
    product's rows are divided by ``sqrt(sum(ss[m]) / width + eps)``;  ``again = (ids, embed, escale)``: ``embed[ids] * escale`` is
    added too."""
    (M, K), N = a.shape, w.shape[0]
    h = torch.empty(M, N, dtype=a.dtype, device=x.device) if then else None
    part = torch.empty(M, N // 256, dtype=torch.float32, device=x.device) if then == THEN_SCALED else None
    ss, width, reps = rms if rms is not None else (None, 1.0, 0.0)
    ids, embed, escale = again if again is not None else (None, None, 0.0)
    rn = ss.shape[1] if ss is not None else 0
    s = stream_ptr(x)
    for lo, hi, f in plan:
        def at(t, row):
            return 0 if t is None else ptr(t) + t.element_size() * lo * row
        rest = (at(x, N), float(scale), at(ss, rn), rn, float(width), float(reps), at(ids, 1), ptr(embed), float(escale), then,
                float(alpha), ptr(nw), ptr(nb), at(h, N), at(part, N // 256), hi - lo, N)
        if f:
            check(lib().k8s_gemm_add(at(a, a.stride(0)), a.stride(0), ptr(w), *rest, K, f, s), "gemm_add")
        else:
            y = proj_planes(a[lo:hi], w)
            check(lib().k8s_add_rows(ptr(y), y.shape[0], *rest, s), "add_rows")
    return h, part


def add_ok(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor) -> bool:
    """Layout :func:`gemm_add` needs of the residual [M, N] (or [M, 1, N]) and the operands."""
    return (_few_ok(a, w) and a.shape[1] == w.shape[1] <= a.stride(0) and x.dtype == torch.float32 and x.is_contiguous()
            and x.data_ptr() % 16 == 0 and x.numel() == a.shape[0] * w.shape[0] and x.device == a.device == w.device)


def silu_scales(M: int, w: torch.Tensor) -> bool:
    """Whether :func:`glu_proj` of ``M`` rows is gemm_big's fused form, which can divide the rows of both products."""
    N, K = w.shape[0] // 2, w.shape[1]
    return (M > DISPATCH_MAX_M and w.dtype == torch.bfloat16 and w.is_contiguous() and w.data_ptr() % 16 == 0 and w.shape[0] == 2 * N
            and K % 256 == 0 and K // 256 <= 16 and swiglu_choice(M, 2 * N, K, False) is None and big_shape_ok(M, N, K, True)
            and big_fused(M, N, K, True))


def gemm_big_silu_scaled(x: torch.Tensor, w: torch.Tensor, part: torch.Tensor, eps: float) -> torch.Tensor:
    """:func:`glu_proj` of the rows ``x`` divided by ``sqrt(sum(part[m]) / K + eps)``."""
    (M, K), N = x.shape, w.shape[0] // 2
    out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    if x.device not in _big_ws and _big_tail:
        reserve_big_ws(x.device)
    check(lib().k8s_gemm_big_silu_scaled(ptr(x), x.stride(0), ptr(w), ptr(out), N, M, N, K, ptr(part), part.shape[1], float(K),
                                         float(eps), stream_ptr(x)), "gemm_big_silu_scaled")
    return out


def proj(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``x @ w.T`` as activations, where neither :func:`batch_plan` nor another rule has it with the 32-column stream form where that is the
    fastest: 17 to 128 rows (below, the skinny kernel) and one wave of strips with the K it was measured at.  us at 17..32 / 64 / 128 rows, hipBLASLt / this:
    8192 x 2048 12.3 / 10.2, 12.8 / 11.1, 15.6 / 13.7;  4736 x 2048 12.3 / 9.7, 12.9 / 10.7, 15.2 / 13.6;  2048 x 2048
    9.2 / 8.3, 10.6 / 8.3, 10.5 / 10.6.  At 273 strips the second wave costs it the lead (8736 x 2048, 64 rows:
    15.3 / 17.2);  a long K over few strips does where the library cuts it (1024 x 2048 at 24 / 128 rows 8.1 / 9.0, 8.4 /
    10.3, 2048 x 2048 11.1 / 9.2, 11.4 / 13.0)."""
    y = _batch(x, w, ROWS_BF16)
    if y is not None:
        return y
    M, K = x.shape
    N = w.shape[0]
    if (16 < M <= NARROW_MAX_M and 32 <= N <= 32 * NARROW_WGS and K <= 2048 and (N, K) not in _dispatch and _few_ok(x, w)
            and rows_plan(M, N, K) is None and (K < 1536 or N > 2048 or M <= 64 and N * K >= 9 << 18)
            and stream_shape_ok(M, N, K, _narrow_cfg(M), 1)):
        return gemm_stream(x, w, _narrow_cfg(M), 1)
    return linear(x, w)


def big_tiles_fill(M: int, N: int, silu: bool, K: int = 4096) -> bool:
    """Whether gemm_big's 256-row tiles fill the 256 compute units far enough over all their waves.  Then its fused epilogue
    beats hipBLASLt and a pass over the result, otherwise the idle last wave costs more than the pass: from four fifths, and
    where the rows themselves (not whole tiles of them, which the library takes smaller) fill half up to a K of 1024, or past
    the first wave seven tenths up to 2048 (within it least is to be had: SwiGLU at 0.75 48.4 / 48.7).  us fused / apart at
    waves of tiles:  squared relu 8192 x 2048 at 0.50 38.6 / 36.8, 0.75 42 / 48, 1.00 49 / 60, 1.12 77 / 72, 1.38 82 / 90, 1.50
    83 / 96, 2.12 123 / 128, 2.38 127 / 141, 5.00 226 / 282, 8192 x 1024 at 0.38 24.0 / 23.6, 0.50 24.9 / 25.3, 1.12 48 / 53;
    SwiGLU 8192 x 2048 at 1.25 96 / 86, 1.50 97 / 99, 2.25 138 / 135, 2.50 137 / 154, 4.25 227 / 239, 6144 x 2048 at 1.31 85 /
    81, 1.50 85 / 89, 8192 x 4096 at 1.50 153 / 148, 2.50 239 / 248;  with rows that end early in a tile, SwiGLU 8192 x 1024 at
    274 rows (0.50 waves, 0.27 of rows) 28 / 22, 16384 x 2048 at 537 (1.50, 1.05) 95 / 89.  Over 256 random sizes between the
    first line and the others 0.84 of the time, none past 1.02."""
    cols = -(-N // (128 if silu else 256))
    tiles = -(-M // 256) * cols
    units = 256 * -(-tiles // 256)
    if 10 * tiles >= 8 * units:
        return True
    return (K <= 1024 or K <= 2048 and tiles > 256) and 10 * M * cols >= (5 if K <= 1024 else 7) * 256 * units


SHORT_K = 512       # up to here what is paid is the result's way through memory, not the tiles


def big_fused(M: int, N: int, K: int, silu: bool) -> bool:
    """Whether a prompt's product takes gemm_big's fused epilogue (N: result columns, of SwiGLU half the weight's rows): a
    short K once the product is large enough to outweigh a wave of tiles that takes 10 to 17 us whatever it holds, a longer
    one where the tiles fill the card.  us apart / fused of the squared relu, M x N in millions: K 128 at 2.5 (256 x 10000)
    11.1 / 10.8, 3.2 (1280 x 2500) 12.4 / 11.3, 0.6 (512 x 1200) 7.5 / 10.4;  K 256 at 2.6 12.7 / 12.7, 3.8 15.0 / 13.3;  K
    512 at 3.2 16.7 / 17.8, 5.1 21.4 / 18.4, 0.3 8.1 / 15.8."""
    if K <= SHORT_K:
        return M * N * (2 if silu else 1) >= (1 << 21) + 4096 * K
    return big_tiles_fill(M, N, silu, K)


def relu_sq_proj(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``max(x @ w.T, 0)^2`` as activations (17 to 64 rows: :func:`batch_plan`).  In one launch for up to 128 rows over one wave of 32-column strips (us apart /
    fused at 8192 x 2048: 1 row 10.5 / 9.8, 16 rows 12.9 / 10.1, 64 rows 15.5 / 11.0, 128 rows 17.9 / 13.9) and for prompts
    (:func:`big_fused`); the fused forms square the fp32 sum.  Not for few rows of up to 4096 columns: the strips are half the
    card, and the skinny kernel and its pass are quicker (2048 x 2048 at 1, 8, 16 rows 6.6 / 9.2, 7.4 / 9.2, 8.0 / 9.2, x 1024
    5.0 / 5.7, 5.7 / 5.9, 6.0 / 5.9, x 512 4.4 / 4.4, 4.9 / 4.7, 5.2 / 4.6)."""
    y = _batch(x, w, ROWS_RELU2)
    if y is not None:
        return y
    M, K = x.shape
    N = w.shape[0]
    if _few_ok(x, w):
        plan = rows_plan(M, N, K, ROWS_RELU2) if M <= ROWS_MAX_M and K == w.shape[1] else None
        if plan is not None:
            return gemm_rows(x, w, plan[0], ROWS_RELU2)
        skinny = N <= 4096 and K > 512 and M <= (8 if K <= 1536 else 16)
        if (0 < M <= NARROW_MAX_M and N <= 32 * NARROW_WGS and K <= 2048 and not skinny
                and stream_shape_ok(M, N, K, _narrow_cfg(M), 1)):
            out = torch.empty((M, N), dtype=x.dtype, device=x.device)
            check(lib().k8s_gemm_stream_act(ptr(x), x.stride(0), ptr(w), ptr(out), N, M, N, K, _narrow_cfg(M), 1,
                                            stream_ptr(x)), "gemm_stream_act")
            return out
        if M > DISPATCH_MAX_M and big_shape_ok(M, N, K) and big_fused(M, N, K, False):
            return gemm_big(x, w, relu2=True)
    return relu_sq(linear(x, w))


def glu_proj(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``silu(x @ Wg.T) * (x @ Wu.T)`` as activations (w = [Wg; Wu]): what a dispatch table says, then one launch by shape, of
    17 to 64 rows as :func:`batch_plan` has it.
    Up to 128 rows (us apart / fused at 1, 16, 64, 128 rows): up to 256 strips of 16 outputs the 32-row strips, except where
    few weight bytes leave the skinny kernel ahead (4096 x 2048 11.4 / 9.9, 13.1 / 10.3, 15.8 / 11.1, 18.2 / 14.1;  2048 x
    2048 7.7 / 9.3, 9.3 / 9.6, 14.8 / 10.4, 17.8 / 13.5;  640 x 384 6.1 / 3.3 .. 9.4 / 4.6); wider weights the 64-row strips
    (6144 x 2048 14.2 / 12.9, 18.5 / 13.4, 19.4 / 14.5, 22.7 / 18.4), from 8192 on the register ring up to 32 rows (8192 x
    2048 17.1 / 16.3, 22.5 / 16.3, then 21.3 / 17.3, 24.6 / 21.7).  Prompts: :func:`big_fused`."""
    a = swiglu_gemm(x, w)
    if a is not None:
        return a
    a = _batch(x, w, ROWS_SILU)
    if a is not None:
        return a
    M, K = x.shape
    I = w.shape[0] // 2
    if _few_ok(x, w):
        plan = rows_plan(M, I, K, ROWS_SILU) if M <= ROWS_MAX_M and w.shape == (2 * I, K) else None
        if plan is not None:
            return gemm_rows(x, w, plan[0], ROWS_SILU)
        if 0 < M <= NARROW_MAX_M:
            if I <= 16 * NARROW_WGS:
                cfg = _narrow_cfg(M) if K <= 2048 and (M > 16 or I > 3072 or K <= 512) else 0
            else:
                cfg = 8 if M <= 32 and I >= 8192 and K % 512 == 0 else 14
            if cfg and stream_shape_ok(M, 2 * I, K, cfg, 1) and I % (16 if cfg > 30 else 32) == 0:
                return gemm_stream_silu(x, w, cfg)
        elif M > DISPATCH_MAX_M and big_shape_ok(M, I, K, True) and big_fused(M, I, K, True):
            return gemm_big(x, w, silu=True)
    if w.shape[0] == 2 * I and _few_f32_ok(x, w):
        out = torch.empty((M, I), dtype=torch.float32, device=x.device)
        check(lib().k8s_few_rows_glu_f32(ptr(x), x.stride(0), ptr(w), ptr(out), M, I, K, stream_ptr(x)), "few_rows_glu_f32")
        return out
    if w.shape[0] == 2 * I:
        a = _split_f32(x, w, glu=True)
        if a is not None:
            return a
    return glu_clamp(linear(x, w), 1.0, math.inf, 0.0)


def reserve_lib_workspace(dev: torch.device, claim_stream: int = None) -> None:
    """Allocate the hipBLASLt workspace (and gemm_big's split-tail workspace)
    before any HIP-graph capture.  ``claim_stream`` (a raw hipStream_t): the
    stream that owns the split tail (the engine's compute stream)."""
    if dev not in _blaslt_ws:
        _blaslt_ws[dev] = torch.empty(BLASLT_WS_BYTES, dtype=torch.uint8, device=dev)
    reserve_big_ws(dev)
    if claim_stream is not None and dev in _big_ws and _big_tail:
        with torch.cuda.device(dev):
            check(lib().k8s_gemm_big_claim_ws(claim_stream), "gemm_big_claim_ws")


def big_tail_foreign(dev: torch.device) -> int:
    """gemm_big launches on ``dev`` that ran without the split tail because
    another stream owns its workspace (reported in the bench line)."""
    if torch.device(dev).type != "cuda":
        return 0
    with torch.cuda.device(dev):
        return int(lib().k8s_gemm_big_tail_foreign())


_big_ws: Dict[torch.device, torch.Tensor] = {}
_big_tail = KNOBS.big_tail


def reserve_big_ws(dev: torch.device, enable: bool = None) -> None:
    """gemm_big's split-tail workspace on ``dev`` (csrc/kernels/gemm_big.hip:
    256 fp32 partial tiles + tickets, zeroed once): without it the kernel runs
    a partial last wave of whole tiles.  ``enable=False`` unregisters it (A/B).

    One workspace per device, so gemm_big launches must not overlap in time on
    that device: two in flight would mix their partial tiles and tickets.  The
    engine issues every projection on its one compute stream (the TP overlap's
    side stream carries only collectives, ``parallel/groups.py``); a second
    stream issuing gemm_big needs its own workspace or an event between them."""
    dev = torch.device(dev)
    if dev.type != "cuda":
        return
    on = _big_tail if enable is None else enable
    with torch.cuda.device(dev):
        if not on:
            check(lib().k8s_gemm_big_set_ws(None), "gemm_big_set_ws")
            return
        t = _big_ws.get(dev)
        if t is None:
            t = _big_ws[dev] = torch.zeros(lib().k8s_gemm_big_ws_bytes(), dtype=torch.uint8, device=dev)
        check(lib().k8s_gemm_big_set_ws(ptr(t)), "gemm_big_set_ws")


# ------------------------------------------------ hipBLASLt solution tables
# (Engine-init tuning of hipBLASLt solutions over an M ladder lost 4 % end to
# end -- profiles/r1_blaslt_tune_8b.txt -- and was retired; the
# bucketed table below, verified per bucket, stays.)


def projection_shapes(mc, tp: int = 1) -> List[Tuple[int, int]]:
    """(N, K) of the dense projections hipBLASLt runs at prefill M (per TP rank)."""
    H, I = mc.hidden, mc.intermediate
    qkv = (mc.n_heads + 2 * mc.n_kv_heads) * mc.head_dim // tp
    out = [(qkv, H), (H, mc.n_heads * mc.head_dim // tp)]
    if not getattr(mc, "n_experts", 0):
        out += [(2 * I // tp, H), (H, I // tp)]
    return out


def lib_algos_path(model: str, tp: int = 1) -> str:
    return os.path.join(DATA_DIR, f"blaslt_algos_{model}" + (f"-tp{tp}" if tp > 1 else "") + ".json")


def load_lib_algos(path: str) -> int:
    """Register the measured hipBLASLt solutions of ``path`` with the native
    front end; returns how many were accepted.  ON by default
    (K8S_BLASLT_ALGOS=0 disables it).

    The file's ``buckets`` (tools/blaslt_tune_buckets.py) hold, per (N, K),
    ``[lo, hi, solution]`` rows: a solution is used for M in [lo, hi] only,
    and was kept only where, registered and re-timed on this call path with
    cold weights, it was no slower than the heuristic's own choice at lo, mid
    and hi and >= 3 % faster over the three -- 14 of 76 buckets, mostly where
    the heuristic's pick misfires just above a tile boundary (down M = 1537:
    328 -> 177 us).  Replayed on 811 recorded prefill-size steps: 11.68 ->
    11.46 s (profiles/r2_blaslt_buckets/).  The older one-point ``algos``
    ladder (tools/blaslt_sweep.py) picked winners of noisy sweeps and applied
    them up to the next ladder point; it measured slower (profiles/r2_blaslt_ab/)
    and is still read for other models' files.  No-op without the native
    library GEMM."""
    if not _native_lib_gemm or not KNOBS.blaslt_algos or not os.path.exists(path):
        return 0
    with open(path) as f:
        d = json.load(f)
    n = 0
    for key, ladder in d.get("algos", {}).items():
        N, K = (int(v) for v in key.split(","))
        for M, idx in sorted(ladder.items(), key=lambda kv: int(kv[0])):
            if lib().k8s_blaslt_set_algo(int(M), N, K, int(idx)) == 0:
                _lib_tuned.setdefault((N, K), []).append((int(M), 1 << 30))
                n += 1
    # bucketed form (tools/blaslt_tune_buckets.py): [lo, hi, solution] per (N, K),
    # each verified on the engine's own call path at the bucket's ends and middle
    for key, rows in d.get("buckets", {}).items():
        N, K = (int(v) for v in key.split(","))
        for lo, hi, idx in rows:
            if lib().k8s_blaslt_set_algo_range(int(lo), int(hi), N, K, int(idx)) == 0:
                _lib_tuned.setdefault((N, K), []).append((int(lo), int(hi)))
                n += 1
    return n


def clear_lib_tuning() -> None:
    lib().k8s_blaslt_clear_tuning()
    _lib_tuned.clear()


# ------------------------------------------------------- measured dispatch
# data/gemm_dispatch_<model>.json (tools/gemm_mid_sweep.py --emit): for each
# (N, K) projection, per M bucket, the fastest of hipBLASLt / skinny / a
# gemm_mid variant measured on MI355X with cold (per-layer) weights.  An M
# between buckets uses the next bucket up (every listed kernel handles any M
# up to its bucket).
DISPATCH_MAX_M = 256
_dispatch: Dict[Tuple[int, int], List[tuple]] = {}


DATA_DIR = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "data")


def dispatch_path(model: str, tp: int = 1) -> str:
    override = KNOBS.gemm_dispatch_file  # A/B of two measured tables
    if override:
        return override
    return os.path.join(DATA_DIR, f"gemm_dispatch_{model}" + (f"-tp{tp}" if tp > 1 else "") + ".json")


def load_dispatch(path: str) -> bool:
    global _dispatch
    if not os.path.exists(path) or not KNOBS.gemm_dispatch:
        return False
    with open(path) as f:
        d = json.load(f)
    tab = {}
    for key, rows in d["shapes"].items():
        fused = key.startswith("silu:")
        n, k = (int(v) for v in key.split(":")[-1].split(","))
        tab[("silu", n, k) if fused else (n, k)] = sorted((int(r["m"]), r["kind"], int(r.get("cfg", -1)), int(r.get("splits", 1))) for r in rows)
    _dispatch = tab
    return True


def clear_dispatch() -> None:
    _dispatch.clear()


def dispatch_table() -> Dict[Tuple[int, int], List[tuple]]:
    return _dispatch


def _lookup(N: int, K: int, M: int, silu: bool = False):
    rows = _dispatch.get(("silu", N, K) if silu else (N, K))
    if not rows:
        return None
    for m, kind, cfg, splits in rows:
        if M <= m:
            return kind, cfg, splits
    return None


def _mid_shape_ok(M: int, N: int, K: int, cfg: int, splits: int) -> bool:
    mt, nt, nw, _, silu = mid_configs()[cfg]
    return not silu and M <= 16 * mt and N % (16 * nt * nw) == 0 and K % (64 * splits) == 0


def _mid_ok(x: torch.Tensor, w: torch.Tensor, cfg: int, splits: int) -> bool:
    mt, nt, nw, _, silu = mid_configs()[cfg]
    M = x.shape[0]
    N, K = w.shape
    return (x.dtype == torch.bfloat16 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and w.is_contiguous()
            and x.shape[1] == (2 * K if silu else K) and M <= 16 * mt and N % (16 * nt * nw) == 0
            and K % (64 * splits) == 0)


_offs_cache = {}


def _grp_ok(x: torch.Tensor, w: torch.Tensor, splits: int) -> bool:
    N, K = w.shape
    return (x.dtype == torch.bfloat16 and x.stride(1) == 1 and w.is_contiguous() and x.shape[1] == K
            and N % 128 == 0 and K % (64 * splits) == 0)


def grp_offsets(dev: torch.device, M: int) -> torch.Tensor:
    """Device [0, M] expert offsets of a single-expert grouped GEMM: a row of
    one table uploaded once per device (a per-M ``torch.tensor`` upload is a
    pageable copy that waits for every queued kernel -- a GPU bubble each
    time a new M shows up mid-run)."""
    tab = _offs_cache.get(dev)
    if tab is None:
        rows = torch.arange(DISPATCH_MAX_M + 1, dtype=torch.int32)
        tab = torch.stack([torch.zeros_like(rows), rows], 1)
        tab = _offs_cache[dev] = tab.to(dev)
    if M <= DISPATCH_MAX_M:
        return tab[M]
    key = (dev, M)
    offs = _offs_cache.get(key)
    if offs is None:
        offs = _offs_cache[key] = torch.tensor([0, M], dtype=torch.int32, device=dev)
    return offs


def gemm_grp(x: torch.Tensor, w: torch.Tensor, splits: int, out: torch.Tensor = None) -> torch.Tensor:
    """``x @ w.T`` on the grouped-GEMM kernel with a single expert (64 x 128
    tiles through swizzled LDS, split-K partials + reduce): the structure that
    streams the MoE down projection at 5.8 TB/s, applied to dense shapes."""
    from . import moe as MO
    M = x.shape[0]
    offs = grp_offsets(x.device, M)
    if out is None:
        out = torch.empty((M, w.shape[0]), dtype=x.dtype, device=x.device)
    return MO.grouped_gemm(x, w.view(1, *w.shape), offs, out=out, splits=splits)


def gemm_stream(x: torch.Tensor, w: torch.Tensor, cfg: int = 8, splits: int = 1,
                out: torch.Tensor = None) -> torch.Tensor:
    """``x @ w.T`` on the W-shared decode kernel (csrc/kernels/gemm_stream.hip):
    a workgroup's 4 waves split the rows of a 64-column strip, W is staged once
    through swizzled LDS, X goes L2 -> registers; ``cfg`` = W register ring
    depth (4 / 8), K split over ``splits`` workgroups (fp32 partials + reduce)."""
    M = x.shape[0]
    N, K = w.shape
    if out is None:
        out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    part = _scratch(x.device, splits * M * N) if splits > 1 else None
    check(lib().k8s_gemm_stream(ptr(x), x.stride(0), ptr(w), ptr(out), out.stride(0), M, N, K, cfg, splits,
                                ptr(part), stream_ptr(x)), "gemm_stream")
    return out


BIG_PIPE = KNOBS.big_var  # schedule variant (gemm_big.hip: 1 = ping-pong)
# Prefill-size dispatch between gemm_big and hipBLASLt: per (N, K) the M ranges
# where the hand-written kernel measured faster, each with its K split count
# (data/gemm_big_<model>.json, tools/big_gemm_ab.py --emit), separately for the
# SwiGLU-fused gate_up form (against hipBLASLt + silu_mul).
# K8SRCA_BIG_GEMM=0 disables it; K8SRCA_BIG_GEMM=all uses gemm_big (no K split)
# for every shape it accepts above DISPATCH_MAX_M (A/B runs).
_big_mode = KNOBS.big_gemm
_big_ranges: Dict[Tuple, List[Tuple[int, int, int]]] = {}


def big_path(model: str, tp: int = 1) -> str:
    return os.path.join(DATA_DIR, f"gemm_big_{model}" + (f"-tp{tp}" if tp > 1 else "") + ".json")


def load_big(path: str) -> int:
    """Register the measured gemm_big M ranges of ``path``; returns how many."""
    _big_ranges.clear()
    if _big_mode == "0" or not os.path.exists(path):
        return 0
    with open(path) as f:
        d = json.load(f)
    n = 0
    for tag in ("ranges", "silu", "rope"):
        for key, rows in d.get(tag, {}).items():
            N, K = (int(v) for v in key.split(","))
            parsed = [(int(r[0]), int(r[1]), int(r[2]) if len(r) > 2 else 1) for r in rows]
            if tag != "ranges" and any(s != 1 for _, _, s in parsed):
                # the SwiGLU / RoPE epilogue forms have no split-K variant
                raise ValueError(f"{path}: {tag} row for {key} carries splits > 1")
            _big_ranges[(tag, N, K) if tag != "ranges" else (N, K)] = parsed
            n += len(rows)
    return n


def rope_choice(M: int, N: int, K: int) -> bool:
    """The qkv projection of M rows on gemm_big with its RoPE + paged KV-write
    epilogue (data file table ``rope``: measured against hipBLASLt +
    k8s_rope_kv)?  ``K8SRCA_BIG_GEMM=all`` takes it wherever the shape fits."""
    if _big_mode == "0" or M <= DISPATCH_MAX_M or not big_shape_ok(M, N, K):
        return False
    if _big_mode == "all":
        return True
    return any(lo <= M <= hi for lo, hi, _ in _big_ranges.get(("rope", N, K), ()))


def gemm_big_rope(x: torch.Tensor, w: torch.Tensor, positions: torch.Tensor, cos_sin: torch.Tensor,
                  slots: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, nq: int, nkv: int,
                  out: torch.Tensor = None, pipe: int = None) -> torch.Tensor:
    """``qkv = x @ w.T`` with q, k rotated and k, v written to their pages in
    the GEMM's epilogue (csrc/kernels/gemm_big.hip MODE 2): bit-identical to
    :func:`gemm_big` + ``ops.attention.rope_kv_write``, one launch and one
    pass over qkv fewer."""
    M, K = x.shape
    N = w.shape[0]
    assert N == (nq + 2 * nkv) * 128 and big_shape_ok(M, N, K) and x.stride(1) == 1 and w.is_contiguous()
    assert positions.dtype == torch.int32 and cos_sin.dtype == torch.float32
    assert slots is None or slots.dtype == torch.int32
    if out is None:
        out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    if M == 0:
        return out
    if x.device not in _big_ws and _big_tail:
        reserve_big_ws(x.device)
    BS = k_cache.shape[2]
    check(lib().k8s_gemm_big_rope(ptr(x), x.stride(0), ptr(w), ptr(out), out.stride(0), M, N, K, ptr(positions),
                                  ptr(cos_sin), ptr(slots), ptr(k_cache), ptr(v_cache), nq, nkv, BS,
                                  BIG_PIPE if pipe is None else pipe, stream_ptr(x)), "gemm_big_rope")
    return out


def big_scratch_elems() -> int:
    """fp32 elements of split-K partials the loaded gemm_big ranges can need
    (the gemm_mid scratch, reserved before any capture)."""
    need = 0
    for key, rows in _big_ranges.items():
        if isinstance(key[0], str):  # ("silu" / "rope", N, K): no split-K form (load_big rejects splits > 1)
            continue
        for lo, hi, splits in rows:
            if splits > 1:
                need = max(need, min(hi, 8192) * key[0] * splits)
    return need


def set_big(mode: str) -> None:
    global _big_mode
    _big_mode = mode


def _big_pick(M: int, N: int, K: int, silu: bool = False) -> int:
    """K splits of gemm_big for this (M, N, K), 0 = not gemm_big.  ``N`` is
    the weight's row count (2I for the SwiGLU form)."""
    if _big_mode == "0" or M <= DISPATCH_MAX_M:
        return 0
    if not big_shape_ok(M, N // 2 if silu else N, K, silu):
        return 0
    if _big_mode == "all":
        return 1
    for lo, hi, splits in _big_ranges.get(("silu", N, K) if silu else (N, K), ()):
        if lo <= M <= hi and big_shape_ok(M, N // 2 if silu else N, K, silu, splits):
            return splits
    return 0


# SwiGLU epilogue on the decode stream kernel: where the dispatch table picks
# gemm_stream with one K split for gate_up, the SwiGLU form of the same strip
# kernel (64-row W strips = 32 gate + 32 up rows) replaces gate_up + silu_mul --
# the same weight bytes, no [M, 2I] write and re-read, one launch fewer.
_stream_silu = KNOBS.stream_silu


def swiglu_choice(M: int, N2: int, K: int, rows: bool = True):
    """(kind, cfg, splits) of the SwiGLU-epilogue gate_up GEMM for ``M`` rows of
    a [N2 = 2I, K] gate_up weight, or ``None`` (gate_up GEMM + silu_mul).
    ``rows``: as in :func:`select_gemm`."""
    if _big_pick(M, N2, K, silu=True):
        return KIND_BIG, BIG_PIPE, 1
    if _stream_silu and _dispatch and M <= DISPATCH_MAX_M and (N2 // 2) % 64 == 0:
        kind, cfg, splits = select_gemm(M, N2, K, rows=rows)
        if kind == KIND_STREAM and splits == 1:
            return KIND_STREAM, cfg, 1
        if kind == KIND_ROWS and splits == 1 and (N2, K) in _dispatch and rows_shape_ok(M, N2 // 2, K, cfg, 1, ROWS_SILU):
            return KIND_ROWS, cfg, 1
    return None


def gemm_stream_silu(x: torch.Tensor, w: torch.Tensor, cfg: int, out: torch.Tensor = None) -> torch.Tensor:
    """``silu(x @ Wg.T) * (x @ Wu.T)`` on the decode stream kernel (w = [Wg; Wu])."""
    M, K = x.shape
    N = w.shape[0] // 2
    if out is None:
        out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    check(lib().k8s_gemm_stream_silu(ptr(x), x.stride(0), ptr(w), ptr(out), out.stride(0), M, N, K, cfg,
                                     stream_ptr(x)), "gemm_stream_silu")
    return out


def swiglu_gemm(y: torch.Tensor, w_gu: torch.Tensor):
    """``silu_mul(y @ w_gu.T)`` in one launch (gemm_big's or the stream kernel's
    SwiGLU epilogue) where :func:`swiglu_choice` picks one; ``None`` otherwise
    (the caller runs the gate_up GEMM + silu_mul)."""
    M, K = y.shape
    if not (y.is_cuda and y.dtype == torch.bfloat16 and y.stride(1) == 1 and y.stride(0) % 8 == 0
            and w_gu.is_contiguous()):
        return None
    ch = swiglu_choice(M, w_gu.shape[0], K, M <= ROWS_MAX_M and rows_ok(y, w_gu))
    if ch is None:
        return None
    if ch[0] == KIND_BIG:
        return gemm_big(y, w_gu, silu=True, pipe=ch[1])
    if ch[0] == KIND_ROWS:
        return gemm_rows(y, w_gu, ch[1], ROWS_SILU)
    return gemm_stream_silu(y, w_gu, ch[1])


def big_shape_ok(M: int, N: int, K: int, silu: bool = False, splits: int = 1) -> bool:
    """What csrc/kernels/gemm_big.hip accepts: 256-column tiles (128 act
    columns for the SwiGLU form), K in pairs of 64-deep tiles per K split
    (split-K only for the plain form)."""
    return (M > 0 and splits >= 1 and K % (128 * splits) == 0 and N % (128 if silu else 256) == 0
            and not (silu and splits > 1))


def gemm_big(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor = None, silu: bool = False,
             pipe: int = None, splits: int = 1, relu2: bool = False) -> torch.Tensor:
    """``x @ w.T`` on the prefill-size MFMA kernel (csrc/kernels/gemm_big.hip:
    256 x 256 x 64 tiles, eight-phase ping-pong schedule, LDS-DMA staging;
    ``pipe`` = the VAR bits (1 = the ping-pong stagger, the default ``BIG_PIPE``;
    +2 static priority, +4 the 32x32x16-MFMA form)).  ``silu=True``: ``w`` is the gate_up weight
    [2I, K] and the result is ``silu(x @ Wg.T) * (x @ Wu.T)`` [M, I] -- the
    SwiGLU epilogue, with the unfused path's bf16 rounding of gate and up.
    ``relu2=True``: ``max(x @ w.T, 0)^2``.
    ``splits`` > 1: K split over that many workgroups per tile (fp32 partials
    in the gemm_mid scratch, then a reduce launch)."""
    assert not (relu2 and (silu or splits > 1))
    M, K = x.shape
    N = w.shape[0] // 2 if silu else w.shape[0]
    if not (x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16 and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and w.is_contiguous() and w.shape[1] == K and big_shape_ok(M, N, K, silu, splits)):
        raise ValueError(f"gemm_big: unsupported operands x {tuple(x.shape)} w {tuple(w.shape)} silu={silu} "
                         f"splits={splits}")
    if out is None:
        out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    if M == 0:
        return out
    var = BIG_PIPE if pipe is None else pipe
    if x.device not in _big_ws and _big_tail:
        reserve_big_ws(x.device)
    if splits > 1:
        part = _scratch(x.device, splits * M * N)
        check(lib().k8s_gemm_big_split(ptr(x), x.stride(0), ptr(w), ptr(out), out.stride(0), M, N, K, var, splits,
                                       ptr(part), stream_ptr(x)), "gemm_big_split")
        return out
    check(lib().k8s_gemm_big(ptr(x), x.stride(0), ptr(w), ptr(out), out.stride(0), M, N, K,
                             3 if relu2 else int(silu), var, stream_ptr(x)), "gemm_big")
    return out


def stream_shape_ok(M: int, N: int, K: int, cfg: int, splits: int) -> bool:
    """What csrc/kernels/gemm_stream.hip's launcher accepts: 64-column strips,
    64-deep chunks, a slice of whole cfg-chunk loop trips, the 8-deep ring only
    up to two 16-row fragments per wave (M <= 128)."""
    # cfg 13..16: the LDS-DMA kernel with 3..6 stages (any chunk count); 23 / 24:
    # the same on 128-column strips with 3 / 4 stages; 34 / 36: on 32-column strips
    # with 4 / 6 stages (M <= 128); 4 / 8: the register ring, whose loop has no partial trip
    ok_cfg = (cfg == 4 or (cfg == 8 and M <= 128) or cfg == 13 or (cfg == 14 and M <= 192)
              or (cfg in (15, 16) and M <= 64) or cfg == 23 or (cfg == 24 and M <= 192)
              or (cfg in (34, 36) and M <= 128))
    bn = 32 if cfg > 30 else 128 if cfg > 20 else 64
    return (ok_cfg and 0 < M <= 256 and N % bn == 0 and splits >= 1 and K % (64 * splits) == 0
            and (cfg > 10 or (K // splits // 64) % cfg == 0))


def stream_candidates(M: int, N: int, K: int):
    """(cfg, splits) of the stream kernel for (M, N, K): 128..2048 workgroups."""
    out = []
    if not (0 < M <= 256 and N % 64 == 0):
        return out
    for cfg in (4, 8, 13, 14, 15, 16, 23, 24):
        for s in (1, 2, 4, 7, 8, 14, 16):
            if not stream_shape_ok(M, N, K, cfg, s):
                continue
            if 128 <= (N // (128 if cfg > 20 else 64)) * s <= 2048:
                out.append((cfg, s))
    return out


def linear_silu(gu: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """``silu_mul(gu) @ w.T`` (the SwiGLU down projection): one SwiGLU-fused
    gemm_mid launch where the dispatch table measured it fastest, else the
    activation kernel followed by :func:`linear`."""
    M = gu.shape[0]
    N, K = w.shape
    if _dispatch and gu.is_cuda and M <= DISPATCH_MAX_M:
        ent = _lookup(N, K, M, silu=True)
        if ent is not None and ent[0] == "mid" and _mid_ok(gu, w, ent[1], ent[2]):
            return gemm_mid(gu, w, ent[1], ent[2])
    from .norm import silu_mul
    return linear(silu_mul(gu), w)

# ------------------------------------------------------------ mid-M GEMM
_mid_cfgs = None
_mid_scratch = {}


def mid_configs():
    """[(mt, nt, nw, u, silu)] of the compiled gemm_mid variants (index = cfg id)."""
    global _mid_cfgs
    if _mid_cfgs is None:
        import ctypes
        L = lib()
        out = []
        buf = (ctypes.c_int * 5)()
        for i in range(L.k8s_gemm_mid_num_cfgs()):
            check(L.k8s_gemm_mid_cfg(i, buf), "gemm_mid_cfg")
            out.append(tuple(buf))
        _mid_cfgs = out
    return _mid_cfgs


# Split-K partial buffers that were replaced by a larger one.  They are never
# freed: a HIP graph captured before the growth still writes (and reads back)
# its partials at the old address on every replay.  Freed, that memory would go
# back to the caching allocator and be handed to some later tensor -- the
# grammar mask table, an activation, a sampling input -- which each replay would
# then overwrite with fp32 partials: silent corruption of every request that
# tensor serves, for the rest of the run.  Growth after the engine's up-front
# reservation is rare (reserve_dispatch_scratch sizes it for the whole table);
# keeping the old buffer costs its bytes once.
_retired_scratch: List[torch.Tensor] = []
scratch_growths = 0


def _scratch(dev: torch.device, n: int) -> torch.Tensor:
    global scratch_growths
    t = _mid_scratch.get(dev)
    if t is None or t.numel() < n:
        if t is not None:
            _retired_scratch.append(t)
            scratch_growths += 1
        t = scratch(max(n, 1 << 20), torch.float32, dev)
        _mid_scratch[dev] = t
    return t


def reserve_mid_scratch(dev: torch.device, max_m: int, max_n: int, max_splits: int = 8) -> None:
    """Allocate the split-K partial buffer up front (before HIP-graph capture)."""
    _scratch(dev, max_m * max_n * max_splits)


def reserve_dispatch_scratch(dev: torch.device) -> None:
    """Size both split-K partial buffers (gemm_mid's and the grouped kernel's)
    for the largest split entry of the loaded dispatch table."""
    from . import moe as MO
    need_mid = need_grp = 0
    for key, rows in _dispatch.items():
        n = key[-2]
        for m, kind, _, splits in rows:
            if kind in ("mid", "stream", "rows") and splits > 1:  # all use the gemm_mid partial buffer
                need_mid = max(need_mid, m * n * splits)
            elif kind == "grp" and splits > 1:
                need_grp = max(need_grp, m * n * splits)
    need_mid = max(need_mid, big_scratch_elems())
    if need_mid:
        _scratch(dev, need_mid)
    if need_grp:
        MO.reserve_split_scratch(dev, need_grp, 1, 1)
    if dev.type == "cuda":
        grp_offsets(dev, 0)  # the offsets table, before any timed step or capture


def gemm_mid(x: torch.Tensor, w: torch.Tensor, cfg: int, splits: int, out: torch.Tensor = None) -> torch.Tensor:
    """``x @ w.T`` on the mid-M kernel (csrc/kernels/gemm_mid.hip), variant
    ``cfg``, K split over ``splits`` workgroups (fp32 partials + reduce).  For
    a SwiGLU variant ``x`` is the gate_up activation [M, 2K] and the product
    is ``silu_mul(x) @ w.T``."""
    M = x.shape[0]
    N, K = w.shape
    if out is None:
        out = torch.empty((M, N), dtype=x.dtype, device=x.device)
    part = _scratch(x.device, splits * M * N) if splits > 1 else None
    check(lib().k8s_gemm_mid(ptr(x), x.stride(0), ptr(w), ptr(out), out.stride(0), M, N, K, cfg, splits,
                             ptr(part), stream_ptr(x)), "gemm_mid")
    return out


def mid_candidates(M: int, N: int, K: int, silu: bool = False):
    """Every (cfg, splits) that applies to (M, N, K): grid of 128..1024 workgroups."""
    out = []
    for i, (mt, nt, nw, u, fused) in enumerate(mid_configs()):
        bn = 16 * nt * nw
        if bool(fused) != silu or M > 16 * mt or M <= 16 * mt // 2 and mt > 2 or N % bn:
            continue
        for s in (1, 2, 4, 7, 8):
            if K % (64 * s) or K // s < 64 * u:
                continue
            if 128 <= (N // bn) * s <= 1024:
                out.append((i, s))
    return out


def candidate_kernels(M: int, N: int, K: int):
    """Hand-written kernels applicable to an (M, N, K) bf16 projection, as
    ``(name, fn(x, w) -> y)`` pairs (used by tools/gemm_mid_sweep.py)."""
    out = []
    if M <= 128 and N % 16 == 0 and K % 256 == 0:
        def skinny(x, w):
            y = torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
            check(lib().k8s_gemm_skinny(ptr(x), x.stride(0), ptr(w), ptr(y), y.stride(0), x.shape[0], w.shape[0],
                                        x.shape[1], stream_ptr(x)), "gemm_skinny")
            return y
        out.append(("skinny", skinny))
    if 16 < M <= 256 and x_ok(K):
        for cfg, s in mid_candidates(M, N, K):
            out.append((f"mid{cfg}:{mid_configs()[cfg][:4]}x{s}", lambda x, w, cfg=cfg, s=s: gemm_mid(x, w, cfg, s)))
    if M <= 256 and N % 128 == 0:
        for s in (1, 2, 4, 8):
            if K % (64 * s) == 0 and (N // 128) * ((M + 63) // 64) * s <= 2048:
                out.append((f"grp:x{s}", lambda x, w, s=s: gemm_grp(x, w, s)))
    for cfg, s in stream_candidates(M, N, K):
        out.append((f"stream{cfg}:x{s}", lambda x, w, cfg=cfg, s=s: gemm_stream(x, w, cfg, s)))
    return out


def silu_candidates(M: int, N: int, K: int):
    """SwiGLU-fused gemm_mid variants for ``silu_mul(gu) @ w.T`` (w [N, K], gu [M, 2K])."""
    out = []
    if 16 < M <= 256 and x_ok(K):
        for cfg, s in mid_candidates(M, N, K, silu=True):
            out.append((f"mid{cfg}:{mid_configs()[cfg][:4]}x{s}", lambda g, w, cfg=cfg, s=s: gemm_mid(g, w, cfg, s)))
    return out


def x_ok(K: int) -> bool:
    return K % 64 == 0
