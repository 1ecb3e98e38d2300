"""A residual's pass without a launch of its own: in a reply chain each costs 3 to 4 us in which the chip waits.

Up to 16 rows (fp32: four) a sublayer's last product takes the pass into its epilogue (:func:`add_product`,
:func:`dyt_product`; csrc/kernels/gemm_step.hip, few_rows_f32.hip): what is behind it then gets the activations, or a
:class:`Scaled`, whose rows the next product divides by their root mean square.  Where that does not pay and there is one row,
the next product makes the pass in every workgroup instead, under the weights' way from memory (:func:`step`,
:func:`dyt_step`, :class:`RowStep`; csrc/kernels/gemm_row_step.hip).  Otherwise it is the launch it was
(:func:`..ops.norm.hyper_step`, :func:`..ops.norm.add_dyt`).  The products below take any of the three, and
:func:`residual` says where the residual is afterwards."""
from typing import Optional

import torch

from . import linear as L
from . import norm as N
from ._lib import check, lib, ptr, stream_ptr, use_hip

MAX_K, COLS, PLANES, SUMS = 2048, 512, 4, 64     # what the kernel takes (kStepMaxK, kStepCols, kStepPlanes, kStepSums)


def plan(n: int, k: int, out_kind: int, planes: bool = False):
    """(16-row fragments a workgroup, K ranges) with which one row's product takes its residual pass in front, or None.
    ``n``: result columns.  Wherever the row-streaming kernel takes one row and a wave can ask for its whole share at once;
    the fragments of the least work on the busiest of 256 compute units, two where that is the same (us of one / two: 8192
    SwiGLU 13.4 / 12.8, 8192 8.0 / 7.4, 32768 23.6 / 23.3, 8736 9.6 / 10.3, 2304 4.4 / 5.4).  K is cut in two only where half
    of the units would stay idle (1088 columns whole / cut 4.0 / 3.7, 2560 4.5 / 5.2)."""
    if (("silu", 2 * n, k) if out_kind == L.ROWS_SILU else (n, k)) in L.dispatch_table():
        return None                              # another kernel was measured for this weight
    if L.rows_plan(1, n, k, out_kind, planes) is None or k > MAX_K or k % COLS:
        return None
    half = out_kind == L.ROWS_SILU
    fits = [nf for nf in (2, 1) if n % ((8 if half else 16) * nf) == 0]
    if not fits:
        return None
    wgs = {nf: n // ((8 if half else 16) * nf) for nf in fits}
    nf = min(fits, key=lambda f: -(-wgs[f] // 256) * f)
    ranges = 2 if planes and wgs[nf] < 128 and k % (2 * COLS) == 0 else 1
    return nf, ranges


class RowStep:
    """``x``: the fp32 residual [1, W], replaced by a new tensor when a product has made the pass; ``h``: its activations,
    once somebody has them."""

    def __init__(self, x: torch.Tensor, act: int, launch, read):
        self.x, self.h, self._act, self._launch, self._read = x, None, act, launch, read

    def read(self) -> torch.Tensor:
        """The activations by the separate pass, the residual updated in place."""
        if self.h is None:
            if self._launch is None:
                raise RuntimeError("the pass was made in front of a product that did not keep its activations")
            self.h = self._read()
        return self.h

    def product(self, w: torch.Tensor, out_kind: int, plain, planes: bool = False, keep: bool = False):
        """``plain(h, w)`` with the pass in front where the kernel takes it.  ``keep``: ``h`` is read again afterwards."""
        n, k = w.shape[0] // (2 if out_kind == L.ROWS_SILU else 1), w.shape[1]
        p = (plan(n, k, out_kind, planes) if self.h is None and self._launch is not None
             and out_kind in (L.ROWS_BF16, L.ROWS_F32, self._act) else None)
        if (p is None or w.dtype != torch.bfloat16 or not w.is_contiguous() or w.data_ptr() % 16 or k != self.x.shape[1]
                or w.device != self.x.device or w.shape[0] % 2 and out_kind == L.ROWS_SILU):
            return plain(self.read(), w)
        out = torch.empty((p[1], 1, n) if planes else (1, n), device=w.device,
                          dtype=torch.float32 if out_kind == L.ROWS_F32 else w.dtype)
        x_out = torch.empty_like(self.x)
        h = torch.empty(1, k, dtype=w.dtype, device=w.device) if keep else None
        self._launch(x_out, h, w, out, n, k, p[0], p[1], out_kind)
        self.x, self.h, self._launch = x_out, h, None
        return out


def rows(h, idx: Optional[torch.Tensor]):
    """The activations of some rows (None: of all)."""
    if idx is None:
        return h
    if isinstance(h, RowStep):
        h = h.read()
    return h.index_select(0, idx) if isinstance(h, torch.Tensor) else h.rows(idx)


def residual(h, x: torch.Tensor) -> torch.Tensor:
    """The residual behind a product of ``h``: ``x`` itself, or where the pass put it."""
    return h.x.view(x.shape) if isinstance(h, RowStep) else x


def _one_row(x: torch.Tensor, y: Optional[torch.Tensor], out_dtype) -> bool:
    W = x.shape[-1]
    return (use_hip(x) and x.numel() == W and COLS <= W <= MAX_K and W % COLS == 0 and y is not None
            and out_dtype == torch.bfloat16 and x.dtype == torch.float32 and x.is_contiguous() and x.data_ptr() % 16 == 0
            and _planes_ok(y, W))


def _planes_ok(y: torch.Tensor, W: int) -> bool:
    return (y.dtype == torch.float32 and y.is_contiguous() and y.data_ptr() % 16 == 0 and y.shape[-2:] == (1, W)
            and y.dim() <= 3 and y.numel() <= PLANES * W)


def _fp32_row(t: torch.Tensor, W: int) -> bool:
    return t.dtype == torch.float32 and t.is_contiguous() and t.numel() == W and t.data_ptr() % 16 == 0


def step(x: torch.Tensor, y: torch.Tensor, one: torch.Tensor, mix: torch.Tensor, nw: torch.Tensor, eps: float, out_dtype,
         again: Optional[tuple] = None, rms: Optional[tuple] = None):
    """:func:`..ops.norm.hyper_step` on one stream that is only added to (``one``, ``mix``: ones; ``x`` [T, 1, W])."""
    if x.shape[0] != 1:                              # (before anything else: prompts pay for one comparison)
        return N.hyper_step(x, y, one, mix, inn=one, nw=nw, eps=eps, out_dtype=out_dtype, again=again, rms=rms)

    def read():
        return N.hyper_step(x, y, one, mix, inn=one, nw=nw, eps=eps, out_dtype=out_dtype, again=again, rms=rms)

    W = x.shape[-1]
    ids, embed, escale = again if again is not None else (None, None, 0.0)
    ss, width, reps = rms if rms is not None else (None, 1.0, 0.0)
    if not (_one_row(x, y, out_dtype) and x.shape[1] == 1 and _fp32_row(nw, W)
            and (ss is None or ss.dtype == torch.float32 and ss.is_contiguous() and ss.shape[0] == 1 and 0 < ss.numel() <= SUMS)
            and (ids is None or ids.dtype == torch.int32 and ids.numel() == 1 and embed.dtype == out_dtype
                 and embed.is_contiguous() and embed.shape[1] == W and embed.data_ptr() % 8 == 0)):
        return read()

    def launch(x_out, h, w, out, n, k, nf, ranges, kind):
        check(lib().k8s_gemm_row_step_rms(ptr(x), ptr(x_out), ptr(y), y.shape[0] if y.dim() == 3 else 1, ptr(ss),
                                          ss.numel() if ss is not None else 0, float(width), float(reps), ptr(ids), ptr(embed),
                                          float(escale), ptr(nw), float(eps), ptr(h), ptr(w), ptr(out), n, k, nf, ranges, kind,
                                          stream_ptr(x)), "gemm_row_step_rms")

    return RowStep(x.view(1, W), L.ROWS_SILU, launch, read)


def dyt_step(x: torch.Tensor, y: Optional[torch.Tensor], sy: float, y2: Optional[torch.Tensor], sy2: float, alpha: float,
             w: Optional[torch.Tensor], b: Optional[torch.Tensor], out_dtype):
    """:func:`..ops.norm.add_dyt`."""
    if x.shape[0] != 1:
        return N.add_dyt(x, y, sy, y2, sy2, alpha, w, b, out_dtype=out_dtype)

    def read():
        return N.add_dyt(x, y, sy, y2, sy2, alpha, w, b, out_dtype=out_dtype)

    W = x.shape[-1]
    if not (w is not None and _one_row(x, y, out_dtype) and (y2 is None or _planes_ok(y2, W)) and _fp32_row(w, W)
            and _fp32_row(b, W)):
        return read()

    def launch(x_out, h, wt, out, n, k, nf, ranges, kind):
        yp, yp2 = (t.shape[0] if t is not None and t.dim() == 3 else 1 for t in (y, y2))
        check(lib().k8s_gemm_row_step_dyt(ptr(x), ptr(x_out), ptr(y), yp, float(sy), ptr(y2), yp2, float(sy2), float(alpha),
                                          ptr(w), ptr(b), ptr(h), ptr(wt), ptr(out), n, k, nf, ranges, kind, stream_ptr(x)),
              "gemm_row_step_dyt")

    return RowStep(x, L.ROWS_RELU2, launch, read)


# ------------------------------------ a sublayer's last product with the residual's pass in its epilogue (gemm_step.hip)
INTO_F32_ROWS = 4
# loads a wave: a pair of kernels each.  Up to 8 every count; past that even ones alone are built, so that K of 9, 11, 13 and 15
# times 512 (4608, 5632, ..) and past 8192 keep planes and the pass, with one row a RowStep.
INTO_ROWS, INTO_LOADS, INTO_STRIP, PARTS = 16, (1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16), 8, 256


def _into_fits(m: int, n: int, k: int, two: bool) -> bool:
    """What csrc/kernels/gemm_step.hip takes (``two``: two products of K ``k``), of weights without a measured kernel."""
    waves = 4 if two else 8
    return (0 < m <= INTO_ROWS and n > 0 and n % INTO_STRIP == 0 and k % (64 * waves) == 0 and k // (64 * waves) in INTO_LOADS
            and (n, k) not in L.dispatch_table())


def into_ok(m: int, n: int, k: int, two: bool = False) -> bool:
    """Whether a product of ``m`` rows takes the residual's pass into its epilogue: sizes at which little of X is read
    (:func:`into_long`: those past them)."""
    return _into_fits(m, n, k, two) and _into_few(m, n, k * 2 if two else k)


def _into_few(m: int, n: int, k: int) -> bool:
    if n < 1536:
        return k <= 2048 or k <= 4096 and m * k <= (32768 if n >= 1024 else 8192)
    return m * k * -(-n // 2048) <= (65536 if n <= 2048 else 49152)


def into_long(m: int, n: int, k: int, two: bool = False) -> bool:
    """The sizes past :func:`into_ok` that take it too: every K up to 4096, and of longer ones as much as its workgroups of 8
    columns, each of which reads all of X, can read meanwhile.  us of planes and the norm's pass / of the fused product, and with
    the tanh pass:  2048 x 2048 at 1, 8, 16 rows 6.5 / 4.0, 7.0 / 4.2, 7.2 / 4.8 and 5.9 / 4.0, 6.3 / 4.2, 6.6 / 4.6;  x 4096 at 16
    8.6 / 6.5 and 8.0 / 6.7;  x 8192 at 1, 8, 9, 16 11.2 / 8.3, 11.2 / 8.3, 11.4 / 9.7, 11.6 / 10.6 and 10.6 / 8.3, 10.5 / 8.2, 10.5 /
    9.5, 11.0 / 10.5.  With the tanh pass:  3072 x 8192 at 9, 12, 16 rows 16.0 / 15.8, 16.6 / 16.8, 17.1 / 17.8;  4096 x 4096 at 16 11.2 /
    10.3, x 8192 at 9, 12 18.0 / 17.4, 17.7 / 18.0;  6144 x 4096 at 16 14.3 / 14.0, x 8192 at 4, 8, 9 24.8 / 19.2, 24.9 / 20.6, 24.9 / 24.8.
    Fewer columns:  1024 x 4096 at 16 6.6 / 6.0, x 8192 at 4, 8, 9 7.5 / 6.5, 7.6 / 7.3, 7.6 / 8.2;  512 x 4096 at 16 5.8 / 5.6, x 8192 at
    2, 4, 8 5.9 / 5.8, 5.9 / 6.1, 6.2 / 6.8."""
    fits = _into_fits(m, n, k, two) and n <= 6144
    k *= 2 if two else 1
    if not fits or _into_few(m, n, k):
        return False
    if k <= 4096:
        return True
    if n < 1536:
        return n >= 1024 and m * k <= 65536
    return m * k * -(-n // 2048) < 196608


class Scaled:
    """Activations whose rows are still to be divided by the root mean square of the residual ``x``: what the products below
    do to their sums.  ``part``: that residual's sums of squares in parts."""

    def __init__(self, x: torch.Tensor, h: torch.Tensor, part: torch.Tensor, nw: torch.Tensor, eps: float):
        self.x, self.h, self.part, self.nw, self.eps = x, h, part, nw, eps

    def read(self) -> torch.Tensor:
        """The activations by the separate pass over the residual."""
        return N.hyper_read(self.x, None, self.nw, self.eps, self.h.dtype) if self.h.shape[0] else self.h

    def rows(self, idx: torch.Tensor) -> "Scaled":
        """Some rows, which may be more than there are (one wanted several times)."""
        return Scaled(*(t.index_select(0, idx) for t in (self.x, self.h, self.part)), self.nw, self.eps)

    def product(self, w: torch.Tensor, out_kind: int, plain, planes: bool = False, keep: bool = False):
        if self.h.shape[0] > INTO_ROWS:              # (chosen rows of fewer have their parts in other sizes)
            if (out_kind == L.ROWS_SILU and w.shape[1] == self.h.shape[1] == 256 * self.part.shape[1]
                    and L.silu_scales(self.h.shape[0], w)):
                return L.gemm_big_silu_scaled(self.h, w, self.part, self.eps)
            return plain(self.read(), w)
        if self.h.dtype == torch.float32:
            return self._product_f32(w, out_kind, plain, planes)
        (m, k), n = self.h.shape, w.shape[0] // (2 if out_kind == L.ROWS_SILU else 1)
        if (out_kind == L.ROWS_RELU2 or keep or k != w.shape[1] or w.shape[0] % 2 and out_kind == L.ROWS_SILU
                or not L.rows_ok(self.h, w) or (("silu", w.shape[0], k) in L.dispatch_table()) or (n, k) in L.dispatch_table()):
            return plain(self.read(), w)
        p = L.rows_plan(m, n, k, out_kind, planes) if m <= INTO_ROWS and self.part.shape[1] % 4 == 0 else None
        if p is None:
            return plain(self.read(), w)
        out = torch.empty((p[1], m, n) if planes else (m, n), device=w.device,
                          dtype=torch.float32 if out_kind == L.ROWS_F32 else w.dtype)
        check(lib().k8s_gemm_rows_scaled(ptr(self.h), k, ptr(w), ptr(out), n, m, n, k, p[0], p[1], out_kind, ptr(self.part),
                                         self.part.shape[1], float(k), float(self.eps), stream_ptr(w)), "gemm_rows_scaled")
        return out

    def _product_f32(self, w: torch.Tensor, out_kind: int, plain, planes: bool):
        glu = out_kind == L.ROWS_SILU
        if (out_kind == L.ROWS_RELU2 or glu and w.shape[0] % 2 or self.h.shape[0] > INTO_F32_ROWS
                or not L._few_f32_ok(self.h, w)):
            return plain(self.read(), w)
        (m, k), n = self.h.shape, w.shape[0] // (2 if glu else 1)
        out = torch.empty((1, m, n) if planes else (m, n), dtype=torch.float32, device=w.device)
        check(lib().k8s_few_rows_f32_scaled(ptr(self.h), k, ptr(w), ptr(out), m, n, k, int(glu), ptr(self.part), float(self.eps),
                                            stream_ptr(w)), "few_rows_f32_scaled")
        return out


def _into_operands(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor, out_dtype) -> bool:
    return (a.is_cuda and out_dtype == torch.bfloat16 and x.dtype == torch.float32 and x.is_contiguous()
            and w.shape == (x.shape[-1], a.shape[1]) and w.device == x.device == a.device and L.rows_ok(a, w)
            and (a.shape[0] == 1 or a.stride(0) >= a.shape[1]))


def _into_f32(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor) -> bool:
    """The same of fp32 operands (csrc/kernels/few_rows_f32.hip).

    Up to four rows, whose sums of squares the product behind reads with a wave each.  us of product, pass and product / of the
    two at 1, 2, 4 and, with two rows a wave, 5, 8 rows:  2048 x 2048, gated 16384 x 2048 28.9 / 27.3, 30.8 / 29.6, 35.1 / 33.9, 37.4 /
    42.9, 48.1 / 46.5;  2048 x 8192, 8192 x 2048 27.7 / 25.3, 28.9 / 25.5, 31.7 / 29.9, 34.4 / 36.0, 36.7 / 36.3;  512 x 2048, 1536 x
    512 9.5 / 7.8, 9.9 / 8.1, 10.8 / 9.1, 11.9 / 10.0, 12.3 / 10.5;  4096 x 4096, 8192 x 4096 37.5 / 35.1, 40.0 / 38.3, 44.9 / 42.2,
    47.7 / 49.4, 52.9 / 53.1."""
    return (a.shape[0] <= INTO_F32_ROWS and L._few_f32_ok(a, w) and x.dtype == torch.float32 and x.is_contiguous()
            and w.shape[0] == x.shape[-1] and w.device == x.device == a.device and w.shape[0] % 16 == 0 and w.shape[0] <= 4096)


def add_product(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor, one: torch.Tensor, mix: torch.Tensor, nw: torch.Tensor,
                eps: float, out_dtype, again: Optional[tuple] = None, rms: Optional[tuple] = None,
                glu: Optional[torch.Tensor] = None):
    """The next sublayer's input behind ``x += a @ w.T`` (:func:`step` of that product): activations, :class:`RowStep` or
    :class:`Scaled`.  ``glu``: the weight of the gated product that is the only one to read it."""
    if a.shape[0] <= INTO_ROWS:                      # (before anything else: prompts pay for one comparison)
        h = _rms_into(x, a, w, nw, eps, out_dtype, again, rms)
        if h is not None:
            return h
    elif a.shape[0] >= L.ADD_MIN_ROWS and out_dtype == torch.bfloat16 == a.dtype:
        then = L.THEN_SCALED if glu is not None and glu.shape[1] == w.shape[0] and L.silu_scales(a.shape[0], glu) else L.THEN_NOTHING
        made = _add(x, a, w, 1.0, then, nw, None, 0.0, rms, again)
        if made is not None:
            return Scaled(x, *made, nw, eps) if then else N.hyper_read(x, None, nw, eps, out_dtype)
    if again is None and rms is None:
        y = L.proj_add(x[:, 0], a, w)
        if y is None:
            return N.hyper_read(x, None, nw, eps, out_dtype)
    else:                                            # (a pass that reads the embedding once more adds the product too)
        y = L.proj_planes(a, w)
    return step(x, y, one, mix, nw, eps, out_dtype, again=again, rms=rms)


def _add(x, a, w, scale, then, nw, nb, alpha, rms=None, again=None):
    """:func:`..ops.linear.gemm_add` where it pays and takes the operands (None: nothing has been done)."""
    M, N = a.shape[0], w.shape[0]
    plan = L.add_plan(M, N, a.shape[1], then)
    if plan is None or not L.add_ok(x, a, w) or x.shape[-1] != N or x.dim() == 3 and x.shape[1] != 1:
        return None
    if then and not (_fp32_row(nw, N) and (nb is None or _fp32_row(nb, N))):
        return None
    if rms is not None and not (rms[0].dtype == torch.float32 and rms[0].is_contiguous() and rms[0].dim() == 2
                                and rms[0].shape[0] == M and 0 < rms[0].shape[1] <= SUMS):
        return None
    if again is not None and not (again[0].dtype == torch.int32 and again[0].is_contiguous() and again[0].numel() == M
                                  and again[1].dtype == torch.bfloat16 and again[1].is_contiguous() and again[1].shape[1] == N
                                  and again[1].data_ptr() % 8 == 0):
        return None
    return L.gemm_add(x, a, w, scale, plan, then, alpha, nw, nb, rms, again)


def add_rest(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor, one: torch.Tensor, mix: torch.Tensor, rms: Optional[tuple] = None):
    """``x += a @ w.T`` [T, 1, W], with nothing that reads it behind (``rms`` as in :func:`..ops.norm.hyper_step`)."""
    if a.shape[0] >= L.ADD_MIN_ROWS and a.dtype == torch.bfloat16 and _add(x, a, w, 1.0, L.THEN_NOTHING, None, None, 0.0, rms) is not None:
        return
    y = L.proj_planes(a, w) if rms is not None else L.proj_add(x[:, 0], a, w)
    if y is not None:
        N.hyper_step(x, y, one, mix, rms=rms)


def _rms_into(x, a, w, nw, eps, out_dtype, again, rms) -> Optional[Scaled]:
    (m, k), W = a.shape, x.shape[-1]
    ids, embed, escale = again if again is not None else (None, None, 0.0)
    ss, width, reps = rms if rms is not None else (None, 1.0, 0.0)
    f32 = out_dtype == torch.float32
    fits = (_into_f32(x, a, w) if f32 else (into_ok(m, W, k) or into_long(m, W, k)) and _into_operands(x, a, w, out_dtype)
            and W % 32 == 0 and W // INTO_STRIP <= PARTS)
    if not (fits and x.shape[:2] == (m, 1) and _fp32_row(nw, W)
            and (ss is None or ss.dtype == torch.float32 and ss.is_contiguous() and ss.shape[0] == m
                 and 0 < ss.numel() <= SUMS * m)
            and (ids is None or ids.dtype == torch.int32 and ids.is_contiguous() and ids.numel() == m
                 and embed.dtype == out_dtype and embed.is_contiguous() and embed.shape[1] == W)):
        return None
    h = torch.empty(m, W, dtype=out_dtype, device=x.device)
    part = torch.empty(m, W // (4 if f32 else INTO_STRIP), dtype=torch.float32, device=x.device)
    launch = lib().k8s_few_rows_f32_add if f32 else lib().k8s_gemm_step_rms
    check(launch(ptr(a), a.stride(0), ptr(w), ptr(x), ptr(ss), ss.numel() // m if ss is not None else 0,
                 float(width), float(reps), ptr(ids), ptr(embed), float(escale), ptr(nw), ptr(h), ptr(part), m, W, k,
                 stream_ptr(x)), "gemm_step_rms")
    return Scaled(x, h, part, nw, eps)


def dyt_product(x: torch.Tensor, a: torch.Tensor, w: torch.Tensor, sy: float, a2: Optional[torch.Tensor],
                w2: Optional[torch.Tensor], sy2: float, alpha: float, nw: Optional[torch.Tensor], nb: Optional[torch.Tensor],
                out_dtype):
    """The next sublayer's input behind ``x += sy a @ w.T (+ sy2 a2 @ w2.T)`` (:func:`dyt_step` of those products)."""
    (m, k), W = a.shape, x.shape[-1]
    two = a2 is not None
    if (m <= INTO_ROWS and nw is not None and (into_ok(m, W, k, two) or into_long(m, W, k, two))
            and _into_operands(x, a, w, out_dtype) and x.shape == (m, W)
            and (a2 is None or a2.shape == a.shape and _into_operands(x, a2, w2, out_dtype))
            and _fp32_row(nw, W) and _fp32_row(nb, W)):
        h = torch.empty(m, W, dtype=out_dtype, device=x.device)
        check(lib().k8s_gemm_step_dyt(ptr(a), a.stride(0), ptr(w), float(sy), ptr(a2), a2.stride(0) if a2 is not None else 0,
                                      ptr(w2), float(sy2), ptr(x), float(alpha), ptr(nw), ptr(nb), ptr(h), m, W, k,
                                      stream_ptr(x)), "gemm_step_dyt")
        return h
    if m >= L.ADD_MIN_ROWS and out_dtype == torch.bfloat16 == a.dtype and x.dim() == 2:
        h = _dyt_add(x, a, w, sy, a2, w2, sy2, alpha, nw, nb)
        if h is not None:
            return h
    y = L.proj_add(x, a, w, sy)
    if a2 is None:
        return dyt_step(x, y, sy, None, 1.0, alpha, nw, nb, out_dtype)
    y2 = L.proj_add(x, a2, w2, sy2)
    add = (y, sy, y2, sy2) if y is not None else (y2, sy2, None, 1.0)
    return dyt_step(x, *add, alpha, nw, nb, out_dtype)


def _dyt_add(x, a, w, sy, a2, w2, sy2, alpha, nw, nb) -> Optional[torch.Tensor]:
    """A prompt's products by :func:`..ops.linear.gemm_add`: the second of two, or the only one, leaves the activations."""
    if nw is None:
        return None
    if a2 is None:
        made = _add(x, a, w, sy, L.THEN_DYT, nw, nb, alpha)
        return made and made[0]
    M, W = x.shape
    if not (L.add_plan(M, W, a2.shape[1], L.THEN_DYT) and L.add_ok(x, a2, w2) and L.add_ok(x, a, w) and _fp32_row(nw, W)
            and _fp32_row(nb, W) and (M >= L.ADD_ROWS or L.add_plan(M, W, a.shape[1], L.THEN_NOTHING))):
        return None
    if _add(x, a, w, sy, L.THEN_NOTHING, None, None, 0.0) is None:
        y = L.proj_add(x, a, w, sy)
        if y is not None:                            # (from ADD_ROWS on it adds itself)
            N.add_dyt(x, y, sy)
    return _add(x, a2, w2, sy2, L.THEN_DYT, nw, nb, alpha)[0]


# ------------------------------------------------------------------------- products of activations, or of what makes them
def proj(h, w: torch.Tensor, keep: bool = False) -> torch.Tensor:
    return L.proj(h, w) if isinstance(h, torch.Tensor) else h.product(w, L.ROWS_BF16, L.proj, keep=keep)


def proj_f32out(h, w: torch.Tensor) -> torch.Tensor:
    return L.proj_f32out(h, w) if isinstance(h, torch.Tensor) else h.product(w, L.ROWS_F32, L.proj_f32out)


def proj_planes(h, w: torch.Tensor) -> torch.Tensor:
    return L.proj_planes(h, w) if isinstance(h, torch.Tensor) else h.product(w, L.ROWS_F32, L.proj_planes, planes=True)


def glu_proj(h, w: torch.Tensor) -> torch.Tensor:
    return L.glu_proj(h, w) if isinstance(h, torch.Tensor) else h.product(w, L.ROWS_SILU, L.glu_proj)


def relu_sq_proj(h, w: torch.Tensor) -> torch.Tensor:
    return L.relu_sq_proj(h, w) if isinstance(h, torch.Tensor) else h.product(w, L.ROWS_RELU2, L.relu_sq_proj)


CONV_TAPS = 4


def conv_proj(h, w: torch.Tensor, conv_w: torch.Tensor, tail: torch.Tensor, seg) -> tuple:
    """``h @ w.T``: its first ``len(conv_w)`` columns behind :func:`..ops.seq_ops.short_conv` with SiLU, the others in fp32.

    Up to 16 single tokens that is one product whose epilogue convolves (csrc/kernels/gemm_rows.hip).  us of three launches /
    one, columns convolved + others x K, 4 taps, at 1, 5, 16 tokens: 2304 + 144 x 2048 10.6 / 5.3, 11.1 / 5.5, 12.4 / 6.2;  2048 +
    64 x 1024 8.3 / 4.0, 9.2 / 4.3, 10.0 / 4.7;  6144 + 256 x 2048 12.8 / 7.3, 13.4 / 7.4, 14.8 / 8.8;  12288 + 512 x 4096 26.2 /
    18.4, 26.8 / 20.1, 33.2 / 25.0."""
    from . import seq_ops as S
    C, taps = conv_w.shape
    if isinstance(h, torch.Tensor) and h.shape[0] <= INTO_ROWS:      # (before anything else: prompts pay for one comparison)
        (m, k), n = h.shape, w.shape[0]
        if (m == seg.n_seg == seg.singles() and 0 < C < n and L.rows_ok(h, w) and w.device == h.device
                and all((c, k) not in L.dispatch_table() for c in (C, n - C, n))
                and 1 <= taps <= CONV_TAPS and conv_w.dtype == torch.float32 == tail.dtype and conv_w.is_contiguous()
                and tail.is_contiguous() and tail.shape[1:] == (taps - 1, C)):
            p = L.rows_plan(m, n, k)
            if p is not None and C % (16 * p[0]) == 0:
                out = torch.empty(m, C, dtype=h.dtype, device=h.device)
                rest = torch.empty(m, n - C, dtype=torch.float32, device=h.device)
                check(lib().k8s_gemm_rows_conv(ptr(h), h.stride(0), ptr(w), ptr(out), C, ptr(rest), m, n, k, p[0], ptr(conv_w),
                                               taps, ptr(tail), ptr(seg.seg_pos0), ptr(seg.seg_slot), 1, stream_ptr(h)),
                      "gemm_rows_conv")
                return out, rest
    x = proj(h, w[:C], keep=True)
    return S.short_conv(x, conv_w, None, tail, seg, act=True), proj_f32out(h, w[C:])
