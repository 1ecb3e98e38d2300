"""Ops of layers that carry per-sequence state besides the paged cache:
sinusoidal positions, the short causal convolution in front of a sublayer, the
minGRU recurrence, the post-sublayer norm of an fp32 residual, attention over a
paged latent cache (``csrc/kernels/seq_ops.hip``, ``latent_attn.hip``), window
attention and recurrent mixers (``mixer_ops.hip``, ``window_attn.hip``), masked
softmax attention behind a q / k preparation pass and matrix-state recurrences
(``masked_attn.hip``, ``matrix_mem.hip``), linear attention on the matrix cores
(``linear_attn.hip``).

A step's rows come in SEGMENTS (:class:`SegMeta`): consecutive rows of one
sequence -- a decode token or a portion of a prompt.  Device tensors run the HIP
kernels; CPU tensors the fp32 PyTorch forms below (the engine's CPU backend).
The residual stream, norms, recurrence and softmax are fp32 in both; ``dt`` is
the activation / weight type (bf16 or fp32).
"""
from __future__ import annotations

import math
from dataclasses import dataclass, field
from typing import Dict, List, Optional, Tuple

import numpy as np

import torch

from ._lib import check, lib, ptr, scratch, stream_ptr, unwatched, use_hip

# Parts a single token's keys are cut into, a workgroup each (csrc/kernels/token_attn.hip).  us at parts of half the size /
# this / twice: masked, 1 row at 200 keys 8.9 / 6.5 / 6.5, at 4000 9.1 / 10.5 / 14.4, 64 rows at 400 14.7 / 12.3 / 10.4, at
# 1500 34.6 / 27.5 / 28.0;  latent, 1 row at 200 9.3 / 11.5 / 11.5, at 4000 15.7 / 14.1 / 15.8, 64 at 400 17.5 / 14.3 / 17.6.
MASK_TOKEN_BLOCKS = 8    # 32-key blocks of the row's own list
LATENT_PART = 128        # keys, from the part of the row's first visible key on
TOKEN_PARTS = 64         # a row with more than so many of them has larger ones
TOKEN_SCRATCH = 1 << 28  # floats of partial results (1 GiB): a step of more takes its rows in groups
MASK_TILE_ROWS = 128     # (token, head) rows of one workgroup of the masked prompt kernel
# A step's prompt rows are taken one by one as well (masked layers) while the keys and values they read stay within so many
# bytes, and they and their parts within two rounds of workgroups: the rows have their keys cut into parts, and a tile's way
# from keys to results is longer, but it reads them once for 128 (row, head) pairs (so two rows may read four times as much).
# us, tiles / rows:  16 heads over 2 of 128, 16 / 64 / 128 rows at 0 keys 11 / 7, 11 / 8, 12 / 8, at 500 20 / 13, 20 / 17,
# 22 / 26, at 2000 18 / 14, 21 / 36, 24 / 63, 2 rows at 30000 26 / 21;  16 over 16, 8 / 32 / 64 rows at 0 keys 10 / 8, 9 / 9,
# 9 / 16, at 500 18 / 13, 17 / 38, 18 / 70, at 8000 25 / 111, 24 / 387, 28 / 760;  4 over 4 of 64, 8 / 32 rows at 2000 16 / 11,
# 14 / 22;  8 over 1 of 64, 64 / 128 / 256 / 300 rows at 0 9 / 8, 10 / 7, 12 / 8, 13 / 16.
MASK_ROW_BYTES = 32 << 20
MASK_ROW_GROUPS = 512


@dataclass
class SegMeta:
    n_seg: int
    row_seg: torch.Tensor      # [T] int32: segment of every row
    seg_row0: torch.Tensor     # [n_seg + 1] int32 row offsets
    seg_pos0: torch.Tensor     # [n_seg] int32 position of the segment's first token
    seg_slot: torch.Tensor     # [n_seg] int32 state slot of the segment's sequence
    block_tables: torch.Tensor  # [n_seg, maxb] int32 cache pages
    row0_host: List[int]
    pos0_host: List[int]
    slot_host: List[int]
    # rows [0, n_single) take the decode kernels (single tokens, short portions); the rest are prompt portions
    n_single: int = 0
    _items: Dict[int, tuple] = field(default_factory=dict)

    def attn_items(self, tokens_per_item: int) -> tuple:
        """Work items of the MFMA attention kernels, made once per step and item size:
        (decode items [n, 4] int32 on the device, prompt items, most keys a decode row sees).
        An item is (segment, first row, tokens, position of the first row's token); a segment's prompt
        items are padded with empty ones to a multiple of four."""
        got = self._items.get(tokens_per_item)
        if got is not None:
            return got
        dec, pre, kmax = [], [], 0
        for s in range(self.n_seg):
            a, b, p0 = self.row0_host[s], self.row0_host[s + 1], self.pos0_host[s]
            if a < self.n_single:
                dec += [(s, r, 1, p0 + r - a) for r in range(a, b)]
                kmax = max(kmax, p0 + b - a)
            else:
                pre += [(s, r, min(tokens_per_item, b - r), p0 + r - a) for r in range(a, b, tokens_per_item)]
                pre += [(s, a, 0, p0)] * (-len(pre) % 4)   # a workgroup's four waves share one segment's keys
        host = torch.from_numpy(np.asarray(dec + pre, dtype=np.int32).reshape(-1, 4))
        dev = self.row_seg.device
        if dev.type == "cuda":
            host = host.pin_memory()
        both = host.to(dev, non_blocking=True)
        got = (both[:len(dec)], both[len(dec):], kmax)
        self._items[tokens_per_item] = got
        return got


    def tile_items(self, tokens_per_item: int) -> torch.Tensor:
        """Every segment cut into tiles of at most ``tokens_per_item`` consecutive tokens ([n, 4] int32 on
        the device: segment, first row, tokens, position of the first token), made once per step."""
        key = ("tiles", tokens_per_item)
        got = self._items.get(key)
        if got is None:
            it = [(s, r, min(tokens_per_item, self.row0_host[s + 1] - r), self.pos0_host[s] + r - self.row0_host[s])
                  for s in range(self.n_seg) for r in range(self.row0_host[s], self.row0_host[s + 1], tokens_per_item)]
            host = torch.from_numpy(np.asarray(it, dtype=np.int32).reshape(-1, 4))
            if self.row_seg.device.type == "cuda":
                host = host.pin_memory()
            got = self._items[key] = host.to(self.row_seg.device, non_blocking=True)
        return got

    def _once(self, key: tuple, make):
        got = self._items.get(key)
        if got is None:
            got = self._items[key] = make()
        return got

    def singles(self) -> int:
        """How many segments of one token stand in front."""
        r = self.row0_host
        for i in range(self.n_seg):
            if r[i + 1] - r[i] != 1:
                return i
        return self.n_seg

    def most_keys(self, first: int, end: int) -> int:
        """Most keys that a row of the segments from ``first`` to ``end`` sees."""
        r, most = self.row0_host, 0
        for i in range(first, end):
            most = max(most, self.pos0_host[i] + r[i + 1] - r[i])
        return most

    def keys_behind(self, first: int, most: int) -> int:
        """Keys that the rows of the segments from ``first`` on see, each row its own, ``most`` of them at most."""
        r, total = self.row0_host, 0
        for i in range(first, self.n_seg):
            n, p = r[i + 1] - r[i], self.pos0_host[i]
            low = max(0, min(n, most - p))          # rows that see all of theirs: p + 1, p + 2 ..
            total += low * p + low * (low + 1) // 2 + (n - low) * most
        return total

    def mask_items(self, tokens_per_item: int, by_rows: bool = False) -> tuple:
        """Work items of the masked attention, made once per step: (items of one token, tiles of at most
        ``tokens_per_item``).  The leading segments of one token are single items, and with ``by_rows`` all rows are."""
        key = ("mask", tokens_per_item, by_rows)
        got = self._items.get(key)
        if got is None:
            n1 = self.n_seg if by_rows else self.singles()
            it, n = [], 0
            for s in range(self.n_seg):
                a, b, p0 = self.row0_host[s], self.row0_host[s + 1], self.pos0_host[s]
                step = 1 if s < n1 else tokens_per_item
                it += [(s, r, min(step, b - r), p0 + r - a) for r in range(a, b, step)]
                if s < n1:
                    n = len(it)
            host = torch.from_numpy(np.asarray(it, dtype=np.int32).reshape(-1, 4))
            if self.row_seg.device.type == "cuda":
                host = host.pin_memory()
            both = host.to(self.row_seg.device, non_blocking=True)
            got = self._items[key] = (both[:n], both[n:])
        return got

    def chunk_ranges(self, rows: int, min_rows: int) -> Optional[tuple]:
        """Segments cut into chunks of at most ``rows`` rows, for recurrences that run the chunks in
        parallel: (chunks [n, 4] int32: segment, first row, rows, 0; seg_chunk0 [n_seg + 1] int32), both on
        the device; None when no segment has more than ``min_rows`` rows (the sequential kernel runs)."""
        key = ("ranges", rows, min_rows)
        if key in self._items:
            return self._items[key]
        out = None
        if max(b - a for a, b in zip(self.row0_host[:-1], self.row0_host[1:])) > min_rows:
            ch, c0 = [], [0]
            for s in range(self.n_seg):
                a, b = self.row0_host[s], self.row0_host[s + 1]
                ch += [(s, r, min(rows, b - r), 0) for r in range(a, b, rows)]
                c0.append(len(ch))
            host = torch.from_numpy(np.asarray([v for c in ch for v in c] + c0, dtype=np.int32))
            if self.row_seg.device.type == "cuda":
                host = host.pin_memory()
            dev = host.to(self.row_seg.device, non_blocking=True)
            out = (dev[:4 * len(ch)].view(-1, 4), dev[4 * len(ch):])
        self._items[key] = out
        return out

    def scan_chunks(self, rows: int) -> Optional[torch.Tensor]:
        """Chunks of at most ``rows`` rows for the time-parallel recurrence ([n, 4] int32 on the device:
        segment, first row, rows, index of the segment's first chunk); None when no segment is longer
        than two chunks (the sequential kernel runs)."""
        key = -rows
        if key in self._items:
            return self._items[key]
        out = None
        if max(b - a for a, b in zip(self.row0_host[:-1], self.row0_host[1:])) > 2 * rows:
            ch = []
            for s in range(self.n_seg):
                a, b, first = self.row0_host[s], self.row0_host[s + 1], len(ch)
                ch += [(s, r, min(rows, b - r), first) for r in range(a, b, rows)]
            host = torch.from_numpy(np.asarray(ch, dtype=np.int32))
            if self.row_seg.device.type == "cuda":
                host = host.pin_memory()
            out = host.to(self.row_seg.device, non_blocking=True)
        self._items[key] = out
        return out


SCAN_CHUNK = 64     # rows per chunk of the time-parallel minGRU
SSM_CHUNK = 64      # rows per chunk of the time-parallel selective scan and retention
SEQ_FILL_LANES = 1 << 18   # sequential lanes (segments x channels) from which the chunk-parallel form stops paying


def _dt(t: torch.dtype) -> int:
    if t == torch.bfloat16:
        return 0
    if t == torch.float32:
        return 1
    raise TypeError(f"activations must be bfloat16 or float32, not {t}")


def embed_sinpos(ids: torch.Tensor, pos: torch.Tensor, embed: torch.Tensor, base: float = 10000.0) -> torch.Tensor:
    """fp32 ``embed[ids] + sinusoid(pos)``: entry 2i = sin(p base^(-2i/W)), entry 2i+1 its cosine."""
    T, W = ids.shape[0], embed.shape[1]
    if use_hip(embed):
        x = torch.empty(T, W, dtype=torch.float32, device=embed.device)
        check(lib().k8s_embed_sinpos(ptr(ids), ptr(pos), ptr(embed), ptr(x), T, W, float(base), _dt(embed.dtype),
                                     stream_ptr(embed)), "embed_sinpos")
        return x
    i2 = (torch.arange(W, dtype=torch.float64) // 2) * 2
    ang = pos.double()[:, None] * torch.exp(-i2 / W * torch.log(torch.tensor(float(base), dtype=torch.float64)))[None]
    pe = torch.where((torch.arange(W) % 2 == 1)[None], ang.cos(), ang.sin()).float()
    return embed[ids.long()].float() + pe


def canon_conv(x: torch.Tensor, w: torch.Tensor, tail: torch.Tensor, seg: SegMeta, out_dtype) -> torch.Tensor:
    """``h = x + conv(x)``: per channel ``conv(x)_t = sum_j w[:, j] x_(t - taps + 1 + j)`` over each sequence
    (zeros before its start).  ``tail`` [slots, taps - 1, W] fp32 holds every sequence's last inputs and is
    advanced by this step's rows."""
    T, W = x.shape
    taps = w.shape[1]
    h = torch.empty(T, W, dtype=out_dtype, device=x.device)
    if use_hip(x):
        assert x.dtype == torch.float32 and x.is_contiguous() and w.is_contiguous() and tail.is_contiguous()
        assert tail.shape[1:] == (taps - 1, W) and w.dtype == out_dtype and taps <= 16
        check(lib().k8s_canon_conv(ptr(x), ptr(w), ptr(tail), ptr(seg.row_seg), ptr(seg.seg_row0), ptr(seg.seg_pos0),
                                   ptr(seg.seg_slot), ptr(h), T, seg.n_seg, W, taps, _dt(out_dtype), stream_ptr(x)),
              "canon_conv")
        return h
    wf = w.float()
    nt = taps - 1
    for s in range(seg.n_seg):
        a, b, p0, sl = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s], seg.slot_host[s]
        prev = tail[sl] if p0 > 0 else torch.zeros(nt, W)
        ext = torch.cat([prev, x[a:b]])                     # inputs pos0 - nt .. pos0 + n - 1
        acc = x[a:b].clone()
        for j in range(taps):
            acc += wf[:, j] * ext[j:j + (b - a)]
        h[a:b] = acc.to(out_dtype)
        if nt:
            tail[sl] = ext[-nt:]
    return h


def mingru_scan(zug: torch.Tensor, bz: torch.Tensor, bu: torch.Tensor, state: torch.Tensor, seg: SegMeta,
                out_dtype) -> torch.Tensor:
    """minGRU over every segment: ``zug`` [T, 3C] fp32 = (z | u | g) projections without biases;
    ``S <- (1 - z) S + z cand`` with ``z = sigmoid(.)``, ``cand = u + 1/2`` for ``u >= 0`` else ``sigmoid(u)``;
    returns ``S * silu(g)``.  ``state`` [slots, C] fp32 is read (past position 0) and advanced."""
    T, C3 = zug.shape
    C = C3 // 3
    y = torch.empty(T, C, dtype=out_dtype, device=zug.device)
    if use_hip(zug):
        assert zug.dtype == torch.float32 and zug.is_contiguous() and state.is_contiguous() and bz.dtype == out_dtype
        chunks = seg.scan_chunks(SCAN_CHUNK)
        if chunks is not None:   # long prompt portions: parallel over time as well as channels
            ab = scratch(chunks.shape[0] * 2 * C, torch.float32, zug.device)
            s0 = scratch(seg.n_seg * C, torch.float32, zug.device)
            check(lib().k8s_mingru_chunked(ptr(zug), ptr(bz), ptr(bu), ptr(state), ptr(chunks), chunks.shape[0],
                                           ptr(seg.seg_row0), ptr(seg.seg_pos0), ptr(seg.seg_slot), ptr(ab), ptr(s0),
                                           ptr(y), C, _dt(out_dtype), stream_ptr(zug)), "mingru_chunked")
            return y
        check(lib().k8s_mingru_scan(ptr(zug), ptr(bz), ptr(bu), ptr(state), ptr(seg.seg_row0), ptr(seg.seg_pos0),
                                    ptr(seg.seg_slot), ptr(y), seg.n_seg, C, _dt(out_dtype), stream_ptr(zug)),
              "mingru_scan")
        return y
    z = torch.sigmoid(zug[:, :C] + bz.float())
    u = zug[:, C:2 * C] + bu.float()
    g = zug[:, 2 * C:]
    cand = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
    for s in range(seg.n_seg):
        a, b, p0, sl = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s], seg.slot_host[s]
        S = state[sl].clone() if p0 > 0 else torch.zeros(C)
        for r in range(a, b):
            S = (1 - z[r]) * S + z[r] * cand[r]
            y[r] = (S * torch.nn.functional.silu(g[r])).to(out_dtype)
        state[sl] = S
    return y


def postnorm_(x: torch.Tensor, y: Optional[torch.Tensor], w: torch.Tensor, alpha: float, eps: float) -> torch.Tensor:
    """In place on the fp32 residual: ``x <- unit_rms(alpha x + y) * (1 + w)`` (``y`` None: no sublayer output)."""
    T, W = x.shape
    if use_hip(x):
        assert x.dtype == torch.float32 and x.is_contiguous()
        assert y is None or (y.is_contiguous() and y.shape == x.shape)
        check(lib().k8s_postnorm(ptr(x), ptr(y), 1 if y is None else _dt(y.dtype), ptr(w), _dt(w.dtype), None, T, W,
                                 float(alpha), float(eps), stream_ptr(x)), "postnorm")
        return x
    v = alpha * x + (y.float() if y is not None else 0.0)
    x.copy_(v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + eps) * (1.0 + w.float()))
    return x


def unit_norm_out(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    """``unit_rms(x) * (1 + w)`` of fp32 rows as activations of ``w``'s type (``x`` is left as it is)."""
    T, W = x.shape
    out = torch.empty(T, W, dtype=w.dtype, device=x.device)
    if use_hip(x):
        assert x.dtype == torch.float32 and x.is_contiguous()
        check(lib().k8s_postnorm(ptr(x), None, 1, ptr(w), _dt(w.dtype), ptr(out), T, W, 1.0, float(eps),
                                 stream_ptr(x)), "unit_norm_out")
        return out
    out.copy_((x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * (1.0 + w.float())).to(w.dtype))
    return out


def latent_norm(dn: torch.Tensor, wq: torch.Tensor, wkv: Optional[torch.Tensor], slots: torch.Tensor,
                cache: Optional[torch.Tensor], q_rank: int, kv_rank: int, eps: float, out_dtype,
                cache_t: Optional[torch.Tensor] = None, tail: int = 0, tail_cs: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Rows of the joint down projection ``dn`` [T, >= q_rank + kv_rank] fp32: the query latent is
    RMS-normed (plain weight) and returned; the key-value latent (``wkv`` given) is RMS-normed and
    written to the paged latent ``cache`` [pages, BS, kv_rank] at ``slots`` (page * BS + offset), and
    to its transposed twin ``cache_t`` [pages, kv_rank, BS] when given (the MFMA kernels' PV operand).
    ``tail`` > 0: as many further columns of ``dn`` are a key part shared by all heads; its neighbouring entries
    2i, 2i + 1 are turned by ``tail_cs`` [T, tail] (a :func:`rope_table`) and stand behind the latent in the cache
    rows [pages, BS, kv_rank + pad], filled up with zeros.  ``dn`` [S, T, ..]: the sum of its planes
    (:func:`.linear.proj_planes`)."""
    planes, pstep = 1, 0
    if dn.dim() == 3:
        if dn.shape[0] == 1:
            dn = dn[0]
        elif use_hip(dn) and not (dn.stride(0) % 4 or dn.stride(1) % 4 or dn.data_ptr() % 16
                                  or (q_rank + (kv_rank if wkv is not None else 0) + tail) % 4):
            planes, pstep, dn = dn.shape[0], dn.stride(0), dn[0]      # added where the rows are read
        else:
            dn = dn.sum(0)
    T = dn.shape[0]
    cq = torch.empty(T, q_rank, dtype=out_dtype, device=dn.device)
    kr = kv_rank if wkv is not None else 0
    pad = cache.shape[-1] - kv_rank if kr else 0
    if use_hip(dn):
        assert dn.dtype == torch.float32 and dn.stride(1) == 1 and wq.dtype == out_dtype
        assert dn.shape[1] >= q_rank + kr + tail and wq.numel() == q_rank
        assert cache is None or (cache.is_contiguous() and cache.dtype == out_dtype and cache.shape[-1] >= kv_rank + tail)
        ct = cache_t if kr else None
        assert ct is None or (ct.is_contiguous() and ct.dtype == out_dtype and ct.shape[1] == kv_rank)
        assert not tail or (kr and tail_cs.dtype == torch.float32 and tail_cs.is_contiguous() and tail_cs.shape == (T, tail))
        check(lib().k8s_latent_norm(ptr(dn), dn.stride(0), ptr(wq), ptr(wkv), ptr(slots), ptr(cq), ptr(cache),
                                    ptr(ct), cache.shape[1] if kr else 1, T, q_rank, kr, float(eps),
                                    _dt(out_dtype), stream_ptr(dn), tail, pad, ptr(tail_cs), planes, pstep), "latent_norm")
        return cq
    q = dn[:, :q_rank]
    cq.copy_((q * torch.rsqrt(q.pow(2).mean(-1, keepdim=True) + eps) * wq.float()).to(out_dtype))
    if kr:
        c = dn[:, q_rank:q_rank + kr]
        c = c * torch.rsqrt(c.pow(2).mean(-1, keepdim=True) + eps) * wkv.float()
        row = torch.cat([c, torch.zeros(T, pad)], 1)
        if tail:
            row[:, kr:kr + tail] = _turn_pairs(dn[:, q_rank + kr:q_rank + kr + tail], tail_cs)
        ok = slots >= 0
        cache.view(-1, kr + pad)[slots[ok].long()] = row[ok].to(cache.dtype)
        if cache_t is not None:
            BS = cache.shape[1]
            sl = slots[ok].long()
            cache_t[sl // BS, :, sl % BS] = c[ok].to(cache_t.dtype)
    return cq


def _turn_pairs(x: torch.Tensor, cs: torch.Tensor) -> torch.Tensor:
    """Neighbouring entries of the last dimension turned by the angles of ``cs`` (cos | sin, broadcast over the rest)."""
    half = cs.shape[-1] // 2
    co, si = cs[..., :half], cs[..., half:]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * co - b * si, b * co + a * si], -1).flatten(-2)


LATENT_STEP_RANKS, LATENT_STEP_ROWS, LATENT_STEP_READ = (256, 512, 768, 1024, 1536, 2048), 16, 56 << 20


def latent_up(dn: torch.Tensor, wq: torch.Tensor, wkv: Optional[torch.Tensor], w: torch.Tensor, slots: torch.Tensor,
              cache: Optional[torch.Tensor], q_rank: int, kv_rank: int, eps: float, out_dtype, cache_t: Optional[torch.Tensor] = None,
              tail: int = 0, tail_cs: Optional[torch.Tensor] = None) -> torch.Tensor:
    """:func:`latent_norm`, then its result ``@ w.T``.

    Up to 16 rows in one launch (csrc/kernels/latent_step.hip), every strip of 16 columns of which reads all rows: the line
    is what all strips read.  us of two launches / one at 1, 7, 16 rows, two planes:  768 + 256 + 64 numbers, 3072 columns
    7.5 / 3.6, 7.9 / 4.1, 8.1 / 4.8;  1536 + 512 + 64, 3072 8.1 / 4.9, 8.5 / 5.7, 9.2 / 6.7;  1024 + 256 + 64, 8192 8.7 / 6.1,
    8.6 / 7.5, 9.0 / 9.0;  2048 + 512 + 64, 6144 at 1, 4, 7 10.8 / 9.7, 11.3 / 10.5, 11.4 / 11.9;  1536 + 512 + 64, 24576 17.8 /
    20.9, 18.7 / 25.7, 20.3 / 31.1."""
    from .linear import dispatch_table, proj
    T, N = dn.shape[-2], w.shape[0]
    # (the rows before anything else: prompts pay for one comparison)
    if 0 < T <= LATENT_STEP_ROWS and use_hip(dn) and wkv is not None and cache is not None:
        planes, pstep = (dn.shape[0], dn.stride(0)) if dn.dim() == 3 else (1, 0)
        pad = cache.shape[-1] - kv_rank
        small = ((wq, q_rank, out_dtype), (wkv, kv_rank, out_dtype), (tail_cs if tail else None, T * tail, torch.float32))
        if (out_dtype == torch.bfloat16 == w.dtype and q_rank in LATENT_STEP_RANKS and planes in (1, 2, 4)
                and N // 16 * q_rank * (32 + 4 * T * planes) <= LATENT_STEP_READ
                and q_rank * planes <= 4096 and N > 0 and N % 16 == 0 and kv_rank + tail <= 2048 and (kv_rank + tail) % 4 == 0
                and tail % 2 == 0 and pad >= tail and pad % 2 == 0 and dn.dtype == torch.float32 and dn.stride(-1) == 1
                and dn.shape[-1] >= q_rank + kv_rank + tail and dn.stride(-2) % 4 == 0 and pstep % 4 == 0
                and dn.stride(-2) >= q_rank + kv_rank + tail and dn.data_ptr() % 16 == 0 == w.data_ptr() % 16
                and w.shape[1] == q_rank and w.is_contiguous() and w.device == dn.device and (N, q_rank) not in dispatch_table()
                and all(t is None or t.dtype == d and t.is_contiguous() and t.numel() == n for t, n, d in small)
                and wq.data_ptr() % 8 == 0 and slots.dtype == torch.int32 and slots.is_contiguous() and slots.numel() >= T
                and (not tail or tail_cs is not None)
                and all(t is None or t.is_contiguous() and t.dtype == out_dtype for t in (cache, cache_t))
                and (cache_t is None or cache_t.shape[1:] == (kv_rank, cache.shape[1]))):
            q = torch.empty(T, N, dtype=out_dtype, device=dn.device)
            check(lib().k8s_latent_step(ptr(dn), dn.stride(-2), planes, pstep, ptr(wq), ptr(wkv), ptr(w), ptr(q), ptr(slots),
                                        ptr(cache), ptr(cache_t), cache.shape[1], T, N, q_rank, kv_rank, float(eps), tail, pad,
                                        ptr(tail_cs) if tail else 0, stream_ptr(dn)), "latent_step")
            return q
    cq = latent_norm(dn, wq, wkv, slots, cache, q_rank, kv_rank, eps, out_dtype, cache_t=cache_t, tail=tail, tail_cs=tail_cs)
    return proj(cq, w)


def rotated_tail(q: torch.Tensor, cs: torch.Tensor, H: int, N: int, pad: int) -> torch.Tensor:
    """The entries behind the first ``N`` of every head of ``q`` [T, H (N + R)], neighbours 2i, 2i + 1 turned by ``cs``
    [T, R] (a :func:`rope_table`), filled up with zeros to ``pad``: [T, H, pad]."""
    T, R = cs.shape
    assert q.shape == (T, H * (N + R)) and pad >= R and pad % 2 == 0
    out = torch.empty(T, H, pad, dtype=q.dtype, device=q.device)
    if use_hip(q):
        assert q.is_contiguous() and cs.dtype == torch.float32 and cs.is_contiguous()
        check(lib().k8s_rotated_tail(ptr(q), ptr(cs), ptr(out), T, H, N, R, pad, _dt(q.dtype), stream_ptr(q)),
              "rotated_tail")
        return out
    out[:, :, :R] = _turn_pairs(q.view(T, H, N + R)[:, :, N:].float(), cs[:, None]).to(q.dtype)
    out[:, :, R:] = 0
    return out


# Rows up to which small products run on the vector pipes (csrc/kernels/small_proj.hip), within :func:`_few_heads` and
# :func:`_few_ranks`.
SMALL_PROJ_ROWS = 128


def _few_heads(T: int, H: int, K: int, N: int, fp32: bool) -> bool:
    """Whether ``T`` rows of ``H`` products K -> N are quicker on the vector pipes than the library's batched product: while
    the multiply-adds hide behind one trip to memory, and while a thread's share of K (an eighth, in turn) is short.  us,
    library / this, bf16 (fp32):  16 heads 128 -> 256 at 1, 16, 64, 128 rows 5.3 / 3.0, 5.2 / 4.5, 6.2 / 5.1, 7.4 / 6.7
    (6.5 / 3.2, 6.5 / 5.0, 11.7 / 5.6, 19.7 / 7.9), 256 -> 128 7.1 / 3.6, 6.2 / 5.2, 6.4 / 5.6, 7.4 / 6.9 (9.4 / 4.2, 8.4 /
    5.5, 11.3 / 6.7, 18.6 / 8.9);  64 heads 128 -> 128 at 16, 32, 64 rows 5.0 / 4.6, 4.9 / 5.1, 5.5 / 6.7;  128 heads 64 ->
    256 at 8, 16 4.8 / 4.2, 4.8 / 5.3;  512 -> 128 at 1, 8, 16 of 4 heads 9.5 / 5.3, 9.6 / 7.8, 7.0 / 7.9 (12.1 / 6.4, 12.4 /
    8.8, 10.8 / 8.8);  128 -> 512 of 4 at 4, 8 3.6 / 3.3, 3.6 / 4.2;  512 -> 512 of 16 at 1, 16 6.7 / 7.1, 6.8 / 10.3;  256 ->
    64 of 4 at 2, 8 4.4 / 4.3, 4.4 / 4.7;  640 and 1024 entries: never."""
    m = T * H * K * N
    if N > 256:
        return T <= 4 and K <= 128 and m <= 1 << 24
    if K > 256:
        return N <= 128 and K <= 512 and (m <= 1 << 26 if fp32 else T <= 8)
    if 2 * N < K and not fp32:
        return T <= 2
    most = (1 << 26 if fp32 else 1 << 25) if K >= 128 else 1 << 24
    if T >= 4 * H and (K < 128 or K * N >= 1 << 15):     # (the library takes the longer the more rows a head has)
        most *= 2
    return m <= most


def _few_ranks(T: int, K0: int, N0: int, K1: int, N1: int) -> bool:
    """The same for two products of low rank.  us, two roundings and two products / this:  64 -> 2048 at 1, 16, 128 rows
    11.9 / 2.3, 11.5 / 3.4, 11.8 / 5.3, 64 -> 8192 at 128 16.8 / 14.9;  256 -> 8192 at 32, 64 18.5 / 15.2, 19.5 / 24.6;  512
    -> 2048 at 4, 8, 16, 64 10.4 / 8.3, 10.7 / 13.0, 11.4 / 13.0, 20.2 / 15.3;  1024 -> 2048 at 2, 64 11.7 / 14.4, 29.5 / 27.6."""
    K = max(K0, K1)
    return T * (K0 * N0 + K1 * N1) <= 1 << 27 and (K <= 256 or K <= 512 and not 4 < T < 64)


def _small_rows(x: torch.Tensor, w: torch.Tensor) -> bool:
    return use_hip(x) and 0 < x.shape[0] <= SMALL_PROJ_ROWS and w.dtype == torch.bfloat16 and w.is_contiguous()


def _small_heads(x: torch.Tensor, w: torch.Tensor, H: int, K: int, *out) -> bool:
    """Whether the products of ``H`` heads with ``w`` [H, K, N] may be launched by address and are quicker so: all else is for
    the library's batched product, which refuses what does not fit."""
    T, (HW, KW, N), dt = x.shape[0], w.shape, x.dtype
    return (use_hip(x) and 0 < T <= SMALL_PROJ_ROWS and dt == w.dtype and (dt == torch.bfloat16 or dt == torch.float32)
            and HW == H > 0 and KW == K > 0 and N > 0 and w.device == x.device and K % 8 == 0 and N % 64 == 0
            and _few_heads(T, H, K, N, dt == torch.float32) and unwatched(x, w, *out)
            and w.is_contiguous() and w.data_ptr() % 8 == 0)


def head_proj(x: torch.Tensor, w: torch.Tensor, out: torch.Tensor) -> torch.Tensor:
    """``out[t, h] = x[t, h] @ w[h]`` of ``x`` [T, H, K] and ``w`` [H, K, N] (the strides of ``x`` and ``out`` [T, H, N]
    but the last are free): a kernel of one launch for few rows, the library's batched product otherwise."""
    T, H, K = x.shape
    N = w.shape[2]
    if (_small_heads(x, w, H, K, out) and x.dtype == out.dtype and out.shape == (T, H, N) and out.device == x.device
            and x.stride(2) == 1 == out.stride(2)):
        check(lib().k8s_head_proj(ptr(x), x.stride(0), x.stride(1), ptr(w), ptr(out), out.stride(0), out.stride(1), T, H, K,
                                  N, None, None, 0, 0, _dt(x.dtype), stream_ptr(x)), "head_proj")
    else:
        torch.bmm(x.transpose(0, 1), w, out=out.transpose(0, 1))
    return out


def latent_queries(q: torch.Tensor, uk: torch.Tensor, cs: Optional[torch.Tensor], H: int, D: int, pad: int) -> tuple:
    """A latent layer's queries from its heads ``q`` [T, H (D + R)]: (their first D entries in latent space by ``uk``
    [H, D, KR], [T, H, KR] and head-major in memory; the R entries behind rotated by ``cs`` as :func:`rotated_tail` has
    them, None without ``cs``)."""
    T, KR = q.shape[0], uk.shape[2]
    x = q.view(T, H, -1)
    R = x.shape[2] - D
    if _small_heads(q, uk, H, D) and R >= 0 and q.is_contiguous():
        qa = torch.empty(H, T, KR, dtype=q.dtype, device=q.device).transpose(0, 1)
        qr = None
        if R:
            assert cs.dtype == torch.float32 and cs.is_contiguous() and cs.shape == (T, R) and pad >= R and pad % 2 == 0
            qr = torch.empty(T, H, pad, dtype=q.dtype, device=q.device)
        check(lib().k8s_head_proj(ptr(q), x.stride(0), x.stride(1), ptr(uk), ptr(qa), qa.stride(0), qa.stride(1), T, H, D,
                                  KR, ptr(cs), ptr(qr), R, pad if R else 0, _dt(q.dtype), stream_ptr(q)), "head_proj")
        return qa, qr
    qr = rotated_tail(q, cs, H, D, pad) if R else None
    return torch.bmm(x[:, :, :D].transpose(0, 1), uk).transpose(0, 1), qr


def low_rank_pair(x: torch.Tensor, c0: int, w0: torch.Tensor, c1: int, w1: torch.Tensor, dtype) -> tuple:
    """``x[:, c:c + K] @ w.T`` in fp32 for two column ranges of fp32 rows, rounded to the activations' ``dtype`` first."""
    from .linear import proj_f32out
    T, (N0, K0), (N1, K1) = x.shape[0], w0.shape, w1.shape
    if (_small_rows(x, w0) and _small_rows(x, w1) and dtype == torch.bfloat16 and x.dtype == torch.float32
            and x.stride(1) == 1 and all(k % 32 == 0 and k > 0 for k in (K0, K1)) and _few_ranks(T, K0, N0, K1, N1)
            and w0.data_ptr() % 16 == 0 == w1.data_ptr() % 16):
        a, b = (torch.empty(T, n, dtype=torch.float32, device=x.device) for n in (N0, N1))
        check(lib().k8s_low_rank_pair(ptr(x), x.stride(0), T, c0, K0, ptr(w0), N0, ptr(a), c1, K1, ptr(w1), N1, ptr(b),
                                      stream_ptr(x)), "low_rank_pair")
        return a, b
    return tuple(proj_f32out(x[:, c:c + w.shape[1]].to(dtype).contiguous(), w) for c, w in ((c0, w0), (c1, w1)))


ROWS_PART = 128     # visible keys per part of the vector-pipe attention
ROWS_HEADS = 8      # heads of one key head per workgroup of it
ROWS_FILL = 512     # workgroups from which it walks a row's parts itself
ROWS_SCRATCH = 1 << 28      # floats of partial results past which it does so as well (1 GiB)


def _rows_parts(seg: SegMeta, T: int, heads: int, per_key: int, V: int, dev, chunk: int = 0, window: int = 0,
                keep_first: int = 0, tiles: bool = False) -> tuple:
    """(parts, scratch for their outputs, for their maxima and sums) of a step of the vector-pipe attention whose rows do
    not fill the chip: a workgroup per part of a row's keys, the same sums either way.  (0, None, None): a workgroup per
    row and group of heads.  One workgroup -> parts, us, fp32, 16 heads over 2 of 128: 2 rows at 340 keys 55 -> 27, 16 at
    1024 visible ones 148 -> 28, 128 at 300 68 -> 52, 256 at 400 113 -> 118 (the line; past it the parts save a tenth at
    most and write heads x parts results per row).  ``per_key``: heads that share a key.

    ``tiles``: the one workgroup uses matrix instructions (whole tiles in fp32), so that with two parts at most half of that
    fills the chip: the same at 128 rows of 150, 200 of 200, 250 of 250 keys 21 / 26, 22 / 26, 25 / 31, latent 256 + 64 numbers 34 /
    38, 33 / 42, 35 / 52;  three parts, 128 rows of 300 32 / 31, 53 / 47;  fewer rows, 64 of 300 31 / 26, 50 / 38."""
    groups = heads // per_key * -(-per_key // ROWS_HEADS) * -(-V // 256)
    if T * groups >= ROWS_FILL:
        return 0, None, None
    most = max((p + b - a for p, a, b in zip(seg.pos0_host, seg.row0_host[:-1], seg.row0_host[1:])), default=0)
    if chunk > 0:
        most = min(most, chunk)
    if window > 0:
        most = min(most, window + keep_first)
    parts = -(-most // ROWS_PART)
    if (parts <= 1 or T * heads * parts * (V + 2) > ROWS_SCRATCH
            or tiles and parts <= 2 and T * groups >= ROWS_FILL // 2):
        return 0, None, None
    return (parts, scratch(T * heads * parts * V, torch.float32, dev), scratch(T * heads * parts * 2, torch.float32, dev))


def mfma_tiles(R: int, dtype, device, tail: int = 0) -> int:
    """Query tiles per wave the MFMA attention kernels run prompt portions with for latent rank ``R`` and cache rows of
    ``R + tail`` numbers (0: they do not take these sizes or this type -- the vector-pipe kernel runs instead)."""
    if dtype != torch.bfloat16 or torch.device(device).type != "cuda":
        return 0
    return int(lib().k8s_latent_attn_mfma_ok(int(R), int(tail)))


def _latent_out(qa: torch.Tensor, dtype, head_major: bool) -> torch.Tensor:
    """[T, H, R], in memory [H][T][R] with ``head_major`` (a batched product over the heads reads it as it is)."""
    T, H, R = qa.shape
    if head_major:
        return torch.empty(H, T, R, dtype=dtype, device=qa.device).transpose(0, 1)
    return torch.empty(T, H, R, dtype=dtype, device=qa.device)


def _token_groups(rows: torch.Tensor, heads: int, parts: int, V: int) -> tuple:
    """Items of single tokens [n, 4] in groups whose partial results fit ``TOKEN_SCRATCH``, and scratch for the largest of
    them: outputs, maxima and sums (None, None: one part, nothing to join)."""
    if parts == 1:
        return [rows], None, None
    per = min(rows.shape[0], max(1, TOKEN_SCRATCH // (heads * parts * (V + 2))))
    return ([rows] if per == rows.shape[0] else rows.split(per), *(scratch(per * heads * parts * n, torch.float32, rows.device) for n in (V, 2)))


def _merge_up(qa: torch.Tensor, up: torch.Tensor, n_parts: int) -> bool:
    """Whether the parts of single tokens are merged by the product behind them (csrc/kernels/token_attn.hip,
    token_merge_proj_kernel): where that product is the vector pipes' and a thread can hold all of its entries' parts (2 to 4 us less
    at 1 to 64 rows and 2 to 16 parts, with both timed there)."""
    T, H, R = qa.shape
    return 2 <= n_parts <= 16 and R in (128, 256) and up.shape[2] % 64 == 0 and _small_heads(qa, up, H, R)


def latent_attention_mfma(qa: torch.Tensor, cache: torch.Tensor, cache_t: torch.Tensor, gate: Optional[torch.Tensor],
                          seg: SegMeta, positions: torch.Tensor, scale: float, qr: Optional[torch.Tensor] = None,
                          window: int = 0, sink: Optional[torch.Tensor] = None, head_major: bool = False,
                          up: Optional[torch.Tensor] = None) -> torch.Tensor:
    """:func:`latent_attention` on the matrix cores: bf16 absorbed queries ``qa`` [T, H, R], the latent
    pages and their transposed twins.  ``up`` [H, R, N]: the result is :func:`head_proj`'s of it, [T, H, N].  Decode rows (the step's first ``seg.n_single``) are split over
    partitions of keys and merged; prompt portions run one wave per group of tokens."""
    T, H, R = qa.shape
    BS, W = cache.shape[1], cache.shape[2]
    tiles = mfma_tiles(R, qa.dtype, qa.device, W - R)
    assert tiles and qa.stride(2) == 1 and cache.is_contiguous() and cache_t.is_contiguous() and BS % 32 == 0
    assert gate is None or (gate.dtype == torch.float32 and gate.stride(1) == 1 and gate.shape[1] >= H)
    assert cache_t.shape[1:] == (R, BS) and seg.block_tables.is_contiguous() and window >= 0
    assert (qr is None) == (W == R) and (qr is None or (qr.dtype == qa.dtype and qr.is_contiguous()
                                                        and qr.shape == (T, H, W - R)))
    assert sink is None or (sink.dtype == torch.float32 and sink.numel() == H)
    tpi = tiles * (16 // min(H, 16))
    dec, pre, kmax = seg.attn_items(tpi)
    L, st = lib(), stream_ptr(qa)
    bt, maxb = seg.block_tables, seg.block_tables.shape[1]
    gs = gate.stride(0) if gate is not None else 0
    part, n_parts, groups, po, pml = LATENT_PART, 1, [], None, None
    if dec.shape[0]:
        n_parts = -(-kmax // part)
        if window > 0:      # a row's parts start at the one its first visible key lies in
            n_parts = min(n_parts, (min(int(window), kmax) + part - 2) // part + 1)
        n_parts = min(n_parts, TOKEN_PARTS)
        groups, po, pml = _token_groups(dec, H, n_parts, R)
    fused = up is not None and dec.shape[0] == T and len(groups) == 1 and _merge_up(qa, up, n_parts)
    out = None if fused else _latent_out(qa, torch.bfloat16, head_major)
    for it in groups:
        check(L.k8s_latent_attn_token(ptr(qa), qa.stride(0), qa.stride(1), ptr(qr), W - R, ptr(cache), ptr(cache_t),
                                      ptr(bt), maxb, ptr(it), it.shape[0], ptr(gate), gs, ptr(sink), ptr(out),
                                      *((0, 0) if fused else out.stride()[:2]), ptr(po), ptr(pml), n_parts, part, TOKEN_PARTS, H,
                                      R, BS, int(window), float(scale), st), "latent_attn_token")
    if fused:
        out = torch.empty(T, H, up.shape[2], dtype=torch.bfloat16, device=qa.device)
        check(L.k8s_latent_merge_proj(ptr(po), ptr(pml), n_parts, ptr(dec), T, ptr(gate), gs, ptr(sink), ptr(up), ptr(out),
                                      out.stride(0), out.stride(1), H, R, up.shape[2], st), "latent_merge_proj")
        return out
    if pre.shape[0]:
        check(L.k8s_latent_attn_mfma(ptr(qa), ptr(cache), ptr(cache_t), ptr(bt), maxb, ptr(pre), pre.shape[0], ptr(gate),
                                     gs, ptr(out), H, R, BS, float(scale), st, qa.stride(0), qa.stride(1), ptr(qr), W - R,
                                     out.stride(0), out.stride(1), int(window), ptr(sink)), "latent_attn_mfma")
    return out if up is None else head_proj(out, up, torch.empty(T, H, up.shape[2], dtype=out.dtype, device=out.device))


def latent_attention(qa: torch.Tensor, cache: torch.Tensor, gate: Optional[torch.Tensor], seg: SegMeta, scale: float,
                     out_dtype, qr: Optional[torch.Tensor] = None, window: int = 0, sink: Optional[torch.Tensor] = None,
                     head_major: bool = False) -> torch.Tensor:
    """Causal attention of absorbed queries ``qa`` [T, H, R] fp32 over the paged latents ``cache``
    [pages, BS, R]: ``p = softmax(scale * qa . c_j)`` over the keys up to the row's own position,
    output ``sigmoid(gate[t, h]) * sum_j p_j c_j`` [T, H, R] (``gate`` fp32, row stride free; None: no gate).
    ``qr`` [T, H, P] fp32: the cache rows are [R + P], a key part shared by the heads behind the latent, and
    ``qr . k_j`` is added to the product.  ``window`` > 0: position i sees j with ``i - j < window``.  ``sink`` [H]
    fp32: ``exp(sink_h)`` is added to head h's denominator.  ``head_major``: the result lies [H][T][R] in memory."""
    T, H, R = qa.shape
    BS, W = cache.shape[1], cache.shape[2]
    assert (qr is None) == (W == R)
    out = _latent_out(qa, out_dtype, head_major)
    if use_hip(qa):
        assert qa.dtype == torch.float32 and qa.stride(2) == 1 and cache.is_contiguous() and cache.dtype == out_dtype
        assert gate is None or (gate.dtype == torch.float32 and gate.stride(1) == 1 and gate.shape[1] >= H)
        assert qr is None or (qr.dtype == torch.float32 and qr.is_contiguous() and qr.shape == (T, H, W - R))
        assert sink is None or (sink.dtype == torch.float32 and sink.numel() == H)
        assert seg.block_tables.is_contiguous()
        parts, po, pml = _rows_parts(seg, T, H, H, R, qa.device, window=int(window),
                                     tiles=cache.dtype == torch.float32 and cache.shape[-1] % 16 == 0 == R % 64)
        check(lib().k8s_latent_attn_rows(ptr(qa), ptr(cache), ptr(seg.block_tables), seg.block_tables.shape[1],
                                         ptr(seg.row_seg), ptr(seg.seg_row0), ptr(seg.seg_pos0), ptr(gate),
                                         gate.stride(0) if gate is not None else 0, ptr(out), 0, T, H, R, BS,
                                         float(scale), _dt(out_dtype), stream_ptr(qa), qa.stride(0), qa.stride(1),
                                         ptr(qr), W - R, out.stride(0), out.stride(1), int(window), ptr(sink), parts,
                                         ptr(po), ptr(pml)), "latent_attn_rows")
        return out
    flat = cache.view(-1, W)
    for s in range(seg.n_seg):
        a, b, p0 = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s]
        n_ctx = p0 + b - a
        pages = seg.block_tables[s].long()
        kp = torch.arange(n_ctx)
        c = flat[pages[kp // BS] * BS + kp % BS].float()                      # [ctx, R (+ P)]
        sc = torch.einsum("thr,jr->thj", qa[a:b].float(), c[:, :R])
        if qr is not None:
            sc = sc + torch.einsum("thr,jr->thj", qr[a:b].float(), c[:, R:])
        dist = (p0 + torch.arange(b - a))[:, None] - kp[None, :]
        vis = dist >= 0
        if window > 0:
            vis &= dist < window
        sc = (sc * scale).masked_fill(~vis[:, None, :], float("-inf"))
        if sink is not None:                                                   # one more score without a value
            p = torch.softmax(torch.cat([sc, sink.view(1, H, 1).expand(b - a, H, 1)], -1), -1)[..., :-1]
        else:
            p = torch.softmax(sc, -1)
        o = torch.einsum("thj,jr->thr", p, c[:, :R])
        out[a:b] = (o if gate is None else o * torch.sigmoid(gate[a:b, :H])[:, :, None]).to(out_dtype)
    return out


# ------------------------------------------------------------------ recurrent mixers and window attention
# (csrc/kernels/mixer_ops.hip, window_attn.hip).  Small parameters (convolution taps, biases, decays,
# A, D, the distance bias and the head-mixing matrix) are fp32 tensors.
@dataclass
class SegStepInputs:
    """One step in the segment layout (:class:`SegMeta`)."""
    input_ids: torch.Tensor        # [T] int32
    positions: torch.Tensor        # [T] int32
    slots: torch.Tensor            # [T] int32 cache slot (page * BS + offset) of every row
    seg: SegMeta
    logits_idx: Optional[torch.Tensor]   # [n] int64 rows whose logits are needed (None, captured steps: every row, in order)


def wanted_rows(inp: SegStepInputs) -> Optional[torch.Tensor]:
    """``logits_idx``, or None where that is every row: with one row the head may take another product than behind a row that
    was picked (ops/row_step.py), and a step's bits are the same captured (None) and not."""
    idx = inp.logits_idx
    return None if idx is not None and inp.input_ids.shape[0] == 1 == idx.numel() else idx


def short_conv(x: torch.Tensor, w: torch.Tensor, b: Optional[torch.Tensor], tail: torch.Tensor, seg: SegMeta,
               act: bool = True) -> torch.Tensor:
    """Causal per-channel convolution with bias and SiLU: ``out_t = act(b + sum_j w[:, j] x_(t - taps + 1 + j))``
    over each sequence (the last column of ``w`` [C, taps] is the current token's; zeros before the
    start).  ``x`` [T, C] may be a column slice of a wider matrix.  ``tail`` [slots, taps - 1, C] fp32
    holds every sequence's last inputs and is advanced by this step's rows."""
    T, C = x.shape
    taps = w.shape[1]
    out = torch.empty(T, C, dtype=x.dtype, device=x.device)
    if use_hip(x):
        assert x.stride(1) == 1 and w.dtype == torch.float32 and w.is_contiguous() and tail.is_contiguous()
        assert tail.shape[1:] == (taps - 1, C) and 1 <= taps <= 16 and (b is None or b.dtype == torch.float32)
        d = _dt(x.dtype)
        items = seg.tile_items(WINDOW_TILE)      # rows in tiles of one segment: metadata once per tile
        lens = [b - a for a, b in zip(seg.row0_host[:-1], seg.row0_host[1:])]
        one = items.shape[0] == seg.n_seg and min(lens, default=0) > 0      # a tile per segment
        check(lib().k8s_short_conv(ptr(x), x.stride(0), d, ptr(w), ptr(b), ptr(tail), ptr(seg.row_seg),
                                   ptr(seg.seg_row0), ptr(seg.seg_pos0), ptr(seg.seg_slot), ptr(out), T, seg.n_seg, C,
                                   taps, int(act), d, stream_ptr(x), ptr(items), items.shape[0], int(one)), "short_conv")
        return out
    nt = taps - 1
    xf = x.float()
    for s in range(seg.n_seg):
        a, e, p0, sl = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s], seg.slot_host[s]
        prev = tail[sl] if p0 > 0 else torch.zeros(nt, C)
        ext = torch.cat([prev, xf[a:e]])
        acc = torch.zeros(e - a, C) if b is None else b.expand(e - a, C).clone()
        for j in range(taps):
            acc += w[:, j] * ext[j:j + (e - a)]
        out[a:e] = (torch.nn.functional.silu(acc) if act else acc).to(x.dtype)
        if nt:
            tail[sl] = ext[-nt:]
    return out


def selective_scan(xc: torch.Tensor, dtp: torch.Tensor, dt_bias: torch.Tensor, dbc: torch.Tensor, R: int,
                   A: torch.Tensor, D: torch.Tensor, z: torch.Tensor, state: torch.Tensor, seg: SegMeta) -> torch.Tensor:
    """Diagonal selective state-space recurrence per channel c and state n, fp32:
    ``dt = softplus(dtp + dt_bias)``; ``S[c, n] <- exp(dt_c A[c, n]) S[c, n] + dt_c x_c B_n``;
    ``y_c = (sum_n S[c, n] C_n + D_c x_c) * silu(z_c)``.  ``dbc`` [T, >= R + 2N] fp32 holds B at column R
    and C at column R + N; ``dtp`` [T, C] fp32; ``xc`` [T, C] and ``z`` (a column slice) activations.
    ``state`` [slots, C, N] fp32 is read (past position 0) and advanced."""
    T, C = xc.shape
    N = A.shape[1]
    y = torch.empty(T, C, dtype=xc.dtype, device=xc.device)
    if use_hip(xc):
        assert xc.is_contiguous() and dtp.dtype == torch.float32 and dtp.is_contiguous() and dtp.shape == (T, C)
        assert dbc.dtype == torch.float32 and dbc.stride(1) == 1 and dbc.shape[1] >= R + 2 * N
        assert z.stride(1) == 1 and z.dtype == xc.dtype and state.is_contiguous() and state.shape[1:] == (C, N)
        assert A.dtype == D.dtype == dt_bias.dtype == torch.float32 and A.is_contiguous()
        # long portions: chunks run in parallel (a pass from zero states, a carry over the chunks, the
        # chunks again from their start states); short ones token by token
        # (with many sequences the token-by-token kernel already fills the chip, at half the exponentials)
        cr = seg.chunk_ranges(SSM_CHUNK, 2 * SSM_CHUNK) if seg.n_seg * C < SEQ_FILL_LANES else None
        chunks, c0, cs, csd, nch = None, None, None, None, 0
        if cr is not None:
            chunks, c0 = cr
            nch = chunks.shape[0]
            cs = scratch(nch * C * N, torch.float32, xc.device)
            csd = scratch(nch * C, torch.float32, xc.device)
        check(lib().k8s_selective_scan(ptr(xc), _dt(xc.dtype), ptr(dtp), ptr(dt_bias), ptr(dbc), dbc.stride(0), R,
                                       ptr(A), ptr(D), ptr(z), z.stride(0), ptr(state), ptr(seg.seg_row0),
                                       ptr(seg.seg_pos0), ptr(seg.seg_slot), ptr(y), seg.n_seg, C, N, T,
                                       stream_ptr(xc), ptr(chunks), nch, ptr(c0), ptr(cs), ptr(csd)), "selective_scan")
        return y
    dt = torch.nn.functional.softplus(dtp + dt_bias)
    xf, zf = xc.float(), z.float()
    Bm, Cm = dbc[:, R:R + N], dbc[:, R + N:R + 2 * N]
    for s in range(seg.n_seg):
        a, e, p0, sl = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s], seg.slot_host[s]
        S = state[sl].clone() if p0 > 0 else torch.zeros(C, N)
        for r in range(a, e):
            S = torch.exp(dt[r][:, None] * A) * S + (dt[r] * xf[r])[:, None] * Bm[r][None, :]
            y[r] = ((S @ Cm[r] + D * xf[r]) * torch.nn.functional.silu(zf[r])).to(xc.dtype)
        state[sl] = S
    return y


def ssd_scan(x: torch.Tensor, bc: torch.Tensor, dtp: torch.Tensor, dt_bias: torch.Tensor, rate: torch.Tensor,
             D: torch.Tensor, z: torch.Tensor, H: int, P: int, G: int, N: int, state: torch.Tensor, seg: SegMeta,
             fast_exp: bool = False) -> torch.Tensor:
    """State-space recurrence with one decay per head and token (state-space duality), fp32.  Head h of ``H`` owns
    the channels ``h P .. h P + P - 1`` of ``x`` [T, H P] and reads B / C group ``h // (H // G)`` of ``bc`` [T, 2 G N]
    = (B [G, N] | C [G, N]):  ``dt = softplus(dtp[:, h] + dt_bias[h])``;  ``S <- exp(-rate[h] dt) S + dt B x^T``
    (``S`` [N, P] per head);  ``y = (S^T C + D[h] x) * silu(z)``.  ``x``, ``bc``, ``z`` are activations of one type and
    may be column slices; ``dtp`` [T, H] fp32 (row stride free).  ``state`` [slots, H P, N] fp32 is read (past
    position 0) and advanced.  Returns y [T, H P] fp32.  ``fast_exp``: the hardware exponentials (relative error
    about 1e-6) instead of ``expf`` / ``log1pf``."""
    T, C = x.shape
    y = torch.empty(T, C, dtype=torch.float32, device=x.device)
    if use_hip(x):
        assert C == H * P and H % G == 0 and 1 <= N <= 128 and bc.shape[1] == 2 * G * N
        assert x.stride(1) == bc.stride(1) == z.stride(1) == dtp.stride(1) == 1 and x.dtype == bc.dtype == z.dtype
        assert dtp.dtype == torch.float32 and dtp.shape[1] == H and z.shape[1] == C
        assert dt_bias.dtype == rate.dtype == D.dtype == torch.float32 and dt_bias.numel() == rate.numel() == D.numel() == H
        assert state.is_contiguous() and state.shape[1:] == (C, N)
        # long portions: chunks in parallel (end states from zero + the sum of step sizes, a carry over the
        # chunks, the chunks again from their start states); short ones, and steps whose sequences x channels
        # already fill the chip, token by token
        cr = seg.chunk_ranges(SSM_CHUNK, 2 * SSM_CHUNK) if seg.n_seg * C < SEQ_FILL_LANES else None
        chunks, c0, cs, csd, nch = None, None, None, None, 0
        if cr is not None:
            chunks, c0 = cr
            nch = chunks.shape[0]
            cs = scratch(nch * C * N, torch.float32, x.device)
            csd = scratch(nch * C, torch.float32, x.device)
        check(lib().k8s_ssd_scan(ptr(x), x.stride(0), ptr(bc), bc.stride(0), _dt(x.dtype), ptr(dtp), dtp.stride(0),
                                 ptr(dt_bias), ptr(rate), ptr(D), ptr(z), z.stride(0), ptr(state), ptr(seg.seg_row0),
                                 ptr(seg.seg_pos0), ptr(seg.seg_slot), ptr(y), seg.n_seg, H, P, G, N, T,
                                 int(fast_exp), stream_ptr(x), ptr(chunks), nch, ptr(c0), ptr(cs), ptr(csd)),
              "ssd_scan")
        return y
    dt = torch.nn.functional.softplus(dtp.float() + dt_bias)                 # [T, H]
    dec = torch.exp(-rate * dt)
    xf, zf = x.float().view(T, H, P), z.float()
    rep = H // G
    Bm = bc[:, :G * N].float().view(T, G, N).repeat_interleave(rep, 1)      # [T, H, N]
    Cm = bc[:, G * N:].float().view(T, G, N).repeat_interleave(rep, 1)
    for s in range(seg.n_seg):
        a, e, p0, sl = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s], seg.slot_host[s]
        S = state[sl].view(H, P, N).clone() if p0 > 0 else torch.zeros(H, P, N)
        for r in range(a, e):
            S = dec[r][:, None, None] * S + (dt[r][:, None] * xf[r])[:, :, None] * Bm[r][:, None, :]
            o = torch.einsum("hpn,hn->hp", S, Cm[r]) + D[:, None] * xf[r]
            y[r] = o.reshape(-1) * torch.nn.functional.silu(zf[r])
        state[sl] = S.reshape(C, N)
    return y


def retention(qkvg: torch.Tensor, H: int, D: int, V: int, decay: torch.Tensor, rot_dims: int, rot_base: float,
              state: torch.Tensor, seg: SegMeta, positions: torch.Tensor, eps: float, out_dtype) -> torch.Tensor:
    """Retention per head, fp32: rows of ``qkvg`` [T, 2HD + 2HV] fp32 = (q | k | v | g).  q and k are
    rotated on their first ``rot_dims`` entries (entry i paired with i + rot_dims / 2, angle
    ``pos * rot_base^(-2i / rot_dims)``), k is scaled by ``D^(-1/2)``; ``S <- decay_h S + k v^T``;
    ``o = S^T q``; the result is ``o / rms(o) * silu(g)`` [T, H * V].  ``state`` [slots, H, D, V] fp32.
    On the device q and k are rotated IN PLACE in ``qkvg``."""
    T = qkvg.shape[0]
    out = torch.empty(T, H * V, dtype=out_dtype, device=qkvg.device)
    if use_hip(qkvg):
        assert qkvg.dtype == torch.float32 and qkvg.stride(1) == 1 and qkvg.shape[1] == 2 * H * (D + V)
        assert state.is_contiguous() and state.shape[1:] == (H, D, V) and decay.dtype == torch.float32
        oraw = scratch(T * H * V, torch.float32, qkvg.device)
        # long portions: chunks in parallel (end states from zero, a carry over the chunks, the chunks
        # again from their start states); short ones token by token
        cr = seg.chunk_ranges(SSM_CHUNK, 2 * SSM_CHUNK) if seg.n_seg * H * V * 8 < SEQ_FILL_LANES else None
        chunks, c0, cs, nch = None, None, None, 0
        if cr is not None:
            chunks, c0 = cr
            nch = chunks.shape[0]
            cs = scratch(nch * H * D * V, torch.float32, qkvg.device)
        check(lib().k8s_retention(ptr(qkvg), qkvg.stride(0), ptr(positions), ptr(decay), ptr(state), ptr(seg.seg_row0),
                                  ptr(seg.seg_pos0), ptr(seg.seg_slot), ptr(out), seg.n_seg, H, D, V, rot_dims,
                                  float(rot_base), float(eps), _dt(out_dtype), stream_ptr(qkvg), T, ptr(oraw),
                                  ptr(chunks), nch, ptr(c0), ptr(cs)), "retention")
        return out
    half = rot_dims // 2
    f = torch.exp(-(2.0 * torch.arange(half, dtype=torch.float64) / max(rot_dims, 1)) * math.log(rot_base))
    ang = positions.double()[:, None] * f[None]
    co, si = ang.cos().float()[:, None, :], ang.sin().float()[:, None, :]

    def rot(x):
        u, v = x[..., :half], x[..., half:rot_dims]
        return torch.cat([u * co - v * si, v * co + u * si, x[..., rot_dims:]], -1)

    q = rot(qkvg[:, :H * D].view(T, H, D))
    k = rot(qkvg[:, H * D:2 * H * D].view(T, H, D)) * D ** -0.5
    v = qkvg[:, 2 * H * D:2 * H * D + H * V].view(T, H, V)
    g = qkvg[:, 2 * H * D + H * V:].view(T, H, V)
    for s in range(seg.n_seg):
        a, e, p0, sl = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s], seg.slot_host[s]
        S = state[sl].clone() if p0 > 0 else torch.zeros(H, D, V)
        for r in range(a, e):
            S = decay[:, None, None] * S + k[r][:, :, None] * v[r][:, None, :]
            o = torch.einsum("hdv,hd->hv", S, q[r])
            o = o * torch.rsqrt(o.pow(2).mean(-1, keepdim=True) + eps) * torch.nn.functional.silu(g[r])
            out[r] = o.reshape(-1).to(out_dtype)
        state[sl] = S
    return out


def decay_attention(x: torch.Tensor, H: int, D: int, V: int, decay: torch.Tensor, state: torch.Tensor, seg: SegMeta,
                    silu: bool = False) -> torch.Tensor:
    """Linear attention with a fixed decay per head, fp32: rows of ``x`` [T, >= 2 H D + H V] = (q | k | v) activations
    (row stride free), with ``silu`` each of them through ``z sigmoid(z)`` first, as activations of ``x``'s type;  ``S <- decay_h S + k v^T``;  ``o = S^T q``.
    ``decay`` [H] fp32.  ``state`` [slots, H, D, V] fp32 is read (past position 0) and advanced.  Returns o [T, H V] fp32."""
    T = x.shape[0]
    out = torch.empty(T, H * V, dtype=torch.float32, device=x.device)
    if use_hip(x):
        assert x.stride(1) == 1 and x.shape[1] >= H * (2 * D + V) and decay.dtype == torch.float32 and decay.numel() == H
        assert state.is_contiguous() and state.dtype == torch.float32 and state.shape[1:] == (H, D, V)
        # long portions: chunks in parallel (end states from zero, a carry over the chunks, the chunks
        # again from their start states); short ones token by token.  On the matrix cores a portion goes in
        # blocks of 64 tokens, and its chunks are ranges of several blocks
        lens, longest = seg._once("lens", lambda: _lens(seg))
        mfma = longest >= LIN_MFMA_ROWS and decay_mfma_ok(D, V, x.dtype, x.device) and x.stride(0) % 4 == 0
        if mfma:
            cr, two = seg._once(("decay", H, D, V, LIN_GROUPS), lambda: _lin_plan(seg, T, lens, H, D, V))
        else:
            cr = seg.chunk_ranges(SSM_CHUNK, 2 * SSM_CHUNK) if seg.n_seg * H * V * 8 < SEQ_FILL_LANES else None
        chunks, c0, cs, nch = None, None, None, 0
        if cr is not None:
            chunks, c0 = cr
            nch = chunks.shape[0]
            cs = scratch(nch * H * D * V, torch.float32, x.device)
        if mfma:
            check(lib().k8s_decay_attn_mfma(ptr(x), x.stride(0), int(silu), ptr(decay), ptr(state), ptr(seg.seg_row0),
                                            ptr(seg.seg_pos0), ptr(seg.seg_slot), ptr(out), seg.n_seg, H, D, V,
                                            stream_ptr(x), ptr(chunks), nch, ptr(c0), ptr(cs),
                                            two), "decay_attn_mfma")
            return out
        check(lib().k8s_decay_attn(ptr(x), x.stride(0), _dt(x.dtype), int(silu), ptr(decay), ptr(state),
                                   ptr(seg.seg_row0), ptr(seg.seg_pos0), ptr(seg.seg_slot), ptr(out), seg.n_seg, H, D, V,
                                   stream_ptr(x), ptr(chunks), nch, ptr(c0), ptr(cs)), "decay_attn")
        return out
    qkv = x[:, :H * (2 * D + V)].float()
    if silu:
        qkv = torch.nn.functional.silu(qkv).to(x.dtype).float()
    q, k, v = qkv[:, :H * D].view(T, H, D), qkv[:, H * D:2 * H * D].view(T, H, D), qkv[:, 2 * H * D:].view(T, H, V)
    for s in range(seg.n_seg):
        a, e, p0, sl = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s], seg.slot_host[s]
        S = state[sl].clone() if p0 > 0 else torch.zeros(H, D, V)
        for r in range(a, e):
            S = decay[:, None, None] * S + k[r][:, :, None] * v[r][:, None, :]
            out[r] = torch.einsum("hdv,hd->hv", S, q[r]).reshape(-1)
        state[sl] = S
    return out


LIN_MFMA_ROWS = 17      # rows of a step's longest portion from which the matrix-core form runs
LIN_CHUNK = 128         # rows at least per range where ranges of a portion run in parallel
LIN_GROUPS = 256        # workgroups (ranges x heads x 128 value columns) a step is cut into


LIN_WALK = 768, 512     # rows the longest portion may walk past the chip's share, with up to 512 workgroups and with more


def _lin_rows(T: int, n_seg: int, H: int, D: int, V: int, lens: Optional[List[int]] = None) -> int:
    """Rows of a range, 0: portions stay whole.  ``lens``: the portions' rows (without them they are taken as equal).  As many
    ranges as give the chip a workgroup per unit;  of the form that two workgroups of a unit share
    (csrc/kernels/linear_attn.hip) two, where no portion has more than a fifth of the rows, as the carry walks all ranges of a
    portion, and one each would be ranges of 512 rows or more than 256 of them (us of 16 heads of 128 at 256 / 512
    workgroups: 31 x 512 + 2048 rows 363 / 299, 7 of 351 to 701 88 / 78, 5 x 1000 107 / 83, but 4 x 1000 64 / 71, 4 x 600 54 /
    60, 1 x 4000 67 / 75, 15 single rows + 4000 198 / 282;  of 4 heads 16 x 1024 65 / 74, 5 x 2000 51 / 60).

    Whole, where the portions are 256 workgroups or more by themselves and the longest is not left walking alone: up to
    ``LIN_WALK`` rows past T H / 256, which is what a unit gets of the step, and fewer of them where not all workgroups run at
    once (whole / cut: 16 x 1024 117 / 184, 15 x 512 + 1024 107 / 167, 15 x 300 + 1000 106 / 128, 31 single rows + 768 133 /
    140, of 64 heads 15 + 512 175 / 188;  past the line 31 x 512 + 2048 378 / 299, 63 x 512 + 3072 850 / 549, 15 x 300 + 1500
    157 / 139, 63 single rows + 1000 222 / 198, 15 + 4000 412 / 198, of 64 heads 15 + 768 259 / 215)."""
    per, lens = H * -(-V // 128), lens or [-(-T // n_seg)] * n_seg
    rows, longest = max(LIN_CHUNK, -(-T // (64 * max(1, LIN_GROUPS // per))) * 64), max(lens)
    if D == 128 and V > 64:
        past = longest - LIN_WALK[n_seg * per > 2 * LIN_GROUPS]
        if n_seg * per >= LIN_GROUPS and past * LIN_GROUPS <= T * per:
            return 0
        if T >= 5 * longest and (rows >= 512 or per * sum(-(-n // rows) for n in lens if n > rows) > LIN_GROUPS):
            rows = max(LIN_CHUNK, -(-T // (64 * max(1, 2 * LIN_GROUPS // per))) * 64)
    return rows


def _lens(seg: SegMeta) -> tuple:
    lens = [b - a for a, b in zip(seg.row0_host[:-1], seg.row0_host[1:])]
    return lens, max(lens)


def _lin_plan(seg: SegMeta, T: int, lens: List[int], H: int, D: int, V: int) -> tuple:
    """(ranges as :meth:`SegMeta.chunk_ranges` gives them or None, whether two workgroups share a unit)."""
    rows = _lin_rows(T, seg.n_seg, H, D, V, lens)
    cut = seg.chunk_ranges(rows, rows) if rows else None       # (None: no portion is longer than a range)
    return cut, int(_lin_two(lens, rows if cut is not None else 0, H, V))


def _lin_two(lens: List[int], rows: int, H: int, V: int) -> bool:
    """Whether two workgroups of :func:`decay_attention` share a compute unit (heads of 128; ``rows``: of a range, 0: portions
    whole): where there are more than 256.  With fewer than 16 heads' columns those of a block (64 rows) or less, reply
    tokens above all, do not count: they end before the others meet (us counted / not: 8 heads, 48 single rows + 16 x 1000
    178 / 140, 63 + 600 112 / 100; 16 heads 24 + 8 x 1000 177 / 208, 31 + 768 134 / 158, 15 + 4000 195 / 206)."""
    per = H * -(-V // 128)
    least = 0 if per >= 16 else 64
    return per * sum(n // rows + (n % rows > least) if rows else n > least for n in lens) > LIN_GROUPS


def decay_mfma_ok(D: int, V: int, dtype, device) -> bool:
    """Whether the matrix-core form of :func:`decay_attention` takes these sizes (bf16 on the device only)."""
    if dtype != torch.bfloat16 or torch.device(device).type != "cuda":
        return False
    return bool(lib().k8s_decay_attn_mfma_ok(int(D), int(V)))


def window_mfma_ok(H: int, G: int, D: int, V: int, dtype, device) -> bool:
    """Whether the matrix-core window attention kernel takes these sizes (bf16 on the device only;
    the vector-pipe kernel runs everything else)."""
    if dtype != torch.bfloat16 or torch.device(device).type != "cuda":
        return False
    return bool(lib().k8s_window_attn_mfma_ok(int(H), int(G), int(D), int(V)))


WINDOW_TILE = 16    # query tokens per work item of the matrix-core window attention kernel
WINDOW_PART = 128   # keys per part when a step of few rows is split over the keys too
WINDOW_SPLIT_ITEMS = 32


def window_kv_write(qkv: torch.Tensor, k_off: int, kc: torch.Tensor, vc: torch.Tensor, slots: torch.Tensor,
                    vt: Optional[torch.Tensor] = None) -> None:
    """The key and value columns of the joint projection's rows (k at ``k_off``, v behind it) go to the
    pages ``kc`` [pages, BS, G D] / ``vc`` [pages, BS, G V] at ``slots`` (page * BS + offset), the values
    also to the transposed twin ``vt`` [pages, G V, BS] when given (the matrix-core kernel's PV operand)."""
    T = qkv.shape[0]
    nk, nv = kc.shape[-1], vc.shape[-1]
    BS = kc.shape[1]
    if use_hip(qkv):
        assert qkv.stride(1) == 1 and kc.is_contiguous() and vc.is_contiguous() and kc.dtype == vc.dtype == qkv.dtype
        assert qkv.shape[1] >= k_off + nk + nv
        assert vt is None or (vt.is_contiguous() and vt.dtype == qkv.dtype and vt.shape[1:] == (nv, BS))
        check(lib().k8s_window_kv_write(ptr(qkv), qkv.stride(0), k_off, nk, nv, ptr(slots), ptr(kc), ptr(vc), T,
                                        _dt(qkv.dtype), stream_ptr(qkv), ptr(vt), BS), "window_kv_write")
        return
    ok = slots >= 0
    sl = slots[ok].long()
    kc.view(-1, nk)[sl] = qkv[ok, k_off:k_off + nk]
    vc.view(-1, nv)[sl] = qkv[ok, k_off + nk:k_off + nk + nv]
    if vt is not None:
        vt[sl // BS, :, sl % BS] = qkv[ok, k_off + nk:k_off + nk + nv]


def window_attention(qkv: torch.Tensor, H: int, G: int, D: int, V: int, kc: torch.Tensor, vc: torch.Tensor,
                     r1: torch.Tensor, r2: torch.Tensor, talk: torch.Tensor, window: int, scale: float,
                     seg: SegMeta, vt: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Sliding-window attention of the rows' queries (the first H D columns of ``qkv``) over the paged
    keys and values, which already hold this step's rows: position i sees j with ``0 <= i - j < window``;
    ``s = scale q.k - r1[h] ln(1 + r2[h] (i - j))``; ``p_j = exp(s_j) / (1 + sum exp(s))`` (a sink of score 0
    without a value); the heads' weights are mixed, ``w_h = sum_g talk[h, g] p_g``, and head h applies
    its mixed weights to the values of key / value head ``h // (H // G)``.  Returns [T, H V].
    With the transposed value pages ``vt`` (bf16, sizes of :func:`window_mfma_ok`) the matrix-core
    kernel runs: tiles of ``WINDOW_TILE`` tokens, the weights rounded to bf16 for the value product."""
    T = qkv.shape[0]
    BS = kc.shape[1]
    out = torch.empty(T, H * V, dtype=qkv.dtype, device=qkv.device)
    if use_hip(qkv):
        assert qkv.stride(1) == 1 and kc.is_contiguous() and vc.is_contiguous() and kc.dtype == vc.dtype == qkv.dtype
        assert kc.shape[-1] == G * D and vc.shape[-1] == G * V and seg.block_tables.is_contiguous()
        assert r1.dtype == r2.dtype == talk.dtype == torch.float32 and talk.is_contiguous() and H % G == 0
        if vt is not None and window_mfma_ok(H, G, D, V, qkv.dtype, qkv.device) and qkv.stride(0) % 8 == 0:
            assert vt.is_contiguous() and vt.shape[1:] == (G * V, BS) and BS % 32 == 0
            items = seg.tile_items(WINDOW_TILE)
            n_items = items.shape[0]
            # steps of few rows (decoding): the keys are split over workgroups as well -- parts of
            # WINDOW_PART keys counted from each tile's first key block, merged in part order
            n_parts, pml, po = 1, None, None
            if n_items <= WINDOW_SPLIT_ITEMS:
                kmax = max(p + b - a for p, a, b in zip(seg.pos0_host, seg.row0_host[:-1], seg.row0_host[1:]))
                span = min(int(window) + WINDOW_TILE + 30, -(-kmax // 32) * 32)
                n_parts = -(-span // WINDOW_PART)
                if n_parts > 1:
                    pml = scratch(n_items * n_parts * H * 32, torch.float32, qkv.device)
                    po = scratch(n_items * n_parts * 16 * H * V, torch.float32, qkv.device)
            check(lib().k8s_window_attn_mfma(ptr(qkv), qkv.stride(0), ptr(kc), ptr(vt), ptr(seg.block_tables),
                                             seg.block_tables.shape[1], ptr(items), n_items, ptr(r1), ptr(r2),
                                             ptr(talk), ptr(out), H, G, D, V, BS, int(window), float(scale),
                                             stream_ptr(qkv), WINDOW_PART, n_parts, ptr(pml), ptr(po)),
                  "window_attn_mfma")
            return out
        check(lib().k8s_window_attn_rows(ptr(qkv), qkv.stride(0), ptr(kc), ptr(vc), ptr(seg.block_tables),
                                         seg.block_tables.shape[1], ptr(seg.row_seg), ptr(seg.seg_row0),
                                         ptr(seg.seg_pos0), ptr(r1), ptr(r2), ptr(talk), ptr(out), T, H, G, D, V, BS,
                                         int(window), float(scale), _dt(qkv.dtype), stream_ptr(qkv)),
              "window_attn_rows")
        return out
    kf, vf = kc.view(-1, G, D), vc.view(-1, G, V)
    rep = H // G
    for s in range(seg.n_seg):
        a, e, p0 = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s]
        n, n_ctx = e - a, p0 + e - a
        lo = max(0, p0 - window + 1)
        kp = torch.arange(lo, n_ctx)
        rows = seg.block_tables[s].long()[kp // BS] * BS + kp % BS
        k = kf[rows].float().repeat_interleave(rep, 1)             # [ctx, H, D]
        v = vf[rows].float().repeat_interleave(rep, 1)             # [ctx, H, V]
        q = qkv[a:e, :H * D].float().view(n, H, D)
        dist = (p0 + torch.arange(n))[:, None] - kp[None, :]       # [n, ctx]
        sc = torch.einsum("thd,jhd->thj", q, k) * scale
        sc = sc - r1[None, :, None] * torch.log1p(r2[None, :, None] * dist.clamp_min(0).float()[:, None, :])
        vis = (dist >= 0) & (dist < window)
        sc = sc.masked_fill(~vis[:, None, :], float("-inf"))
        m = sc.amax(-1, keepdim=True).clamp_min(0.0)
        ex = torch.exp(sc - m)
        p = ex / (torch.exp(-m) + ex.sum(-1, keepdim=True))
        pm = torch.einsum("hg,tgj->thj", talk, p)
        out[a:e] = torch.einsum("thj,jhv->thv", pm, v).reshape(n, H * V).to(qkv.dtype)
    return out


# ------------------------------------------------------------------ masked softmax attention with a prepared q / k,
# and matrix-state recurrences (csrc/kernels/masked_attn.hip, matrix_mem.hip)
@dataclass
class Rope:
    """A rotation of the first ``dims`` entries of every head: pair i turns by ``pos * freq[i]`` and cos and sin are
    multiplied by ``amp``.  ``pairs``: pair i is the neighbouring entries 2i and 2i + 1 (else i and i + dims / 2)."""
    dims: int
    freq: torch.Tensor         # [dims / 2] fp64, on the model's device
    amp: float = 1.0
    pairs: bool = False


def make_rope(dims: int, base: float, device, pairs: bool = False, yarn: Optional[Tuple[float, float, float, float]] = None,
              stretch: Optional[Tuple[float, float, float, float]] = None) -> Rope:
    """:class:`Rope` with ``freq[i] = base^(-2 i / dims)``.  ``yarn = (factor, original, fast, slow)``: a pair that turns
    more than ``fast`` times within ``original`` positions keeps its frequency, one that turns less than ``slow`` times
    has it divided by ``factor``, with a linear ramp over the pair index between the two, and
    ``amp = 0.1 ln(factor) + 1``.  ``stretch = (factor, low, high, original)``: by wavelength ``l = 2 pi / freq`` -- kept
    below ``original / high``, divided by ``factor`` above ``original / low``, and between the two a mix of both by
    ``s = (original / l - low) / (high - low)``, the kept one's share."""
    f = torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=torch.float64)
    amp = 1.0
    if yarn is not None:
        factor, original, fast, slow = (float(v) for v in yarn)

        def border(turns):
            return dims * math.log(original / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

        lo, hi = max(math.floor(border(fast)), 0), min(math.ceil(border(slow)), dims - 1)
        ramp = ((torch.arange(dims // 2, dtype=torch.float64) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f = f / factor * ramp + f * (1.0 - ramp)
        amp = 0.1 * math.log(factor) + 1.0
    if stretch is not None:
        factor, low, high, original = (float(v) for v in stretch)
        turns = original * f / (2.0 * math.pi)                     # original / wavelength
        s = ((turns - low) / (high - low) if high != low else torch.zeros_like(turns))
        f = torch.where(turns > high, f, torch.where(turns < low, f / factor, (1.0 - s) * f / factor + s * f))
    return Rope(dims, f.to(device), amp, pairs)


def rope_table(positions: torch.Tensor, rope: Rope) -> torch.Tensor:
    """[T, dims] fp32: ``amp cos(pos freq)`` | ``amp sin(pos freq)`` of a step's positions, made once for all its layers."""
    T, half = positions.shape[0], rope.dims // 2
    if use_hip(positions):
        assert positions.dtype == torch.int32 and rope.freq.dtype == torch.float64 and rope.freq.device == positions.device
        cs = torch.empty(T, rope.dims, dtype=torch.float32, device=positions.device)
        check(lib().k8s_rope_table(ptr(positions), ptr(rope.freq), float(rope.amp), ptr(cs), T, half,
                                   stream_ptr(positions)), "rope_table")
        return cs
    ang = positions.double()[:, None] * rope.freq[None]
    return torch.cat([ang.cos().float(), ang.sin().float()], 1) * rope.amp


class RopeTables:
    """:func:`rope_table` of a step's rotations: tensors that the launch which embeds the step's tokens fills
    (:func:`.norm.hyper_embed`, :func:`.norm.embed_scale_dyt`: up to two of them), and further ones, filled at once."""
    IN_EMBED = 2

    def __init__(self, positions: torch.Tensor, ropes):
        self.positions, self.ropes = positions, list(ropes)[:self.IN_EMBED]
        self.cs = [torch.empty(positions.shape[0], r.dims, dtype=torch.float32, device=positions.device) for r in self.ropes]
        self._of = {id(r): cs for r, cs in zip(self.ropes, self.cs)}
        for r in list(ropes)[self.IN_EMBED:]:
            self._of[id(r)] = rope_table(positions, r)

    def of(self, rope: Optional[Rope]) -> Optional[torch.Tensor]:
        return None if rope is None else self._of[id(rope)]

    def fill(self) -> None:
        for r, cs in zip(self.ropes, self.cs):
            cs.copy_(rope_table(self.positions, r))

    def args(self) -> tuple:
        """What the launch takes."""
        assert self.positions.dtype == torch.int32 and self.positions.is_contiguous()
        out = [ptr(self.positions)]
        for r, cs in zip(self.ropes, self.cs):
            assert r.freq.dtype == torch.float64 and r.freq.device == self.positions.device
            out += [ptr(r.freq), float(r.amp), r.dims // 2, ptr(cs)]
        return tuple(out + [0, 0.0, 0, 0] * (self.IN_EMBED - len(self.ropes)))


def attn_prep(qkv: torch.Tensor, bias: Optional[torch.Tensor], H: int, G: int, D: int, V: int,
              positions: torch.Tensor, slots: torch.Tensor, kc: Optional[torch.Tensor], vc: Optional[torch.Tensor],
              out_dtype, norm=False, q_w: Optional[torch.Tensor] = None, k_w: Optional[torch.Tensor] = None,
              eps: float = 0.0, rot_dims: int = 0, rot_base: float = 10000.0, lam: float = 0.0,
              v_other: Optional[torch.Tensor] = None, v_keep: Optional[torch.Tensor] = None,
              vt: Optional[torch.Tensor] = None, maps: int = 1, v_is_k: bool = False,
              q_temp: Optional[Tuple[float, int]] = None, rope: Optional[Rope] = None,
              rope_cs: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Between the joint projection and attention, one pass over the fp32 rows of ``qkv`` [T, H M D + G M D + G V]
    = (q | k | v) with ``M = maps`` score maps per head (q and k laid out [head][map][D]):  add ``bias`` (fp32, same
    width, optional);  rotate q and k on their first ``rot_dims`` entries per head (entry i paired with
    i + rot_dims / 2, angle ``pos * rot_base^(-2 i / rot_dims)``);  with ``norm`` (True or "head") divide every q and k
    head by its root mean square (``eps`` inside the root) and multiply by ``q_w`` / ``k_w`` [D] where given -- behind
    the rotation;  with ``norm="all"`` divide q, and k, by the root mean square of the WHOLE projection and multiply by
    ``q_w`` [H M D] / ``k_w`` [G M D] -- in front of the rotation;  with ``q_temp = (coef, every)`` multiply q by
    ``1 + coef ln(floor((pos + 1) / every) + 1)``;  with ``rope`` (:class:`Rope`) its frequencies, pairing and amplitude
    replace ``rot_dims`` / ``rot_base`` (``rope_cs``: its :func:`rope_table` of these rows, where several layers share
    one);  ``v_keep`` [T, G V] fp32 receives the values as projected;  with
    ``v_other`` the values become ``(1 - lam) v + lam v_other``.  ``v_is_k``: there are no value columns, the values
    are the keys as projected (before norm and rotation; V = M D).  k and v go to the pages ``kc`` [pages, BS, G M D] /
    ``vc`` [pages, BS, G V] at ``slots`` (and v to the transposed twin ``vt`` when given, then ``vc`` may be None); q is returned [T, H M D] as
    activations.  ``G = 0``: only queries (a layer that reads another layer's pages).  ``qkv`` [S, T, ..]: the sum of its
    planes (:func:`.linear.proj_planes`)."""
    planes, pstep = 1, 0
    by16 = (kc is None or kc.data_ptr() % 16 == 0) and (rope_cs is None or rope_cs.data_ptr() % 16 == 0)    # (attn_prep_half)
    if qkv.dim() == 3:
        if qkv.shape[0] > 1 and use_hip(qkv) and by16 and norm in (False, None, True, "head") and not q_temp and 8 <= D <= 512 \
                and D & (D - 1) == 0 and (rope is None or (rope_cs is not None and not rope.pairs and rope.dims % 8 == 0)) \
                and not (rope is None and rot_dims) and qkv.stride(1) % 4 == 0 and qkv.data_ptr() % 16 == 0 \
                and qkv.stride(0) % 4 == 0 and qkv.shape[1] <= 1024 and (norm or bias is not None):
            planes, pstep, qkv = qkv.shape[0], qkv.stride(0), qkv[0]      # added where the rows are read
        else:
            qkv = qkv[0] if qkv.shape[0] == 1 else qkv.sum(0)
    T = qkv.shape[0]
    HQ, GK = H * maps, G * maps
    NQ, NK, NV = HQ * D, GK * D, G * V
    mode = {False: 0, None: 0, True: 1, "head": 1, "all": 2}[norm]
    v_col = NQ if v_is_k else NQ + NK
    assert not v_is_k or NV == NK
    q_out = torch.empty(T, NQ, dtype=out_dtype, device=qkv.device)
    BS = kc.shape[1] if kc is not None else 1
    tq_coef, tq_every = (float(q_temp[0]), int(q_temp[1])) if q_temp else (0.0, 0)
    if rope is not None:
        rot_dims = rope.dims
    if use_hip(qkv):
        assert qkv.dtype == torch.float32 and qkv.stride(1) == 1 and qkv.shape[1] == v_col + NV
        if G:
            assert kc.is_contiguous() and kc.dtype == out_dtype and kc.shape[-1] == NK and (vc is not None or vt is not None)
            assert vc is None or (vc.is_contiguous() and vc.dtype == out_dtype and vc.shape[-1] == NV)
        assert rope is None or (rope.freq.dtype == torch.float64 and rope.freq.device == qkv.device)
        assert rot_dims % 2 == 0 and 0 <= rot_dims <= D
        for t, n in ((bias, v_col + NV), (q_w, NQ if mode == 2 else D), (k_w, NK if mode == 2 else D)):
            assert t is None or (t.dtype == torch.float32 and t.is_contiguous() and t.numel() == n)
        for t in (v_other, v_keep):
            assert t is None or (t.dtype == torch.float32 and t.is_contiguous() and t.shape == (T, NV))
        assert vt is None or (vt.is_contiguous() and vt.dtype == out_dtype and vt.shape[1:] == (NV, BS))
        assert rope_cs is None or (rope_cs.dtype == torch.float32 and rope_cs.is_contiguous()
                                   and rope_cs.shape == (T, rot_dims))
        if (mode == 0 and bias is None and v_other is None and v_keep is None and not tq_every and D % 4 == 0
                and qkv.stride(0) % 4 == 0 and qkv.data_ptr() % 16 == 0
                and (rot_dims == 0 or (rope is not None and rope.pairs and rope_cs is not None))):
            # nothing couples a row's entries beyond their rotation pair: memory to memory
            check(lib().k8s_attn_prep_pairs(ptr(qkv), qkv.stride(0), HQ, GK, D, NV, v_col, ptr(slots), ptr(kc), ptr(vc),
                                            ptr(vt), BS, ptr(q_out), _dt(out_dtype), int(rot_dims), ptr(rope_cs), T,
                                            stream_ptr(qkv)), "attn_prep_pairs")
            return q_out
        if (mode < 2 and by16 and not tq_every and 8 <= D <= 512 and D & (D - 1) == 0
                and qkv.stride(0) % 4 == 0 and qkv.data_ptr() % 16 == 0 and rot_dims % 8 == 0
                and (rot_dims == 0 or (rope is not None and not rope.pairs and rope_cs is not None))):
            # a head's entries meet in its rotation and its norm alone: a few lanes per head, no LDS
            check(lib().k8s_attn_prep_half(ptr(qkv), qkv.stride(0), HQ, GK, D, NV, v_col, ptr(bias), ptr(slots), ptr(kc),
                                           ptr(vc), ptr(vt), BS, ptr(q_out), _dt(out_dtype), int(rot_dims), ptr(rope_cs),
                                           mode, ptr(q_w), ptr(k_w), float(eps), T, stream_ptr(qkv), float(lam),
                                           ptr(v_other), ptr(v_keep), planes, pstep), "attn_prep_half")
            return q_out
        check(lib().k8s_attn_prep(ptr(qkv), qkv.stride(0), ptr(bias), HQ, GK, D, NV, ptr(positions), ptr(slots),
                                  ptr(kc), ptr(vc), ptr(vt), BS, ptr(q_out), _dt(out_dtype), mode, ptr(q_w),
                                  ptr(k_w), float(eps), int(rot_dims), float(rot_base), float(lam), ptr(v_other),
                                  ptr(v_keep), T, stream_ptr(qkv), v_col, tq_coef, tq_every,
                                  ptr(rope.freq) if rope is not None else None, rope.amp if rope is not None else 1.0,
                                  int(rope is not None and rope.pairs), ptr(rope_cs)), "attn_prep")
        return q_out
    x = qkv + bias if bias is not None else qkv
    q, k, v = x[:, :NQ], x[:, NQ:NQ + NK], x[:, v_col:v_col + NV]
    if mode == 2:
        q = q * torch.rsqrt(q.pow(2).mean(-1, keepdim=True) + eps) * (q_w if q_w is not None else 1.0)
        if NK:
            k = k * torch.rsqrt(k.pow(2).mean(-1, keepdim=True) + eps) * (k_w if k_w is not None else 1.0)
    q, k = q.reshape(T, HQ, D), k.reshape(T, GK, D)
    if rot_dims:
        half = rot_dims // 2
        if rope is None:
            f = torch.exp(-(2.0 * torch.arange(half, dtype=torch.float64) / rot_dims) * math.log(rot_base))
            rope_cs = rope_table(positions, Rope(rot_dims, f))
        elif rope_cs is None:
            rope_cs = rope_table(positions, rope)
        co, si = rope_cs[:, None, :half], rope_cs[:, None, half:]

        def rot(z):
            if rope is not None and rope.pairs:
                a, b = z[..., 0:rot_dims:2], z[..., 1:rot_dims:2]
                ab = torch.stack([a * co - b * si, b * co + a * si], -1).flatten(-2)
                return torch.cat([ab, z[..., rot_dims:]], -1)
            a, b = z[..., :half], z[..., half:rot_dims]
            return torch.cat([a * co - b * si, b * co + a * si, z[..., rot_dims:]], -1)

        q, k = rot(q), rot(k)
    if mode == 1:
        q = q * torch.rsqrt(q.pow(2).mean(-1, keepdim=True) + eps)
        k = k * torch.rsqrt(k.pow(2).mean(-1, keepdim=True) + eps)
        if q_w is not None:
            q = q * q_w
        if k_w is not None:
            k = k * k_w
    if tq_every:
        temp = 1.0 + tq_coef * torch.log(torch.div(positions + 1, tq_every, rounding_mode="floor").float() + 1.0)
        q = q * temp[:, None, None]
    if v_keep is not None:
        v_keep.copy_(v)
    if v_other is not None:
        v = (1.0 - lam) * v + lam * v_other
    if G:
        ok = slots >= 0
        sl = slots[ok].long()
        kc.view(-1, NK)[sl] = k.reshape(T, NK)[ok].to(kc.dtype)
        if vc is not None:
            vc.view(-1, NV)[sl] = v[ok].to(vc.dtype)
        if vt is not None:
            vt[sl // BS, :, sl % BS] = v[ok].to(vt.dtype)
    q_out.copy_(q.reshape(T, NQ).to(out_dtype))
    return q_out


def masked_attention(q: torch.Tensor, H: int, G: int, D: int, V: int, kc: torch.Tensor, vc: Optional[torch.Tensor],
                     seg: SegMeta, scale: float, softcap: float = 0.0, chunk: int = 0, window: int = 0,
                     keep_first: int = 0, sink: Optional[torch.Tensor] = None, gate: Optional[torch.Tensor] = None,
                     vt: Optional[torch.Tensor] = None, maps: int = 1, out_f32: bool = False) -> torch.Tensor:
    """Softmax attention of the rows' queries ``q`` [T, H D] over the paged keys and values (which already
    hold this step's rows), query head h reading key / value head ``h // (H // G)``.  Position i sees j <= i
    with, for ``chunk`` > 0, ``i // chunk == j // chunk`` and, for ``window`` > 0, ``i - j < window or j < keep_first``
    (positions count from the sequence's start).  ``s = scale q.k``, then ``softcap * tanh(s / softcap)`` for
    ``softcap`` > 0.  ``sink`` [H] fp32 adds ``exp(sink_h)`` to head h's denominator (no key, no value).  ``gate``
    [T, >= H] fp32 (row stride free): head h's output is multiplied by ``sigmoid(gate[t, h])``.
    Returns [T, H V].  With the transposed value pages ``vt`` (bf16, sizes of :func:`masked_mfma_ok`) the
    matrix-core kernel runs and ``vc`` is not read (it may be None).
    ``maps`` = M > 1: every head has M score maps -- ``q`` is [T, H M D] and the key pages [.., G M D], both laid out
    [head][map][D]; map m of head h scores against key head ``(h // (H // G)) M + m``, has a softmax of its own and
    applies it to value head ``h // (H // G)``; the result is [T, H M V], every map's by itself (``sink`` and ``gate``
    then count H M).  ``out_f32``: the result in fp32 whatever the activation type."""
    T = q.shape[0]
    BS = kc.shape[1]
    HQ = H * maps
    out = torch.empty(T, HQ * V, dtype=torch.float32 if out_f32 else q.dtype, device=q.device)
    if use_hip(q):
        assert q.is_contiguous() and q.shape[1] == HQ * D and kc.is_contiguous() and H % G == 0
        assert kc.dtype == q.dtype and kc.shape[-1] == G * maps * D
        assert vc is None or (vc.is_contiguous() and vc.dtype == q.dtype and vc.shape[-1] == G * V)
        assert seg.block_tables.is_contiguous() and chunk >= 0 and window >= 0 and keep_first >= 0
        assert sink is None or (sink.dtype == torch.float32 and sink.shape[0] == HQ)
        assert gate is None or (gate.dtype == torch.float32 and gate.stride(1) == 1 and gate.shape[1] >= HQ)
        gs = gate.stride(0) if gate is not None else 0
        if vt is not None and masked_mfma_ok(H, G, D, V, q.dtype, q.device):
            assert vt.is_contiguous() and vt.shape[1:] == (G * V, BS) and BS % 32 == 0
            common = (ptr(sink), ptr(gate), gs, ptr(out), H, G, D, V, BS, int(chunk), int(window), int(keep_first),
                      float(scale), float(softcap), stream_ptr(q))
            rows, r_parts, tiles, t_parts, pb, row0 = seg._once(
                ("mask plan", H, G, D, V, chunk, window, keep_first, maps),
                lambda: _mask_plan(seg, H, G, D, V, int(chunk), int(window), int(keep_first), int(maps)))
            bt, maxb = seg.block_tables, seg.block_tables.shape[1]
            if rows.shape[0]:
                groups, po, pml = _token_groups(rows, HQ, r_parts, V)
                for it in groups:
                    check(lib().k8s_masked_attn_token(ptr(q), ptr(kc), ptr(vt), ptr(bt), maxb, ptr(it), it.shape[0],
                                                      *common, MASK_TOKEN_BLOCKS, TOKEN_PARTS, r_parts, ptr(pml), ptr(po),
                                                      int(maps), int(out_f32)), "masked_attn_token")
            if tiles.shape[0]:
                po = pml = None
                if t_parts > 1:
                    po, pml = (scratch((T - row0) * HQ * t_parts * n, torch.float32, q.device) for n in (V, 2))
                check(lib().k8s_masked_attn_prompt(ptr(q), ptr(kc), ptr(vt), ptr(bt), maxb, ptr(tiles), tiles.shape[0],
                                                   *common, int(maps), int(out_f32), t_parts, pb, row0, T - row0, ptr(po),
                                                   ptr(pml)), "masked_attn_prompt")
            return out
        assert vc is not None          # the vector-pipe kernel reads token-major values
        parts, po, pml = _rows_parts(seg, T, HQ, H // G, V, q.device, int(chunk), int(window), int(keep_first),
                                     tiles=q.dtype == torch.float32 and D % 16 == 0 == V % 64)
        check(lib().k8s_masked_attn_rows(ptr(q), ptr(kc), ptr(vc), ptr(seg.block_tables), seg.block_tables.shape[1],
                                         ptr(seg.row_seg), ptr(seg.seg_row0), ptr(seg.seg_pos0), ptr(sink), ptr(gate),
                                         gs, ptr(out), T, H, G, D, V, BS, int(chunk), int(window), int(keep_first),
                                         float(scale), float(softcap), _dt(q.dtype), stream_ptr(q), int(maps),
                                         int(out_f32), parts, ptr(po), ptr(pml)), "masked_attn_rows")
        return out
    kf, vf = kc.view(-1, G, maps, D), vc.view(-1, G, V)
    rep = H // G
    for s in range(seg.n_seg):
        a, e, p0 = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s]
        n, n_ctx = e - a, p0 + e - a
        kp = torch.arange(n_ctx)
        rows = seg.block_tables[s].long()[kp // BS] * BS + kp % BS
        k = kf[rows].float().repeat_interleave(rep, 1).reshape(n_ctx, HQ, D)                  # [ctx, H M, D]
        v = vf[rows].float().repeat_interleave(rep, 1).repeat_interleave(maps, 1)             # [ctx, H M, V]
        qi = (p0 + torch.arange(n))[:, None]
        vis = kp[None, :] <= qi
        if chunk > 0:
            vis &= (qi // chunk) == (kp[None, :] // chunk)
        if window > 0:
            vis &= ((qi - kp[None, :]) < window) | (kp[None, :] < keep_first)
        sc = torch.einsum("thd,jhd->thj", q[a:e].float().view(n, HQ, D), k) * scale
        if softcap > 0:
            sc = softcap * torch.tanh(sc / softcap)
        sc = sc.masked_fill(~vis[:, None, :], float("-inf"))
        m = sc.amax(-1, keepdim=True)
        if sink is not None:
            m = torch.maximum(m, sink[None, :, None])
        ex = torch.exp(sc - m)
        den = ex.sum(-1, keepdim=True)
        if sink is not None:
            den = den + torch.exp(sink[None, :, None] - m)
        o = torch.einsum("thj,jhv->thv", ex / den, v)
        if gate is not None:
            o = o * torch.sigmoid(gate[a:e, :HQ])[:, :, None]
        out[a:e] = o.reshape(n, HQ * V).to(out.dtype)
    return out


# Workgroups up to which the attention of single tokens prepares rows of 64-entry heads itself: past that the registers that
# hold the row take workgroups off the compute units.  us apart / together, 16 heads over 16 of 64:  7 rows at 700 keys (336
# workgroups) 15.7 / 14.4, 16 at 450 (512) 17.2 / 16.2, 7 at 1500 (672) 20.9 / 23.8, 64 at 512 (2048) 40 / 47.  Heads of 128
# gain at any number:  16 over 2 of 128 at 1 row and 100 keys 8.1 / 7.0, 7 at 700 14.0 / 12.2, 64 at 512 19.4 / 17.8;  8 over 8
# 8.9 / 8.0, 16.4 / 14.1, 41 / 38, 64 at 1500 (3072) 91 / 89.
PREP_GROUPS = 512


def proj_prep(h: torch.Tensor, w: torch.Tensor, bias: Optional[torch.Tensor], H: int, G: int, D: int, V: int, slots: torch.Tensor,
              kc: torch.Tensor, vc: Optional[torch.Tensor], vt: Optional[torch.Tensor], seg: SegMeta, norm=False,
              q_w: Optional[torch.Tensor] = None, k_w: Optional[torch.Tensor] = None, eps: float = 0.0, lam: float = 0.0,
              v_other: Optional[torch.Tensor] = None, v_keep: Optional[torch.Tensor] = None, rope: Optional[Rope] = None,
              rope_cs: Optional[torch.Tensor] = None) -> Optional[tuple]:
    """:func:`attn_prep` of the first ``(H + G) D + G V`` columns of ``h @ w.T`` and the other columns in fp32 (None where there are
    none), of many rows in one launch (csrc/kernels/gemm_prep.hip), or None: sizes, types or places that it does not take, or where
    :func:`.linear.prep_plan` leaves product and pass apart."""
    from . import linear as LIN
    T = slots.shape[0]
    if T < LIN.PREP_MIN_ROWS or T == seg.n_seg or not isinstance(h, torch.Tensor):
        return None
    NQ, NK, NV = H * D, G * D, G * V
    n, (N, K), rot = NQ + NK + NV, w.shape, rope.dims if rope is not None else 0
    if not (vt is not None and use_hip(h) and D in (64, 128) and norm in (False, None, True, "head") and N >= n and N % 4 == 0
            and NQ % 256 == NK % 256 == NV % 256 == 0 and NV > 0 and h.shape == (T, K) and LIN._few_ok(h, w) and h.stride(0) >= K
            and (rope is None or not rope.pairs and rope_cs is not None and 8 <= rot <= D and rot & (rot - 1) == 0)
            and unwatched(h, w)):
        return None
    BS, dt = kc.shape[1], torch.bfloat16
    small = ((bias, n), (q_w, D), (k_w, D), (v_other, T * NV), (v_keep, T * NV), (rope_cs, T * rot))
    if not (all(t is None or t.dtype == torch.float32 and t.is_contiguous() and t.numel() == m and t.data_ptr() % 16 == 0
                and t.device == h.device for t, m in small)
            and all(t is None or t.is_contiguous() and t.dtype == dt and t.data_ptr() % 16 == 0 for t in (kc, vc, vt))
            and all(t is None or t.shape == (T, m) for t, m in ((v_other, NV), (v_keep, NV), (rope_cs, rot)))
            and kc.shape[2] == NK and (vc is None or vc.shape[1:] == (BS, NV)) and vt.shape[1:] == (NV, BS)
            and slots.dtype == torch.int32 and slots.is_contiguous()):
        return None
    f = LIN.prep_plan(T, N, K, n)
    if f is None:
        return None
    q = torch.empty(T, NQ, dtype=dt, device=h.device)
    rest = torch.empty(T, N - n, dtype=torch.float32, device=h.device) if N > n else None
    check(lib().k8s_gemm_prep(ptr(h), h.stride(0), ptr(w), T, N, K, f, ptr(bias), ptr(rope_cs), rot, int(bool(norm)), ptr(q_w), ptr(k_w),
                              float(eps), float(lam), ptr(v_other), ptr(v_keep), ptr(slots), ptr(q), ptr(kc), ptr(vt), ptr(vc), BS, NQ, NK,
                              NV, D, ptr(rest), N - n, stream_ptr(h)), "gemm_prep")
    return q, rest


def prep_attention(x: torch.Tensor, bias: Optional[torch.Tensor], H: int, G: int, D: int, V: int, positions: torch.Tensor,
                   slots: torch.Tensor, kc: torch.Tensor, vc: Optional[torch.Tensor], vt: Optional[torch.Tensor], seg: SegMeta,
                   out_dtype, scale: float, prep: dict, mask: dict) -> torch.Tensor:
    """:func:`attn_prep` (keywords ``prep``) and :func:`masked_attention` (keywords ``mask``) of the same rows; in one launch
    where every sequence has one row."""
    return _prep_attention(x, bias, H, G, D, V, positions, slots, kc, vc, vt, seg, out_dtype, scale, prep, mask)


def _prep_attention(x, bias, H, G, D, V, positions, slots, kc, vc, vt, seg, out_dtype, scale, prep, mask, beside=None):
    o = _prep_tokens(x, bias, H, G, D, V, slots, kc, vc, vt, seg, out_dtype, scale, **prep, **mask, beside=beside)
    if o is not None:
        return o
    q = attn_prep(x, bias, H, G, D, V, positions, slots, kc, vc, out_dtype, vt=vt, **prep)
    return masked_attention(q, H, G, D, V, kc, vc, seg, scale, vt=vt, **mask)


def _prep_tokens(x, bias, H, G, D, V, slots, kc, vc, vt, seg, out_dtype, scale, norm=False, q_w=None, k_w=None, eps=0.0,
                 lam=0.0, v_other=None, v_keep=None, rope=None, rope_cs=None, softcap=0.0, chunk=0, window=0, keep_first=0,
                 sink=None, gate=None, beside=None) -> Optional[torch.Tensor]:
    """``beside`` (:class:`_MemoryStep`): made in the same launch, and marked so, where that takes it."""
    T = x.shape[-2]
    if T != seg.n_seg:                               # (before anything else: prompts pay for one comparison)
        return None
    planes, pstep = (x.shape[0], x.stride(0)) if x.dim() == 3 else (1, 0)
    rot, NV, cols = rope.dims if rope is not None else 0, G * V, (H + G) * D + G * V
    if not (use_hip(x) and vt is not None and D in (64, 128) and norm in (False, None, True, "head")
            and seg.singles() == T and masked_mfma_ok(H, G, D, V, out_dtype, x.device) and x.dtype == torch.float32
            and x.shape[-1] == cols and x.stride(-1) == 1 and x.stride(-2) % 4 == 0 and pstep % 4 == 0
            and (rope is None or not rope.pairs and rope_cs is not None and rot % 8 == 0 and rot <= D)):
        return None
    BS = kc.shape[1]
    small = ((bias, cols), (q_w, D), (k_w, D), (v_other, T * NV), (v_keep, T * NV), (rope_cs, T * rot), (sink, H))
    if not (all(t is None or t.dtype == torch.float32 and t.is_contiguous() and t.numel() == n for t, n in small)
            and all(t is None or t.data_ptr() % 16 == 0 for t in (x, kc, vc, rope_cs, v_other, v_keep))
            and all(t is None or t.is_contiguous() and t.dtype == out_dtype for t in (kc, vc, vt))
            and kc.shape[2] == G * D and (vc is None or vc.shape[2] == NV) and vt.shape[1:] == (NV, BS) and BS % 32 == 0
            and slots.dtype == torch.int32 and slots.is_contiguous() and seg.block_tables.is_contiguous()
            and chunk >= 0 and window >= 0 and keep_first >= 0
            and (gate is None or gate.dtype == torch.float32 and gate.stride(1) == 1 and gate.shape[1] >= H)):
        return None
    rows, parts, _, _, _, _ = seg._once(("mask plan", H, G, D, V, chunk, window, keep_first, 1),
                                        lambda: _mask_plan(seg, H, G, D, V, int(chunk), int(window), int(keep_first), 1))
    if D == 64 and T * G * -(-(H // G) // 16) * parts > PREP_GROUPS:
        return None
    out = torch.empty(T, H * V, dtype=out_dtype, device=x.device)
    groups, po, pml = _token_groups(rows, H, parts, V)
    joint = (beside is not None and H > G and D + V > 128 and softcap == 0.0 and parts < TOKEN_PARTS and MASK_TOKEN_BLOCKS <= 8
             and len(groups) == 1 and out_dtype == torch.bfloat16 == beside.out.dtype and (beside.dim, beside.vdim) != (128, 128))
    for it in groups:
        args = (
            ptr(x), x.stride(-2), planes, pstep, ptr(bias), ptr(q_w), ptr(k_w), float(eps), int(bool(norm)), ptr(rope_cs), rot,
            float(lam), ptr(v_other), ptr(v_keep), ptr(slots), ptr(vc), ptr(kc), ptr(vt), ptr(seg.block_tables),
            seg.block_tables.shape[1], ptr(it), it.shape[0], ptr(sink), ptr(gate), gate.stride(0) if gate is not None else 0,
            ptr(out), H, G, D, V, BS, int(chunk), int(window), int(keep_first), float(scale), float(softcap), stream_ptr(x),
            MASK_TOKEN_BLOCKS, TOKEN_PARTS, parts, ptr(pml), ptr(po))
        if joint:
            check(lib().k8s_masked_attn_memory(*args, *beside.args), "masked_attn_memory")
            beside.done = True
        else:
            check(lib().k8s_masked_attn_token_prep(*args), "masked_attn_token_prep")
    return out


def attention_and_memory(x: torch.Tensor, H: int, G: int, D: int, V: int, positions: torch.Tensor, slots: torch.Tensor, kc, vc, vt,
                         seg: SegMeta, out_dtype, scale: float, prep: dict, mask: dict, xm: torch.Tensor, *memory) -> tuple:
    """:func:`prep_attention` (without a bias) of ``x`` and :func:`memory_layer` of ``xm`` (with the further arguments), columns of
    the same rows.

    Of single tokens in one launch (csrc/kernels/token_attn.hip, MEM), at every number of them: us of both launches / one, 16 heads
    over 2 of 128 beside 16 of 64 x 128:  1 row at 100 keys 11.1 / 7.1, 5 at 1100 15.9 / 11.8, 64 at 450 34.7 / 31.5, 128 at 300 51.7 /
    49.9;  12 over 3 of 64 + 128 beside 32 of 64 x 64 10.6 / 6.9, 15.1 / 11.2, 37.3 / 33.4, 57.1 / 57.0.  Heads of 128 x 128 stay
    apart: their state does not fit beside the attention's registers."""
    # (the rows before anything else: prompts pay for one comparison)
    step = _memory_step(xm, *memory) if xm.shape[0] == seg.n_seg else None
    o = _prep_attention(x, None, H, G, D, V, positions, slots, kc, vc, vt, seg, out_dtype, scale, prep, mask, beside=step)
    return o, memory_layer(xm, *memory) if step is None else step.launch()


# Prompt tiles cut over their keys where few of them would leave the chip idle behind a long context.  us, whole / cut, 16
# heads over 2 of 128: 200 rows at 1000 keys 39 / 21, at 2000 62 / 26, at 8000 205 / 40;  1200 rows 64 / 50, 87 / 61, 227 /
# 136;  4 over 4 of 64 at 8000, 500 rows 242 / 24 (tiles of 16 tokens, cut over 32 parts, 74).  The more workgroups there are
# already, the longer a part has to be to pay for its share of the results' way to the merge: 16 over 2, 1200 rows in a window
# of 1024 (150 workgroups, 18 blocks) 37 whole, 41 in two parts;  32 over 8, 800 rows from 0 (200, 13) 30 / 35;  500 rows in
# the window (128, 18) 46 / 37.
MASK_TILE_FILL = 512     # workgroups the chip holds at once
MASK_TILE_BLOCKS = 4     # 64-key blocks of a part at least, and a fifteenth of the workgroups


def _tile_parts(groups: int, nblk: int) -> tuple:
    """(parts a tile's keys are cut into, 64-key blocks of a part) for a launch of ``groups`` workgroups without a cut."""
    n = min(MASK_TILE_FILL // groups, nblk // max(MASK_TILE_BLOCKS, groups // 15))
    if n < 2:
        return 1, 0
    pb = -(-nblk // n)
    return -(-nblk // pb), pb


def _mask_plan(seg: SegMeta, H: int, G: int, D: int, V: int, chunk: int, window: int, keep_first: int, maps: int) -> tuple:
    """How a step's rows are shared out, made once per step and kind of layer (5 us of the host): (items of one token, parts
    of their keys; tiles, parts of theirs, 64-key blocks of a part, the first tile's first row)."""
    def row_parts(kmax: int) -> int:      # parts of a row of so many keys: 32-key blocks
        nblk = -(-kmax // 32)
        if window > 0:     # the window from a block's border on; + the kept blocks
            nblk = min(nblk, (window + 62) // 32 + -(-keep_first // 32))
        if chunk > 0:
            nblk = min(nblk, (chunk + 62) // 32)
        return min(-(-nblk // MASK_TOKEN_BLOCKS), TOKEN_PARTS)

    tpi, hpg, T = max(1, MASK_TILE_ROWS // (H // G)), H // G, seg.row0_host[-1]
    per_row, n1, end = G * maps * -(-hpg // 16), seg.singles(), seg.n_seg
    tmax, row0 = seg.most_keys(n1, end), seg.row0_host[n1]
    most = min(chunk or 1 << 30, window + keep_first if window > 0 else 1 << 30)
    few = (row0 == T or (T - row0) * per_row * row_parts(tmax) <= MASK_ROW_GROUPS
           and (1 - 1.5 / (T - row0)) * seg.keys_behind(n1, most) * per_row * (D + V) * 2 <= MASK_ROW_BYTES)
    rows, tiles = seg.mask_items(tpi, few)
    r_parts, t_parts, pb = 1, 1, 0
    if rows.shape[0]:
        r_parts = row_parts(seg.most_keys(0, end if few else n1))
    if tiles.shape[0]:
        nblk = -(-tmax // 64)
        if window > 0:     # the first token's window from a block's border to the last token; + the kept blocks
            nblk = min(nblk, (window + tpi + 125) // 64 + -(-keep_first // 64))
        if chunk > 0:
            nblk = min(nblk, (chunk + tpi + 125) // 64)
        t_parts, pb = _tile_parts(tiles.shape[0] * G * maps * -(-hpg // MASK_TILE_ROWS), nblk)
    return rows, r_parts, tiles, t_parts, pb, row0


def masked_mfma_ok(H: int, G: int, D: int, V: int, dtype, device) -> bool:
    """Whether the matrix-core form of :func:`masked_attention` takes these sizes (bf16 on the device only)."""
    if dtype != torch.bfloat16 or torch.device(device).type != "cuda":
        return False
    fn = getattr(lib(), "k8s_masked_attn_mfma_ok", None)
    return bool(fn(int(H), int(G), int(D), int(V))) if fn is not None else False


def head_norm_gate(o: torch.Tensor, gate: Optional[torch.Tensor], w: Optional[torch.Tensor], H: int, V: int, eps: float,
                   out_dtype, mul: Optional[torch.Tensor] = None, sub_lambda: Optional[float] = None,
                   out_scale: float = 1.0) -> torch.Tensor:
    """``u / rms(u over each head's V) * w * sigmoid(gate) * out_scale`` of fp32 rows ``o`` [T, H V], ``u = o * mul`` with
    ``mul`` [T, H] where given; ``w`` [V] (shared by the heads) or [H V] or None; ``gate`` [T, H V] fp32 or bf16 (row
    stride free) or None.  With ``sub_lambda`` the rows hold two results per head, [T, H, 2, V], and
    ``u = o[:, :, 0] - sub_lambda * o[:, :, 1]`` (two score maps over the same values, joined)."""
    T = o.shape[0]
    out = torch.empty(T, H * V, dtype=out_dtype, device=o.device)
    sub = sub_lambda is not None
    if use_hip(o):
        assert o.dtype == torch.float32 and o.is_contiguous() and o.shape[1] == H * V * (2 if sub else 1)
        assert gate is None or (gate.dtype in (torch.float32, torch.bfloat16) and gate.stride(1) == 1
                                and gate.shape[1] >= H * V)
        assert w is None or (w.dtype == torch.float32 and w.numel() in (V, H * V))
        assert mul is None or (mul.dtype == torch.float32 and mul.is_contiguous() and mul.numel() == T * H)
        check(lib().k8s_head_norm_gate(ptr(o), ptr(gate), gate.stride(0) if gate is not None else 0, ptr(w),
                                       V if w is not None and w.numel() == H * V else 0,
                                       ptr(out), T, H, V, float(eps), _dt(out_dtype), stream_ptr(o), ptr(mul),
                                       int(sub), float(sub_lambda or 0.0), float(out_scale),
                                       _dt(gate.dtype) if gate is not None else 1), "head_norm_gate")
        return out
    if sub:
        oh = o.view(T, H, 2, V)
        oh = oh[:, :, 0] - sub_lambda * oh[:, :, 1]
    else:
        oh = o.view(T, H, V)
    if mul is not None:
        oh = oh * mul.view(T, H, 1)
    oh = oh * torch.rsqrt(oh.pow(2).mean(-1, keepdim=True) + eps) * out_scale
    if w is not None:
        oh = oh * (w.view(H, V) if w.numel() == H * V else w.view(1, V))
    if gate is not None:
        oh = oh * torch.sigmoid(gate[:, :H * V].float()).view(T, H, V)
    out.copy_(oh.reshape(T, H * V).to(out_dtype))
    return out


MAT_CHUNK = 64      # rows per chunk of the chunk-parallel matrix-state recurrences
MAT_FILL_GROUPS = 1024   # workgroups (segments x heads x 64-column blocks) from which token by token fills the chip


def _mat_chunks(seg: SegMeta, H: int, V: int):
    """The chunk ranges of a step for the matrix-state recurrences, or None where they run token by token:
    no long portion, or enough sequences that the sequential form fills the chip at less than half the work."""
    if seg.n_seg * H * -(-V // 64) >= MAT_FILL_GROUPS:
        return None
    return seg.chunk_ranges(MAT_CHUNK, 2 * MAT_CHUNK)


MAT_TILE = 16       # tokens per tile of the matrix-core form


def _long_and_few(seg: SegMeta, H: int, D: int, V: int) -> bool:
    """Whether the matrix memory of a step is a long serial chain beside a nearly idle chip.  The tiles walk a sequence at 0.9
    (D 16) to 2.1 us (D 128) a tile in a workgroup per head and 64 columns; chunks of 64 tokens run beside each other, until
    they too fill the chip, with 4 D bytes of state per thread.  us chunks / tiles at 1000, 2000, 4000 tokens, by workgroups:
    D 32, 4 73 / 79, 98 / 142, 148 / 279, 32 86 / 89, 127 / 160, 218 / 299, 64 100 / 93, 167 / 167;  D 64, 8 96 / 102, 136 /
    193, 233 / 368, 16 111 / 108, 187 / 198, 342 / 378, 32 160 / 114, 295 / 207;  D 128, 4 183 / 148, 212 / 280, 327 / 536, 8
    190 / 152, 274 / 284, 506 / 541, 16 249 / 156, 453 / 288;  D 16, 8 102 / 70, 129 / 127, 191 / 241, 32 110 / 74, 170 / 136,
    312 / 252."""
    longest = max(b - a for a, b in zip(seg.row0_host[:-1], seg.row0_host[1:]))
    if longest < (2048 if D < 32 else 1024 if D <= 64 else 1792):
        return False
    groups = H * -(-V // 64) * (seg.row0_host[-1] / longest)     # short sequences beside it count by their tokens
    return groups <= (1024 // D if D >= 32 else 16)


def _mat_tiles(seg: SegMeta, kind: int, H: int, D: int, V: int):
    """(tiles, first tile of every segment, floats of workspace) for the matrix-core form of the delta rule (``kind`` 0) or
    the matrix memory (1), or None: no portion is long enough, or no form for ``D``.  Where the line lies (16 heads, D 64,
    V 128; token by token or in chunks -> tiles, us):  delta rule, one sequence of 16 / 17 / 129 tokens 21 -> 21 / 23 -> 19 /
    165 -> 29, 64 of 17 tokens 72 -> 52;  memory, one of 17 / 33 / 129 tokens 23 -> 27 / 30 -> 28 / 73 -> 29, 64 of 17 tokens
    68 -> 48 -- its own steps are cheaper, so that few sequences need two tiles before the tiles' launch pays, and long ones of
    few heads go in chunks (:func:`_long_and_few`)."""
    if kind == 1 and _long_and_few(seg, H, D, V):
        return None
    per = lib().k8s_tile_state_ws(kind, D)      # floats per (tile, head)
    few = seg.n_seg * H * -(-V // 64) < MAT_FILL_GROUPS
    cr = seg.chunk_ranges(MAT_TILE, 2 * MAT_TILE if kind == 1 and few else MAT_TILE) if per else None
    return None if cr is None else (*cr, cr[0].shape[0] * H * per + 256)


UNIT_EPS = 1e-6     # q and k of the delta rule: x / sqrt(sum(x^2) + UNIT_EPS)


MAT_SCRATCH = 1 << 28   # floats of the tiles' workspace (1 GiB): a step of more goes in several ones


def _mat_pieces(seg: SegMeta, tiles: int, floats: int) -> list:
    """A step whose ``tiles`` take ``floats`` of workspace as several steps, cut at tile borders: [(first row, end, SegMeta)].
    A sequence that is cut goes on from its slot, as it does from one portion of a prompt to the next."""
    dev, out = seg.row_seg.device, []
    most = max(2, MAT_SCRATCH * tiles // floats)
    todo = [(s, a, b) for s, (a, b) in enumerate(zip(seg.row0_host[:-1], seg.row0_host[1:])) if b > a]
    while todo:
        take, left = [], most
        while todo and left and not (take and take[-1][0] == todo[0][0]):
            s, a, b = todo.pop(0)
            n = min(b - a, left * MAT_TILE)
            take.append((s, a, a + n))
            left -= -(-n // MAT_TILE)
            if a + n < b:
                todo.insert(0, (s, a + n, b))
        r0 = [0]
        for _, a, b in take:
            r0.append(r0[-1] + b - a)
        pos = [seg.pos0_host[s] + a - seg.row0_host[s] for s, a, _ in take]
        slots = [seg.slot_host[s] for s, _, _ in take]
        i32 = [torch.tensor(v, dtype=torch.int32, device=dev)
               for v in ([i for i, (_, a, b) in enumerate(take) for _ in range(a, b)], r0, pos, slots, [[0]] * len(take))]
        out.append((take[0][1], take[-1][2], SegMeta(len(take), *i32, r0, pos, slots)))
    return out


def gated_delta(qkv: torch.Tensor, H: int, G: int, D: int, V: int, a: torch.Tensor, rate: torch.Tensor,
                dt_bias: torch.Tensor, beta: torch.Tensor, state: torch.Tensor, seg: SegMeta) -> torch.Tensor:
    """Gated delta rule per head, fp32.  Rows of ``qkv`` [T, 2 G D + H V] = (q | k | v) activations; head h
    reads q / k head ``h // (H // G)``; q and k become unit vectors (``UNIT_EPS``), q times ``D^(-1/2)``.
    Decay per head and key channel ``g = exp(-rate_h softplus(a + dt_bias))`` from ``a`` [T, H D] fp32;
    ``beta`` [T, >= H] fp32 before its sigmoid (row stride free).  Per token
    ``S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q`` with ``S`` [D, V].
    ``state`` [slots, H, D, V] fp32 is read (past position 0) and advanced.  Returns o [T, H V] fp32."""
    T = qkv.shape[0]
    out = torch.empty(T, H * V, dtype=torch.float32, device=qkv.device)
    if use_hip(qkv):
        assert qkv.is_contiguous() and qkv.shape[1] == 2 * G * D + H * V and H % G == 0
        assert a.dtype == torch.float32 and a.is_contiguous() and a.shape == (T, H * D)
        assert beta.dtype == torch.float32 and beta.stride(1) == 1 and beta.shape[1] >= H
        assert rate.dtype == dt_bias.dtype == torch.float32 and rate.numel() == H and dt_bias.numel() == H * D
        assert state.is_contiguous() and state.shape[1:] == (H, D, V)
        got = _mat_tiles(seg, 0, H, D, V)
        if got is not None:
            tiles, t0, n = got
            if n > MAT_SCRATCH and tiles.shape[0] > 2:
                return torch.cat([gated_delta(qkv[i:j], H, G, D, V, a[i:j], rate, dt_bias, beta[i:j], state, m)
                                  for i, j, m in _mat_pieces(seg, tiles.shape[0], n)])
            ws = scratch(n, torch.float32, qkv.device)
            check(lib().k8s_gated_delta_tiles(ptr(qkv), _dt(qkv.dtype), ptr(a), ptr(rate), ptr(dt_bias), ptr(beta),
                                              beta.stride(0), ptr(state), ptr(seg.seg_row0), ptr(seg.seg_pos0),
                                              ptr(seg.seg_slot), ptr(out),
                                              seg.n_seg, H, G, D, V, float(UNIT_EPS), stream_ptr(qkv), ptr(tiles),
                                              tiles.shape[0], ptr(t0), ptr(ws)),
                  "gated_delta_tiles")
            return out
        # other sizes, long portions: chunks in parallel (end states and step-matrix products from zero / identity, a
        # carry over the chunks, the chunks again from their start states); short ones token by token
        cr = _mat_chunks(seg, H, V)
        chunks, c0, cs, cx, nch = None, None, None, None, 0
        if cr is not None:
            chunks, c0 = cr
            nch = chunks.shape[0]
            cs = scratch(nch * H * D * V, torch.float32, qkv.device)
            cx = scratch(nch * H * D * D, torch.float32, qkv.device)
        check(lib().k8s_gated_delta(ptr(qkv), _dt(qkv.dtype), ptr(a), ptr(rate), ptr(dt_bias), ptr(beta),
                                    beta.stride(0), ptr(state), ptr(seg.seg_row0), ptr(seg.seg_pos0),
                                    ptr(seg.seg_slot), ptr(out), seg.n_seg, T, H, G, D, V, float(UNIT_EPS),
                                    stream_ptr(qkv), ptr(chunks), nch, ptr(c0), ptr(cs), ptr(cx)), "gated_delta")
        return out
    x = qkv.float()
    q = x[:, :G * D].view(T, G, D)
    k = x[:, G * D:2 * G * D].view(T, G, D)
    v = x[:, 2 * G * D:].view(T, H, V)
    q = q * torch.rsqrt(q.pow(2).sum(-1, keepdim=True) + UNIT_EPS) * D ** -0.5
    k = k * torch.rsqrt(k.pow(2).sum(-1, keepdim=True) + UNIT_EPS)
    rep = H // G
    q, k = q.repeat_interleave(rep, 1), k.repeat_interleave(rep, 1)      # [T, H, D]
    g = torch.exp(-rate.view(1, H, 1) * torch.nn.functional.softplus(a + dt_bias.view(1, -1)).view(T, H, D))
    bt = torch.sigmoid(beta[:, :H])
    for s in range(seg.n_seg):
        r0, r1, p0, sl = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s], seg.slot_host[s]
        S = state[sl].clone() if p0 > 0 else torch.zeros(H, D, V)
        for r in range(r0, r1):
            S = g[r][:, :, None] * S
            u = bt[r][:, None] * (v[r] - torch.einsum("hdv,hd->hv", S, k[r]))
            S = S + k[r][:, :, None] * u[:, None, :]
            out[r] = torch.einsum("hdv,hd->hv", S, q[r]).reshape(-1)
        state[sl] = S
    return out


DEN_EPS = 1e-6      # matrix memory: o = S^T q / (max(|n.q|, exp(-m)) + DEN_EPS)


def matrix_memory(x: torch.Tensor, H: int, D: int, V: int, gate_bias: torch.Tensor, cap: float,
                  state: torch.Tensor, nstate: torch.Tensor, mstate: torch.Tensor, seg: SegMeta,
                  defer_scale: bool = False):
    """Matrix memory with exponential gates per head, fp32.  Rows of ``x`` [T, 2 H D + 2 H V + 2 H] fp32 =
    (q | k | v | . | i | f): q is scaled by ``D^(-1/2)``; the log gates are ``i = cap tanh((i + b_i) / cap)`` and
    ``f = logsigmoid(cap tanh((f + b_f) / cap))`` with ``gate_bias`` [2 H] = (b_i | b_f).  With the running maximum
    ``m`` (0 at the start of a sequence):  ``m' = max(f + m, i)``;  ``S <- e^(f + m - m') S + e^(i - m') k v^T``;  n likewise
    with k alone;  ``o = S^T q / (max(|n.q|, e^(-m')) + DEN_EPS)``.  ``state`` [slots, H, D, V], ``nstate`` [slots, H, D],
    ``mstate`` [slots, H] fp32 are read (past position 0) and advanced.  Returns o [T, H V] fp32; with
    ``defer_scale`` (o', mul) with ``o = o' * mul[:, :, None]``, ``mul`` [T, H], for :func:`head_norm_gate` to apply."""
    T = x.shape[0]
    out = torch.empty(T, H * V, dtype=torch.float32, device=x.device)
    if use_hip(x):
        assert x.dtype == torch.float32 and x.stride(1) == 1 and x.shape[1] == 2 * H * (D + V) + 2 * H
        assert gate_bias.dtype == torch.float32 and gate_bias.numel() == 2 * H
        assert state.is_contiguous() and state.shape[1:] == (H, D, V) and nstate.is_contiguous()
        assert nstate.shape[1:] == (H, D) and mstate.is_contiguous() and mstate.shape[1:] == (H,)
        got = _mat_tiles(seg, 1, H, D, V)
        if got is not None and got[2] > MAT_SCRATCH and got[0].shape[0] > 2:
            parts = [matrix_memory(x[i:j], H, D, V, gate_bias, cap, state, nstate, mstate, m, defer_scale)
                     for i, j, m in _mat_pieces(seg, got[0].shape[0], got[2])]
            return tuple(torch.cat(t) for t in zip(*parts)) if defer_scale else torch.cat(parts)
        ab = scratch(T * H * 3, torch.float32, x.device)
        nq = scratch(T * H, torch.float32, x.device)
        mul = scratch((T, H), torch.float32, x.device)
        # other sizes, long portions: chunks in parallel (end states from zero, a carry over the chunks, the chunks again
        # from their start states); short ones token by token
        cr = _mat_chunks(seg, H, V) if got is None else None
        chunks, c0, cs, cx, cdec, nch, tws = None, None, None, None, None, 0, None
        if got is not None:
            chunks, c0, n = got
            nch, tws = chunks.shape[0], scratch(n, torch.float32, x.device)
        elif cr is not None:
            chunks, c0 = cr
            nch = chunks.shape[0]
            cs = scratch(nch * H * D * V, torch.float32, x.device)
            cx = scratch(nch * H * D, torch.float32, x.device)
            cdec = scratch(nch * H, torch.float32, x.device)
        check(lib().k8s_matrix_memory(ptr(x), x.stride(0), ptr(gate_bias), float(cap), ptr(state), ptr(nstate),
                                      ptr(mstate), ptr(seg.seg_row0), ptr(seg.seg_pos0), ptr(seg.seg_slot), ptr(ab),
                                      ptr(nq), ptr(mul), ptr(out), seg.n_seg, T, H, D, V, float(DEN_EPS),
                                      0 if defer_scale else 1, stream_ptr(x), ptr(chunks), nch, ptr(c0), ptr(cs),
                                      ptr(cx), ptr(cdec), ptr(tws)), "matrix_memory")
        return (out, mul) if defer_scale else out
    HD, HV = H * D, H * V
    q = x[:, :HD].view(T, H, D) * D ** -0.5
    k = x[:, HD:2 * HD].view(T, H, D)
    v = x[:, 2 * HD:2 * HD + HV].view(T, H, V)
    gi = x[:, 2 * HD + 2 * HV:2 * HD + 2 * HV + H] + gate_bias[:H]
    gf = x[:, 2 * HD + 2 * HV + H:] + gate_bias[H:]
    gi = cap * torch.tanh(gi / cap)
    gf = torch.nn.functional.logsigmoid(cap * torch.tanh(gf / cap))
    for s in range(seg.n_seg):
        r0, r1, p0, sl = seg.row0_host[s], seg.row0_host[s + 1], seg.pos0_host[s], seg.slot_host[s]
        if p0 > 0:
            S, n, m = state[sl].clone(), nstate[sl].clone(), mstate[sl].clone()
        else:
            S, n, m = torch.zeros(H, D, V), torch.zeros(H, D), torch.zeros(H)
        for r in range(r0, r1):
            mn = torch.maximum(gf[r] + m, gi[r])
            fa, ia = torch.exp(gf[r] + m - mn), torch.exp(gi[r] - mn)
            S = fa[:, None, None] * S + ia[:, None, None] * k[r][:, :, None] * v[r][:, None, :]
            n = fa[:, None] * n + ia[:, None] * k[r]
            m = mn
            den = torch.maximum((n * q[r]).sum(-1).abs(), torch.exp(-m)) + DEN_EPS
            out[r] = (torch.einsum("hdv,hd->hv", S, q[r]) / den[:, None]).reshape(-1)
        state[sl], nstate[sl], mstate[sl] = S, n, m
    return (out, None) if defer_scale else out


# ------------------------------------------------------------------ one token per sequence through a matrix state
# (csrc/kernels/state_step.hip): the state update with its gates, norm and output gate in one launch.  us, token-by-token
# kernel with its gate and norm passes / this, 16 heads of 128 x 128 at 1 / 8 / 64 / 256 sequences: delta rule 14.1 / 7.1,
# 16.6 / 7.3, 49.5 / 27.2, 181 / 111;  matrix memory 17.0 / 7.3, 20.7 / 6.7, 54.4 / 30.3, 181 / 109;  decaying attention
# 9.4 / 5.8, 11.0 / 6.0, 40.1 / 28.4, 142 / 107.  The states' bytes, in and out, take 0.4, 3.4, 27 and 109
# at the rate of a large copy; of 268 MB the caches hold a part from one call to the next.
def _step_ok(x: torch.Tensor, seg: SegMeta, D: int, V: int, state: torch.Tensor, gate: torch.Tensor,
             w: Optional[torch.Tensor]) -> bool:
    """Whether a step is one token each and rows, states, gates and weights can be read by 16 bytes."""
    return (use_hip(x) and seg.n_seg == x.shape[0] and seg.row0_host[-1] == seg.n_seg and D in (64, 128) and V in (64, 128)
            and min((b - a for a, b in zip(seg.row0_host[:-1], seg.row0_host[1:])), default=0) == 1
            and x.stride(1) == 1 and x.stride(0) % 4 == 0 and x.data_ptr() % 16 == 0 and state.data_ptr() % 16 == 0
            and gate.stride(1) == 1 and gate.stride(0) % 4 == 0 and gate.data_ptr() % 16 == 0
            and (w is None or (w.dtype == torch.float32 and w.is_contiguous() and w.data_ptr() % 16 == 0)))


DELTA_LOW_RANK, DELTA_LOW_HEAD, DELTA_LOW_ALL = 128, 24576, 6 << 20     # ranks; entries of a head's weights; of all that is read


def delta_layer(qkv: torch.Tensor, H: int, G: int, D: int, V: int, a: torch.Tensor, rate: torch.Tensor,
                dt_bias: torch.Tensor, beta: torch.Tensor, state: torch.Tensor, seg: SegMeta, gate: torch.Tensor,
                w: Optional[torch.Tensor], eps: float, out_dtype) -> torch.Tensor:
    """:func:`gated_delta`, then :func:`head_norm_gate` over each head."""
    if (_step_ok(qkv, seg, D, V, state, gate, w) and gate.dtype == torch.float32 and out_dtype == qkv.dtype
            and qkv.is_contiguous()):
        T = qkv.shape[0]
        assert qkv.shape[1] == 2 * G * D + H * V and H % G == 0 and state.is_contiguous() and state.shape[1:] == (H, D, V)
        assert a.dtype == torch.float32 and a.is_contiguous() and a.shape == (T, H * D)
        assert beta.dtype == torch.float32 and beta.stride(1) == 1 and beta.shape[1] >= H and gate.shape[1] >= H * V
        assert rate.dtype == dt_bias.dtype == torch.float32 and rate.numel() == H and dt_bias.numel() == H * D
        assert w is None or w.numel() in (V, H * V)
        out = torch.empty(T, H * V, dtype=out_dtype, device=qkv.device)
        check(lib().k8s_delta_step(ptr(qkv), _dt(qkv.dtype), ptr(a), ptr(rate), ptr(dt_bias), ptr(beta), beta.stride(0),
                                   ptr(state), ptr(seg.seg_pos0), ptr(seg.seg_slot), ptr(gate), gate.stride(0), ptr(w),
                                   V if w is not None and w.numel() == H * V else 0, ptr(out), T, H, G, D, V, float(eps),
                                   float(UNIT_EPS), stream_ptr(qkv)), "delta_step")
        return out
    o = gated_delta(qkv, H, G, D, V, a, rate, dt_bias, beta, state, seg)
    return head_norm_gate(o, gate, w, H, V, eps, out_dtype)


def delta_low_rank(qkv: torch.Tensor, H: int, G: int, D: int, V: int, lr: torch.Tensor, wa: torch.Tensor, wg: torch.Tensor,
                   rate: torch.Tensor, dt_bias: torch.Tensor, state: torch.Tensor, seg: SegMeta, w: Optional[torch.Tensor],
                   eps: float, out_dtype) -> torch.Tensor:
    """:func:`delta_layer` with decays' and output gates as products of low rank: ``lr`` [T, ra + rg + H] fp32 holds their inputs
    and beta's (:func:`low_rank_pair`, ``wa`` [H D, ra], ``wg`` [H V, rg]).

    Of single tokens the state's kernel makes them itself, every workgroup (a head of one token) with its own head's weights.
    us of two launches / one, H, D, V, both ranks:  16, 64, 128, 64, 64 at 1, 5, 32, 64 tokens 7.4 / 6.4, 8.9 / 7.5, 13.3 / 11.9,
    18.9 / 23.3;  4, 64, 64, 32, 32 at 1, 64 7.0 / 5.4, 9.0 / 6.8;  64, 64, 128, 128, 128 at 1, 3, 5, 16 9.1 / 8.9, 10.5 / 9.8,
    12.8 / 13.1, 21.7 / 27.6;  32, 128, 128, 64, 128 at 5, 16, 32 12.8 / 11.0, 20.4 / 19.8, 42.1 / 43.4: the line is what all of
    them read.  And past 48 KB a head one token waits for them: 16, 128, 128, 128, 128 at 1, 3, 8 8.5 / 8.9, 10.1 / 10.4,
    12.3 / 11.4."""
    ra, rg, T = wa.shape[1], wg.shape[1], qkv.shape[0]
    mine = wa.shape[0] // H * ra + wg.shape[0] // H * rg
    if (0 < T * H * mine <= DELTA_LOW_ALL and mine <= DELTA_LOW_HEAD and qkv.dtype == torch.bfloat16 == out_dtype
            and _small_rows(qkv, wa) and _small_rows(qkv, wg)
            and all(32 <= k <= DELTA_LOW_RANK and k % 32 == 0 and t.data_ptr() % 16 == 0 for k, t in ((ra, wa), (rg, wg)))
            and _step_ok(qkv, seg, D, V, state, qkv, w) and qkv.is_contiguous() and lr.dtype == torch.float32
            and lr.stride(1) == 1 and lr.shape == (T, ra + rg + H)):
        assert qkv.shape[1] == 2 * G * D + H * V and H % G == 0 and state.is_contiguous() and state.shape[1:] == (H, D, V)
        assert wa.shape[0] == H * D and wg.shape[0] == H * V and (w is None or w.numel() in (V, H * V))
        assert rate.dtype == dt_bias.dtype == torch.float32 and rate.numel() == H and dt_bias.numel() == H * D
        out = torch.empty(T, H * V, dtype=out_dtype, device=qkv.device)
        check(lib().k8s_delta_step_low(ptr(qkv), ptr(lr), lr.stride(0), ra, rg, ptr(wa), ptr(wg), ptr(rate), ptr(dt_bias),
                                       ptr(state), ptr(seg.seg_pos0), ptr(seg.seg_slot), ptr(w),
                                       V if w is not None and w.numel() == H * V else 0, ptr(out), T, H, G, D, V, float(eps),
                                       float(UNIT_EPS), stream_ptr(qkv)), "delta_step_low")
        return out
    # [T, H D] before bias and softplus, [T, H V] before the sigmoid, both fp32
    dec, gate = low_rank_pair(lr, 0, wa, ra, wg, out_dtype)
    return delta_layer(qkv, H, G, D, V, dec, rate, dt_bias, lr[:, ra + rg:], state, seg, gate, w, eps, out_dtype)


class _MemoryStep:
    """What a launch of one token per sequence through the matrix memory takes, and its result."""

    def __init__(self, x, H, D, V, gate_bias, cap, state, nstate, mstate, seg, w, eps, out_dtype, gate):
        assert x.dtype == torch.float32 and x.shape[1] == 2 * H * (D + V) + 2 * H
        assert gate_bias.dtype == torch.float32 and gate_bias.numel() == 2 * H and (w is None or w.numel() in (V, H * V))
        assert state.is_contiguous() and state.shape[1:] == (H, D, V) and nstate.is_contiguous()
        assert nstate.shape[1:] == (H, D) and mstate.is_contiguous() and mstate.shape[1:] == (H,)
        self.heads, self.dim, self.vdim = H, D, V
        self.done = False
        self.out = torch.empty(x.shape[0], H * V, dtype=out_dtype, device=x.device)
        self.args = (ptr(x), x.stride(0), ptr(gate_bias), float(cap), ptr(state), ptr(nstate), ptr(mstate), ptr(seg.seg_pos0),
                     ptr(seg.seg_slot), ptr(gate), gate.stride(0), ptr(w), V if w is not None and w.numel() == H * V else 0,
                     ptr(self.out), H, D, V, float(eps), float(DEN_EPS))

    def launch(self) -> torch.Tensor:
        """The result, by a launch of its own if no other has made it."""
        if not self.done:
            check(lib().k8s_memory_step(*self.args[:14], _dt(self.out.dtype), self.out.shape[0], *self.args[14:],
                                        stream_ptr(self.out)), "memory_step")
            self.done = True
        return self.out


def _memory_gate(x: torch.Tensor, H: int, D: int, V: int) -> torch.Tensor:
    return x[:, 2 * H * D + H * V:2 * H * (D + V)]


def _memory_step(x, H, D, V, gate_bias, cap, state, nstate, mstate, seg, w, eps, out_dtype) -> Optional[_MemoryStep]:
    gate = _memory_gate(x, H, D, V)
    if not _step_ok(x, seg, D, V, state, gate, w):
        return None
    return _MemoryStep(x, H, D, V, gate_bias, cap, state, nstate, mstate, seg, w, eps, out_dtype, gate)


def memory_layer(x: torch.Tensor, H: int, D: int, V: int, gate_bias: torch.Tensor, cap: float, state: torch.Tensor,
                 nstate: torch.Tensor, mstate: torch.Tensor, seg: SegMeta, w: Optional[torch.Tensor], eps: float,
                 out_dtype) -> torch.Tensor:
    """:func:`matrix_memory`, then :func:`head_norm_gate` over each head with the gates that stand behind the values."""
    step = _memory_step(x, H, D, V, gate_bias, cap, state, nstate, mstate, seg, w, eps, out_dtype)
    if step is not None:
        return step.launch()
    gate = _memory_gate(x, H, D, V)
    o, mul = matrix_memory(x, H, D, V, gate_bias, cap, state, nstate, mstate, seg, defer_scale=True)
    return head_norm_gate(o, gate, w, H, V, eps, out_dtype, mul=mul)


def decay_slices(T: int, H: int, V: int) -> int:
    """Workgroups of a head in :func:`decay_layer`'s steps of ``T`` single tokens: four of 32 columns while half of the compute
    units would have none.  A unit takes a state in and gives it back at some 48 to 68 KB a us (both counted, a launch's 2.6 us left
    out).  us with 1 / 2 / 4 of them, states no cache holds:  16 heads of 128 x 128 at 1, 4, 7, 16, 32 tokens 4.5 / 3.8 / 3.3, 4.9 / 4.2 /
    3.8, 5.3 / 4.7 / 4.7, 7.2 / 7.6 / 7.6, 13.4 / 15.0 / 15.2;  8 heads at 7, 16, 32 4.9 / 4.2 / 3.8, 5.4 / 4.8 / 5.1, 7.3 / 7.2 / 7.8;  16 of 64 x 128
    at 1, 7, 16 3.6 / 3.3 / 3.1, 4.0 / 3.8 / 3.9, 5.0 / 5.0 / 5.5."""
    return 4 if V == 128 and T * H <= 128 and 4 * H <= 64 else 1      # (64 sums of squares a row: what the products behind take)


def decay_layer(x: torch.Tensor, H: int, D: int, V: int, decay: torch.Tensor, state: torch.Tensor, seg: SegMeta,
                gate: torch.Tensor, w: torch.Tensor, eps: float, out_dtype) -> tuple:
    """:func:`decay_attention` with silu, then one norm over all heads, its weight and the gates: (y, None), or for steps of
    single tokens (y without the division by the row's root mean square, (sums of squares [T, .], H V, eps)), which
    :func:`.norm.hyper_step` makes up for behind the output projection."""
    if (_step_ok(x, seg, D, V, state, gate, w) and gate.dtype == x.dtype == out_dtype and w.numel() == H * V):
        T = x.shape[0]
        assert x.shape[1] >= H * (2 * D + V) and gate.shape[1] >= H * V
        assert decay.dtype == torch.float32 and decay.numel() == H
        assert state.is_contiguous() and state.dtype == torch.float32 and state.shape[1:] == (H, D, V)
        out = torch.empty(T, H * V, dtype=out_dtype, device=x.device)
        slices = decay_slices(T, H, V)
        ss = torch.empty(T, H * slices, dtype=torch.float32, device=x.device)
        check(lib().k8s_decay_step(ptr(x), x.stride(0), _dt(x.dtype), ptr(decay), ptr(state), ptr(seg.seg_pos0),
                                   ptr(seg.seg_slot), ptr(gate), gate.stride(0), ptr(w), ptr(out), ptr(ss), T, H, D, V,
                                   stream_ptr(x), slices), "decay_step")
        return out, (ss, H * V, eps)
    o = decay_attention(x, H, D, V, decay, state, seg, silu=True)
    return head_norm_gate(o, gate, w, 1, H * V, eps, out_dtype), None

