"""LLM engine, part 3 of 4: HIP-graph decode steps.

Pure-decode steps replay one captured graph per batch bucket; the decode work
list, its item count and the keys per item are read on the device, so one
graph serves every context mix.  Static input buffers are filled from one
pinned staging copy per replay.

Models in the segment layout that declare ``segment_graphs`` replay one graph
per (rows, block-table width): see :meth:`GraphRunnerMixin._seg_graph_step`.
"""
from __future__ import annotations

import contextlib
import json
import logging
import math
import os
import threading
import gc
import time
from typing import Callable, Dict, List, Optional, Sequence as Seq, Tuple

import numpy as np
import torch

from ..knobs import KNOBS
from ..ops import attention as A
from ..ops import sampling as SMP
from ..ops._lib import scratch
from ..ops.row_step import RowStep
from ..ops.seq_ops import SegMeta, SegStepInputs
from ..utils import tracing
from .structured import GrammarState
from .types import PART_MIN, SPEC, InFlight, Request, Sequence, _LazySample, _spec_tok

log = logging.getLogger("k8s_llm_rca_amd.engine.engine")


# A capture takes 1.1 to 1.4 ms in place of an eager step, a replay saves 0.4 to 0.5 ms (fikerax-1b, 1 / 7 / 64 rows: 1.14 /
# 1.20 / 1.85 ms of which the host's launches take most -> 0.71 / 0.88 / 1.38; lizesun-1b, 8 layers: 1.17 / 1.27 / 1.66 ->
# 0.77 / 0.87 / 1.10).  Generation of 64 replies, ms of an engine's second round, eager / captured whenever a shape had come
# three times / paid for by replays: a reply ends every second step 222 / 272 / 235 (8 captures, none in later rounds), every
# fourth 422 / 371 / 363; 24 replies of 4 to 200 tokens 255 / 164 / 164.
SEG_GRAPH_AFTER = 3     # eager steps of a shape before it is captured (they leave nothing to be set up inside the capture)
SEG_GRAPHS = 32         # graphs an engine keeps (least recently replayed ones go)
SEG_PRICE = 3           # replays that pay for a capture
SEG_AHEAD = 8           # captures an engine makes before replays have paid for them
SEG_LONG = 64           # eager steps of a shape after which it is captured on no account but its own
SEG_BACKOFF = 256       # steps of a shape between a capture that failed and the next try


class SegGraphCache:
    """Which shapes of steps have a graph, and which are worth one.  A batch that shrinks and grows runs through many shapes
    of a few steps each, so captures are paid for by replays: an engine is never more than ``SEG_AHEAD`` captures behind
    what eager steps alone would have taken, but for one per ``SEG_LONG`` eager steps of a shape.  A graph that gives way
    to others has to be earned again."""

    def __init__(self):
        self.graphs: Dict[tuple, tuple] = {}       # least recently replayed first
        self.seen: Dict[tuple, int] = {}           # eager steps of a shape without a graph
        self.credit = SEG_AHEAD * SEG_PRICE        # replays
        self.off = False                           # a capture could not be ended

    def get(self, key: tuple) -> Optional[tuple]:
        """The graph of a shape, for a replay."""
        got = self.graphs.pop(key, None)
        if got is not None:
            self.graphs[key] = got
            self.credit = min(self.credit + 1, SEG_GRAPHS * SEG_PRICE)
        return got

    def worth(self, key: tuple) -> bool:
        """Counts a step of a shape without a graph: whether to capture it."""
        if self.off:
            return False
        if len(self.seen) > 4096:
            self.seen.clear()
        n = self.seen[key] = self.seen.get(key, 0) + 1
        return n > SEG_GRAPH_AFTER and (self.credit >= SEG_PRICE or n > SEG_LONG)

    def room(self) -> bool:
        return len(self.graphs) < SEG_GRAPHS

    def put(self, key: tuple, graph: tuple) -> None:
        while not self.room():
            self.graphs.pop(next(iter(self.graphs)))
        self.graphs[key] = graph
        self.seen.pop(key, None)
        self.credit = max(0, self.credit - SEG_PRICE)

    def failed(self, key: tuple) -> None:
        self.seen[key] = -SEG_BACKOFF


class _DecodeSegments(SegMeta):
    """The segments of a step of single tokens whose work items lie in a captured graph's static input."""

    def attn_items(self, tokens_per_item: int) -> tuple:
        return self.items, self.items[:0], self.pos0_host[0] + 1

    def mask_items(self, tokens_per_item: int, by_rows: bool = False) -> tuple:
        return self.items, self.items[:0]

    def tile_items(self, tokens_per_item: int) -> torch.Tensor:
        return self.items


class GraphRunnerMixin:
    def _graphs_ok(self) -> bool:
        """Decode steps replay HIP graphs at TP=1, and under TP when every
        all-reduce of a decode step runs on the capturable xGMI kernel."""
        if self.pc.tp_size == 1:
            return True
        car = self.pc.custom_ar
        return car is not None and getattr(car, "max_bytes", 0) >= max(self.cfg.graph_batch_sizes) * self.mc.hidden * 2

    @staticmethod
    def _n_parts(max_ctx: int) -> int:
        """Partition count bound at the smallest partition size (buffer sizing)."""
        n = max(1, (max_ctx + PART_MIN - 1) // PART_MIN)
        return 1 << (n - 1).bit_length()

    # ---------------------------------------------------------- HIP graphs
    def _bucket(self, n: int) -> int:
        for b in self.cfg.graph_batch_sizes:
            if b >= n:
                return b
        return n

    def _ensure_static(self):
        if self._static is not None:
            return self._static
        Bmax = max(self.cfg.graph_batch_sizes)
        mb = self.max_blocks_per_seq
        npmax = self._n_parts(self.max_context)
        self._max_items = Bmax * npmax
        dev = self.device
        st = {
            "ids": torch.zeros(Bmax, dtype=torch.int32, device=dev),
            "pos": torch.zeros(Bmax, dtype=torch.int32, device=dev),
            "slots": torch.full((Bmax,), -1, dtype=torch.int32, device=dev),
            "bt": torch.zeros(Bmax, mb, dtype=torch.int32, device=dev),
            "ctx": torch.ones(Bmax, dtype=torch.int32, device=dev),
            "qs": torch.arange(Bmax + 1, dtype=torch.int32, device=dev),
            "sidx": torch.arange(Bmax, dtype=torch.int64, device=dev),
            "part_o": scratch(Bmax * self.model.nq * npmax * self.model.D, torch.float32, dev),
            "part_ml": scratch(Bmax * self.model.nq * npmax * 2, torch.float32, dev),
            "items": torch.zeros(Bmax * npmax, 4, dtype=torch.int32, device=dev),
            "n_items": torch.zeros(2, dtype=torch.int32, device=dev),  # {item count, keys per item}
            # two pinned staging buffers, alternated per graph step; each is
            # reused only after the event recorded behind its last H2D copy
            "host": [torch.zeros(Bmax * (3 + mb + 2) + 2 + Bmax * npmax * 4, dtype=torch.int32).pin_memory()
                     for _ in range(2)],
            "host_ev": [None, None],
            "host_i": 0,
        }
        self._static = st
        return st

    def _graph_inputs(self, B: int, part: int):
        from ..models.llama import StepInputs

        st = self._static
        # work-list decode: the grid is the resident-wave count and the item
        # count is read on the device, so one graph serves every item list
        meta = A.AttnMeta(block_tables=st["bt"][:B], ctx_lens=st["ctx"][:B], q_start=st["qs"][:B + 1], num_seqs=B,
                          decode=True, n_parts=self._n_parts(self.max_context), part_size=part,
                          part_o=st["part_o"], part_ml=st["part_ml"], items=st["items"], n_items=0,
                          d_n_items=st["n_items"], grid_waves=A.DECODE_WAVE_SLOTS)
        return StepInputs(st["ids"][:B], st["pos"][:B], st["slots"][:B], B, meta, None, st["sidx"][:B])

    def _capture(self, B: int, part: int):
        """Graph of a ``B``-row decode step.  ``part`` only seeds the capture:
        the decode kernels read each replay's keys-per-item from the device."""
        key = B
        g = self._graphs.get(key)
        if g is not None:
            return g
        t0 = time.perf_counter()
        inp = self._graph_inputs(B, part)
        s = torch.cuda.Stream(self.device)
        s.wait_stream(torch.cuda.current_stream(self.device))
        with torch.cuda.stream(s):
            for _ in range(2):
                self._model_fwd(inp)
        torch.cuda.current_stream(self.device).wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        if self._graph_pool is None:
            self._graph_pool = torch.cuda.graph_pool_handle()
        # thread_local: the graph-query batcher keeps issuing on its own stream from its
        # own thread while a bucket is captured mid-run
        # no cyclic collection while the stream captures: a collector run that happens to start inside the
        # capture would destroy graphs and free device memory of engines that are already gone, which a
        # capturing stream does not allow (torch.cuda.graph collects once, before the capture begins)
        gc_was_on = gc.isenabled()
        gc.disable()
        try:
            with torch.cuda.graph(graph, pool=self._graph_pool, capture_error_mode="thread_local"):
                out = self._model_fwd(inp)
        finally:
            if gc_was_on:
                gc.enable()
        self._graphs[key] = (graph, out)
        self.stats["captures"] += 1
        self.stats["capture_s"] += time.perf_counter() - t0
        return self._graphs[key]

    def _forward_graph(self, decode: List[Tuple[Sequence, int]], spec=None, sample_idx: Optional[List[int]] = None):
        """``decode``: decode-attention rows (sequence, token offset past
        n_cached); the logits of the ``sample_idx`` rows are returned (all rows
        when every row samples)."""
        st = self._ensure_static()
        B = len(decode)
        if sample_idx is None:
            sample_idx = list(range(B))
        Bb = self._bucket(B)
        if Bb > max(self.cfg.graph_batch_sizes):
            return self._forward_eager(decode, [], sample_idx, spec)
        BS = self.kv.block_size
        mb = self.max_blocks_per_seq
        ctx = np.ones(Bb, dtype=np.int32)
        ids = np.zeros(Bb, dtype=np.int32)
        pos = np.zeros(Bb, dtype=np.int32)
        slots = np.full(Bb, -1, dtype=np.int32)
        bt = np.zeros((Bb, mb), dtype=np.int32)
        for i, (s, j) in enumerate(decode):
            p = s.n_cached + j
            ids[i] = s.tokens[p]
            pos[i] = p
            slots[i] = s.blocks[p // BS] * BS + p % BS
            ctx[i] = p + 1
            bt[i, : len(s.blocks)] = s.blocks
        # plan on the real rows; padded rows (ctx 1) still get a one-key item
        # (sorted last) so every output row the graph produces is finite
        chain = self._decode_chain(decode)
        _, part = A.plan_decode_split(self._plan_ctx(ctx[:B], chain), self.model.nkv,
                                      max_parts=self._n_parts(self.max_context))
        if self.stats["graph_steps"] % 32 == 0:  # how often decode attention re-reads a shared KV block
            used = np.concatenate([s.blocks[: (s.n_cached + j + BS) // BS] for s, j in decode])
            self.stats["kv_read_blocks_sampled"] += used.size
            self.stats["kv_unique_blocks_sampled"] += np.unique(used).size
        if chain is not None:
            chain = np.concatenate([chain, np.zeros(Bb - B, dtype=bool)])
        items = A.build_decode_items(ctx, np.arange(Bb), part, chain, self._dec_gmax)
        n_items = items.shape[0]
        assert n_items <= self._max_items
        flat = np.concatenate([ids, pos, slots, ctx, bt.reshape(-1), np.array([n_items, part], np.int32),
                               items.reshape(-1).astype(np.int32)])
        sel = np.asarray(sample_idx if len(sample_idx) != B else [], dtype=np.int32)
        if self._chan is not None:
            from ..parallel.channel import FWD_GRAPH
            meta = np.array([B, Bb, part, n_items, mb], dtype=np.int32)
            self._chan.send(FWD_GRAPH, [meta, flat, sel] + ([spec[0]] if spec is not None else []))
        return self._graph_run(B, Bb, part, n_items, mb, flat, spec, sel)

    def _graph_run(self, B: int, Bb: int, part: int, n_items: int, mb: int, flat: np.ndarray, spec=None,
                   sel: Optional[np.ndarray] = None):
        """Upload a packed decode step into the static graph inputs (pinned
        staging, one async copy) and replay bucket ``Bb``'s graph (rank 0, and
        every TP worker from the channel's message).  ``spec`` = (src[B], tok):
        row i's input id is ``tok[src[i]]`` where ``src[i] >= 0``."""
        st = self._ensure_static()
        assert mb == self.max_blocks_per_seq
        if self._sim:
            self.sim_rows[Bb] = self.sim_rows.get(Bb, 0) + 1
        hi = st["host_i"] = st["host_i"] ^ 1
        if st["host_ev"][hi] is not None:
            st["host_ev"][hi].synchronize()  # its previous upload has long completed in practice
        host = st["host"][hi]
        hv = host.numpy()
        n = flat.size
        hv[:n] = flat
        if spec is not None:
            hv[n:n + B] = spec[0]
            n_src = n
            n += B
        n_sel = 0 if sel is None else sel.size
        if n_sel:  # rows that sample (tiny-chunk rows other than a chunk's last do not)
            hv[n:n + n_sel] = sel
            o_sel = n
            n += n_sel
        dev_flat = torch.empty(n, dtype=torch.int32, device=self.device)
        dev_flat.copy_(host[:n], non_blocking=True)
        self._trace_mark()
        ev = st["host_ev"][hi] = st["host_ev"][hi] or torch.cuda.Event(blocking=KNOBS.blocking_sync)
        ev.record()
        # the upload scattered into the graph's static inputs in one launch (csrc/kernels/norm_act.hip),
        # the speculative decode ids (spec) taken from the device tokens in the same launch; before a
        # capture too: its warm-up forwards read these ids
        from ..ops._lib import check, lib, stream_ptr
        tok = _spec_tok(spec) if spec is not None else None  # launches the previous step's sampling
        fused_spec = tok is not None and tok.dtype == torch.int32 and tok.is_contiguous()
        check(lib().k8s_unpack_step(dev_flat.data_ptr(), Bb, mb, n_items, st["ids"].data_ptr(), st["pos"].data_ptr(),
                                    st["slots"].data_ptr(), st["ctx"].data_ptr(), st["bt"].data_ptr(),
                                    st["n_items"].data_ptr(), st["items"].data_ptr(),
                                    dev_flat[n_src:].data_ptr() if fused_spec else None,
                                    tok.data_ptr() if fused_spec else None, B if fused_spec else 0,
                                    stream_ptr(dev_flat)), "unpack_step")
        if tok is not None and not fused_spec:
            self._apply_spec(st["ids"], dev_flat[n_src:n_src + B], tok)
        graph, out = self._capture(Bb, part)  # one graph per bucket: the plan's part size is read on the device
        graph.replay()
        if n_sel:
            return out.index_select(0, dev_flat[o_sel:o_sel + n_sel].long())
        return out[:B]

    # ------------------------------------------- HIP graphs of the segment layout
    def _seg_graph_step(self, decode: List[Tuple[Sequence, int]], sample_idx: List[int]) -> Optional[torch.Tensor]:
        """A step of one token each for ``decode``'s sequences as a graph replay; None: the step runs eagerly (several rows
        of one sequence, too many rows, or a shape that has not come often enough).  A graph fixes the number of rows
        and how many cache pages the attention's grids are laid out for (the width of the block tables: a power of two up to
        8 pages, then in steps of 8, past 128 of 32); everything else a step's kernels need -- tokens, positions, cache and state slots,
        pages, work items -- is read from one static buffer that each step fills with one copy.  The last product is a launch
        behind the graph, into memory of the step's own: what a step returns stays the caller's, without a copy of it (2 to 6 us
        of 350 to 500 with one to seven rows of 32000 columns).  A capture that fails -- it takes memory beside the allocator's
        free blocks -- has run nothing, so the step runs eagerly."""
        B, BS = len(decode), self.kv.block_size
        if B > max(self.cfg.graph_batch_sizes) or len(set(id(s) for s, _ in decode)) != B or KNOBS.sync_debug:
            return None                        # (a capture has no room for the synchronisation behind every launch)
        pages = max(s.n_cached + j for s, j in decode) // BS + 1
        width = 1 << (pages - 1).bit_length() if pages <= 8 else -(-pages // 8) * 8 if pages <= 128 else -(-pages // 32) * 32
        cache, key = self._seg, (B, width)
        if self._seg_loads != self.model.loads:       # other weights: no graph of the old ones is replayed any more
            if cache.graphs:
                torch.cuda.current_stream(self.device).synchronize()
                cache.graphs.clear()
            self._seg_loads = self.model.loads
        got = cache.get(key)
        if got is None and not cache.worth(key):
            return None
        flat = np.zeros(8 * B + B * width, dtype=np.int32)
        ids, pos, slots, slot = flat[:4 * B].reshape(4, B)
        items, bt = flat[4 * B:8 * B].reshape(B, 4), flat[8 * B:].reshape(B, width)
        for i, (s, j) in enumerate(decode):
            p = s.n_cached + j
            n = p // BS + 1
            ids[i], pos[i], slots[i] = s.tokens[p], p, s.blocks[n - 1] * BS + p % BS
            if self.states is not None:
                if s.slot is None:
                    raise RuntimeError(f"sequence {s.id} runs without a state slot")
                slot[i] = s.slot
            items[i] = i, i, 1, p
            bt[i, :n] = s.blocks[:n]
        host = torch.from_numpy(flat).pin_memory()
        if got is None:
            if not cache.room():
                torch.cuda.current_stream(self.device).synchronize()       # the last replay of the one that goes may still run
            try:
                got = self._seg_capture(B, width, host)
            except Exception as e:                 # (what is wrong with the step itself shows again in the eager one)
                log.warning("capture of a step of %d rows failed, the step runs eagerly: %s", B, e)
                cache.failed(key)
                return None
            cache.put(key, got)
        else:
            got[1].copy_(host, non_blocking=True)
        self._trace_mark()
        graph, _, h, whole, _ = got
        graph.replay()
        out = h.clone() if whole else self.model.logits(h)
        if sample_idx == list(range(B)):
            return out
        return out.index_select(0, torch.tensor(sample_idx, dtype=torch.long).pin_memory().to(self.device,
                                                                                              non_blocking=True))

    def _seg_capture(self, B: int, width: int, host: torch.Tensor) -> tuple:
        """(graph, its static input holding ``host``, what the model makes logits of -- or, where their product cannot be made
        again and again, the logits [B, vocab] themselves and True --, its step) of a step of ``B`` single tokens.  The step is
        kept with the graph: every tensor in it is read by each replay, the row offsets too, which no copy fills."""
        t0 = time.perf_counter()
        cur = torch.cuda.current_stream(self.device)
        flat = host.to(self.device, non_blocking=True)
        ids, pos, slots, slot = flat[:4 * B].view(4, B).unbind(0)
        rows = torch.arange(B + 1, dtype=torch.int32, device=self.device)
        seg = _DecodeSegments(n_seg=B, row_seg=rows[:B], seg_row0=rows, seg_pos0=pos, seg_slot=slot,
                              block_tables=flat[8 * B:].view(B, width), row0_host=list(range(B + 1)),
                              pos0_host=[width * self.kv.block_size - 1] * B, slot_host=[0] * B, n_single=B)
        seg.items = flat[4 * B:8 * B].view(B, 4)
        inp = SegStepInputs(ids, pos, slots, seg, None)
        states = self.states.t if self.states is not None else {}
        if not self._seg.graphs:                   # (a pool goes with the last graph that holds it)
            self._seg_pool = torch.cuda.graph_pool_handle()
        if self._seg_stream is None:
            self._seg_stream = torch.cuda.Stream(self.device)
        graph = torch.cuda.CUDAGraph()
        # (not torch.cuda.graph: it gives the allocator's free blocks back to the device, which the next prompt then
        # has to take anew; no cyclic collection while the stream captures, as in _capture)
        gc_was_on = gc.isenabled()
        gc.disable()
        self._seg_stream.wait_stream(cur)
        try:
            with torch.cuda.stream(self._seg_stream):
                graph.capture_begin(pool=self._seg_pool, capture_error_mode="thread_local")
                try:
                    out = self.model.forward(inp, *self.kv.tensors(), states, head=False)
                    whole = isinstance(out, RowStep)
                    if whole:
                        out = self.model.logits(out)
                except BaseException:
                    self._seg.off = True           # until the capture has ended
                    with contextlib.suppress(RuntimeError):        # (the first error is the one to report)
                        graph.capture_end()
                        self._seg.off = False
                    raise
                self._seg.off = True
                graph.capture_end()
                self._seg.off = False
        finally:
            if gc_was_on:
                gc.enable()
        cur.wait_stream(self._seg_stream)
        self.stats["captures"] += 1
        self.stats["capture_s"] += time.perf_counter() - t0
        return graph, flat, out, whole, inp
