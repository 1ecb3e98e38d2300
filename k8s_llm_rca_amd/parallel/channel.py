"""Host-side step channel from the TP leader (rank 0) to the TP workers.

Under tensor parallelism every rank runs the same forward (its shard of every
layer; two all-reduces per layer), but only rank 0 owns the scheduler.  The
step metadata -- token ids, positions, KV slots, block tables, the attention
work plan, sampling inputs -- therefore travels from rank 0 to the workers
every step.  Sending it as device tensors over RCCL made each worker block on
a ``.cpu()`` of the header to size the next receive (a full GPU sync per
step).  This channel moves the metadata between HOST memories
(gloo over loopback on one node): a worker receives step k+1's inputs while
its GPU is still executing step k, uploads them with a pinned async copy and
issues the forward -- the GPUs synchronise only inside the forward, at the
all-reduces, as the TP math requires.

A message is a kind plus a list of int32 / int64 / float32 numpy arrays
(float32 travels bit-cast as int32).  Two gloo broadcasts per message: a
fixed 16-int header (kind, array count, per-array length and dtype code), then
one flat int32 payload.
"""
from __future__ import annotations

from typing import List, Optional, Tuple

import numpy as np
import torch
import torch.distributed as dist

MAX_ARRAYS = 7
_DT = {0: np.int32, 1: np.int64, 2: np.float32}
_CODE = {np.dtype(np.int32): 0, np.dtype(np.int64): 1, np.dtype(np.float32): 2}

STOP, FWD_EAGER, FWD_GRAPH, SAMPLE = 0, 1, 2, 3


class StepChannel:
    def __init__(self, group, src_global_rank: int = 0):
        self.group = group
        self.src = src_global_rank
        self.sent = 0
        self.bytes = 0

    def send(self, kind: int, arrays: List[np.ndarray]) -> None:
        assert len(arrays) <= MAX_ARRAYS
        hdr = np.zeros(16, dtype=np.int32)
        hdr[0], hdr[1] = kind, len(arrays)
        parts = []
        for i, a in enumerate(arrays):
            a = np.ascontiguousarray(a)
            code = _CODE[a.dtype]
            flat = a.reshape(-1).view(np.int32)
            hdr[2 + 2 * i], hdr[3 + 2 * i] = flat.size, code
            parts.append(flat)
        payload = np.concatenate(parts) if parts else np.zeros(0, np.int32)
        dist.broadcast(torch.from_numpy(hdr), src=self.src, group=self.group)
        if payload.size:
            dist.broadcast(torch.from_numpy(payload), src=self.src, group=self.group)
        self.sent += 1
        self.bytes += 64 + 4 * payload.size

    def recv(self) -> Tuple[int, List[np.ndarray]]:
        hdr = torch.zeros(16, dtype=torch.int32)
        dist.broadcast(hdr, src=self.src, group=self.group)
        h = hdr.numpy()
        kind, n = int(h[0]), int(h[1])
        sizes = [int(h[2 + 2 * i]) for i in range(n)]
        total = sum(sizes)
        payload = torch.zeros(total, dtype=torch.int32)
        if total:
            dist.broadcast(payload, src=self.src, group=self.group)
        flat = payload.numpy()
        out, o = [], 0
        for i, sz in enumerate(sizes):
            out.append(flat[o:o + sz].view(_DT[int(h[3 + 2 * i])]))
            o += sz
        return kind, out


def make_channel(pc) -> Optional[StepChannel]:
    """A gloo channel over ``pc.tp_group``'s ranks (collective: every TP rank
    calls this at engine init, in the same order)."""
    if pc.tp_size <= 1:
        return None
    ranks = dist.get_process_group_ranks(pc.tp_group) if pc.tp_group is not None else list(range(pc.tp_size))
    if dist.get_backend(pc.tp_group) == "gloo":
        g = pc.tp_group
    else:
        g = dist.new_group(ranks=ranks, backend="gloo")
    return StepChannel(g, ranks[0])
