"""HIP-graph replay of the whole per-micro-batch forward (resident weights).

The reference dispatches every op of every layer from Python, one prompt at a
time (``/root/reference/utils.py:239-291``).  With small batches (a few short
prompts, or the ``--num_gen_token`` loop that re-runs the full model once per
generated token, ``main.py:65-90``) the GPU work per layer is a few tens of
microseconds and host-side dispatch dominates.

When every shard of this rank is resident in HBM the weight pointers never
change, so embed -> all decoder layers -> final norm -> LM head + softmax of one
micro-batch is captured ONCE as a HIP graph (``torch.cuda.CUDAGraph`` is
hipGraph on ROCm) and replayed with a single launch.  Batch shapes are
bucketed so replays are reused across calls and generation steps:

* tokens -> multiple of ``TOKEN_BUCKET`` (the GEMM M tile; padded rows compute
  garbage that no valid row ever reads: GEMM / RMSNorm rows are independent and
  no attention work item covers them),
* attention work items -> multiple of ``WORK_BUCKET`` (padding items have
  ``q_len = 0``; the kernels return before touching memory),
* scored rows -> multiple of ``SCORE_BUCKET`` (padding gathers row 0; ignored; the
  last decoder layer's single-query work items are padded with ``q_len = 0``).

The metadata of a new batch is copied into the graph's static input tensors
before the replay; the probabilities come out of its static output tensor.
All graphs share one memory pool and are replayed in order on one stream, so
intermediates are shared between them.
"""
from __future__ import annotations

import contextlib
import gc
import threading
from collections import OrderedDict
from typing import Callable, Dict, List, Optional, Tuple

import numpy as np
import torch

from .batch import WORK_ITEM_FIELDS, PackedBatch
from .hostmem import alloc_host

TOKEN_BUCKET = 256
WORK_BUCKET = 32
SCORE_BUCKET = 16


def _ceil(n: int, m: int) -> int:
    return max(m, (n + m - 1) // m * m)


def bucket_key(batch: PackedBatch) -> Tuple[int, int, int]:
    return (_ceil(batch.num_tokens, TOKEN_BUCKET), _ceil(batch.work.shape[0], WORK_BUCKET),
            _ceil(batch.n_scored, SCORE_BUCKET))


def padded_meta(batch: PackedBatch, key) -> Dict[str, np.ndarray]:
    T, W, S = key
    ids = np.zeros(T, np.int32)
    ids[:batch.num_tokens] = batch.ids
    pos = np.zeros(T, np.int32)
    pos[:batch.num_tokens] = batch.positions
    work = np.zeros((W, WORK_ITEM_FIELDS), np.int32)
    work[:batch.work.shape[0]] = batch.work
    seg_lo = np.zeros(T, np.int32)                         # padding rows: never a query of any item
    seg_lo[:batch.num_tokens] = batch.seg_lo
    last = np.zeros(S, np.int32)
    last[:batch.n_scored] = batch.last_idx
    last_pos = pos[last]                                   # positions of the scored rows
    wl = np.zeros((S, WORK_ITEM_FIELDS), np.int32)        # padding items: q_len 0
    wl[:batch.work_last.shape[0]] = batch.work_last
    return {"ids": ids, "positions": pos, "work": work, "seg_lo": seg_lo, "last_idx": last, "last_pos": last_pos,
            "work_last": wl}


class _Arrays:
    """int32 arrays of one step back to back in one buffer, each from a 64-byte boundary behind ``head`` entries."""

    def __init__(self, host: Dict[str, np.ndarray], head: int = 0):
        self.shapes = {k: v.shape for k, v in host.items()}
        self.at, n = {}, head
        for k, v in host.items():
            self.at[k] = n
            n += _ceil(v.size, 16)
        self.size = n

    def views(self, flat) -> dict:
        """The arrays in ``flat`` (a tensor or an array) by name."""
        out = {}
        for k, shape in self.shapes.items():
            part = flat[self.at[k]:self.at[k] + int(np.prod(shape, dtype=np.int64))]
            out[k] = part.reshape(shape) if isinstance(flat, np.ndarray) else part.view(shape)
        return out


class _CollectorHeld:
    """Python's automatic collections off while any thread is in the context; when the last one leaves they are as the first one found them."""

    def __init__(self):
        self.lock, self.holders, self.collects = threading.Lock(), 0, False

    def __enter__(self):
        with self.lock:
            if self.holders == 0:
                self.collects = gc.isenabled()
            self.holders += 1
            gc.disable()

    def __exit__(self, *exc):
        with self.lock:
            self.holders -= 1
            if self.holders == 0 and self.collects:
                gc.enable()


_collector_held = _CollectorHeld()


@contextlib.contextmanager
def _capturing(graph: torch.cuda.CUDAGraph, pool, stream):
    """Capture into ``graph`` without automatic collections: one could free what a runner left in a cycle (pinned memory, events, graphs),
    which is an error while a stream captures."""
    with _collector_held, torch.cuda.graph(graph, pool=pool, stream=stream):
        yield


class _Graph:
    def __init__(self, meta: Dict[str, torch.Tensor]):
        self.meta = meta                     # static device inputs
        self.graph = torch.cuda.CUDAGraph()
        self.out = None                      # static device output: llama.Scored, or a step's (logits, argmax)
        self.replays = 0
        self.arrays: Optional[_Arrays] = None      # DecodeGraphs: ``meta``'s places in ``flat``
        self.flat: Optional[torch.Tensor] = None
        self.staging: List[Tuple[Dict[str, np.ndarray], torch.Tensor, Optional[torch.cuda.Event]]] = []
        self.next_stage = 0


class GraphedForward:
    """LRU cache of captured whole-model forwards, keyed by the bucketed shape.

    ``forward(meta, batch) -> llama.Scored`` must run embed..head for one micro-batch
    on the current stream using only ``meta`` (device tensors) and resident
    weights; it is called eagerly once (warm-up) and then under capture.
    """

    def __init__(self, device, forward: Callable, max_graphs: int = 8):
        self.dev = torch.device(device)
        self.forward = forward
        self.max_graphs = max_graphs
        self.pool = torch.cuda.graph_pool_handle()
        self.graphs: "OrderedDict[tuple, _Graph]" = OrderedDict()
        self.captures = 0
        self.replays = 0

    def _capture(self, key, batch: PackedBatch) -> _Graph:
        host = padded_meta(batch, key)
        meta = {k: torch.from_numpy(v).to(self.dev) for k, v in host.items()}
        g = _Graph(meta)
        s = torch.cuda.Stream(self.dev)
        s.wait_stream(torch.cuda.current_stream(self.dev))
        with torch.cuda.stream(s):
            self.forward(meta, batch)                       # warm-up (lazy inits, autotune)
        torch.cuda.current_stream(self.dev).wait_stream(s)
        torch.cuda.synchronize(self.dev)
        with _capturing(g.graph, self.pool, s):
            g.out = self.forward(meta, batch)
        torch.cuda.synchronize(self.dev)
        self.captures += 1
        return g

    def run(self, batch: PackedBatch):
        """Replay (capturing on first sight of the bucket) -> the scored rows on the device (llama.Scored)."""
        key = bucket_key(batch)
        g = self.graphs.get(key)
        if g is None:
            if len(self.graphs) >= self.max_graphs:
                self.graphs.popitem(last=False)
            g = self._capture(key, batch)
            self.graphs[key] = g
        else:
            self.graphs.move_to_end(key)
            for k, v in padded_meta(batch, key).items():
                g.meta[k].copy_(torch.from_numpy(v), non_blocking=False)
        g.graph.replay()
        g.replays += 1
        self.replays += 1
        n = batch.n_scored
        return g.out._replace(probs=g.out.probs[:n], greedy=g.out.greedy[:n], flat=g.out.flat if n == g.out.probs.shape[0] else None)


class DecodeGraphs:
    """Graph replay of decode-like calls: the later steps of ``--num_gen_token`` with the prefix
    and suffix K/V caches (every prompt's prefix K/V and its suffixes' earlier tokens come from
    the cache, one new row per suffix is computed) when every weight is in HBM (resident, or the
    HBM cache holding every shard).  Such a step is ~800 launches of a few tens of microseconds
    each; one graph replays them all.

    Unlike :class:`GraphedForward` the shapes are EXACT (no bucket padding: a padded row would
    also be captured into the suffix K/V cache), keyed by the batch's array shapes; consecutive steps of
    one generation have the same shapes, so one capture serves them all, and the steps of other cache entries of the
    same shapes: nothing of an entry is in a graph.  The metadata of each step (new token ids, positions, work items,
    cache rows and windows, and the addresses of the entry's per-layer K/V buffers, which the kernels read and write in
    place) is copied into the graph's static inputs before the replay.  (A capture is 3 ms of a generation's 21: 16 steps
    of 16 rows through four 7B layers.)"""

    def __init__(self, device, forward: Callable, max_graphs: int = 4):
        self.dev = torch.device(device)
        self.forward = forward
        self.max_graphs = max_graphs
        self.pool = torch.cuda.graph_pool_handle()
        self.graphs: "OrderedDict[tuple, _Graph]" = OrderedDict()
        self.captures = 0
        self.replays = 0

    @staticmethod
    def key(batch: PackedBatch, entry) -> tuple:
        """The layers whose K/V the graph reads and writes, and the step's shapes."""
        return (tuple(entry.layers), batch.r2_q_block, batch.q_block) + tuple(
            (k, v.shape) for k, v in sorted(batch.host_meta().items()))

    @staticmethod
    def _put_addresses(words: np.ndarray, entry) -> None:
        """``words``: the int32 head of a step's arrays, 64 bits a layer in the key's order."""
        words[:2 * len(entry.layers)].view(np.int64)[:] = [t.data_ptr() for t in entry.layers.values()]

    # pinned staging sets per graph: a replay may be enqueued while the previous one (and its
    # metadata copies) still runs, so a set is refilled only after the copies that read it ran
    STAGING_SETS = 2

    def _upload(self, g: _Graph, host: Dict[str, np.ndarray], entry) -> None:
        """One stream-ordered copy of all metadata from the graph's persistent pinned staging buffers (with a copy for each of
        the 12 arrays, 17 steps of 16 rows through four 7B layers took 22.3 ms, with one 21.3)."""
        if not g.staging:
            for _ in range(self.STAGING_SETS):
                pinned = torch.empty(g.arrays.size, dtype=torch.int32, pin_memory=True)
                g.staging.append((g.arrays.views(pinned.numpy()), pinned, None))
        views, pinned, ev = g.staging[g.next_stage]
        if ev is not None:
            ev.synchronize()                                 # the copy that last read this set ran
        for k, v in host.items():
            np.copyto(views[k], v, casting="no")
        self._put_addresses(pinned.numpy(), entry)
        g.flat.copy_(pinned, non_blocking=True)
        ev = torch.cuda.Event()
        ev.record(torch.cuda.current_stream(self.dev))
        g.staging[g.next_stage] = (views, pinned, ev)
        g.next_stage = (g.next_stage + 1) % len(g.staging)

    def run(self, batch: PackedBatch, entry, ids_dev: Optional[torch.Tensor] = None):
        """Replay (capture on the first sight of the shape) -> the static output (llama.Scored).
        ``ids_dev``: the batch's token ids as a device int32 tensor, copied over ``batch.ids`` on
        the stream (a speculative step whose new tokens are the previous step's device argmax).
        The metadata goes in by a stream-ordered copy from pinned memory, so a replay can be
        enqueued while an earlier one still runs (its static inputs are overwritten after it)."""
        key = self.key(batch, entry)
        host = batch.host_meta()
        g = self.graphs.get(key)
        if g is None:
            if len(self.graphs) >= self.max_graphs:
                self.graphs.popitem(last=False)
            arrays = _Arrays(host, _ceil(2 * len(entry.layers), 16))
            up = np.zeros(arrays.size, np.int32)
            for k, dst in arrays.views(up).items():
                np.copyto(dst, host[k], casting="no")
            self._put_addresses(up, entry)
            flat = torch.from_numpy(up).to(self.dev)
            meta = arrays.views(flat)
            meta["kv_at"] = {name: flat.data_ptr() + 8 * i for i, name in enumerate(entry.layers)}
            if ids_dev is not None:
                meta["ids"].copy_(ids_dev)
            g = _Graph(meta)
            g.arrays, g.flat = arrays, flat
            s = torch.cuda.Stream(self.dev)
            s.wait_stream(torch.cuda.current_stream(self.dev))
            with torch.cuda.stream(s):
                eager = self.forward(meta, batch)            # this step's result (+ lazy inits)
            torch.cuda.current_stream(self.dev).wait_stream(s)
            torch.cuda.synchronize(self.dev)
            with _capturing(g.graph, self.pool, s):
                g.out = self.forward(meta, batch)            # captured, not run: the eager pass computed
            torch.cuda.synchronize(self.dev)                 # this step (its cache writes are idempotent)
            self.captures += 1
            self.graphs[key] = g
            return eager
        self.graphs.move_to_end(key)
        self._upload(g, host, entry)
        if ids_dev is not None:
            g.meta["ids"].copy_(ids_dev, non_blocking=True)
        g.graph.replay()
        g.replays += 1
        self.replays += 1
        return g.out


class _StepInputs:
    """A decode shape's index arrays behind ``head`` entries: ``up`` (pinned) and ``flat`` (device), and ``meta``, the device
    arrays by name."""

    def __init__(self, host: Dict[str, np.ndarray], B: int, head: int, dev):
        arrays = _Arrays(host, head)
        self.up = torch.empty(arrays.size, dtype=torch.int32, pin_memory=True)
        self.flat = torch.empty(arrays.size, dtype=torch.int32, device=dev)
        words = self.up.numpy()
        self.address = words[:2].view(np.int64)
        self.views = list(arrays.views(words).values())
        self.meta = arrays.views(self.flat)
        self.meta.update(n_seqs=B, max_rows=1, all_rows=True)          # (every row's logits)

    def fill(self, host: Dict[str, np.ndarray], address: int) -> None:
        """(the step that last read ``up`` has been waited for)"""
        self.address[0] = address
        for dst, v in zip(self.views, host.values()):
            dst[...] = v


class StepGraphs:
    """Captured decode steps of a stateful (hybrid) model: one token per request, resident weights.

    A step mutates per-request state (K/V pages, recurrence slots), so there is no warm-up run: the
    first step of a shape runs eagerly (and does every lazy initialisation), the second is captured
    (capture executes nothing) and replayed, later ones only replayed.  The key is (requests in the
    step, widths of the page table and of the block page tables rounded up to ``TABLE_BUCKET`` pages, the state
    cache's generation): the
    pools' addresses are baked into the graph, so a pool that grew starts a new generation and the old
    graphs are dropped.  Every row's logits are computed (``want_idx`` = all rows); the caller picks
    the wanted ones.

    A step's index arrays are segments of one int32 buffer that the graph's first kernel fetches from pinned memory, and its
    logits and their argmax go straight to pinned memory, by the kernels that make them, at the address the buffer begins with (0, where
    no row is wanted: nowhere): a step is one launch and one wait (with a copy before the graph and two behind it the GPU idled 60 of 650 us of a step of 8
    requests)."""

    TABLE_BUCKET = 16
    KEYS = ("ids", "tok_seq", "tok_pos", "cu", "pos0", "slot", "page_table", "kv_slot", "want_idx")
    MAX_SEEN = 128
    ADDRESS = 16                # entries of the buffer before its first array; the results' address is in two of them

    def __init__(self, device, forward: Callable, ops, vocab: int, max_graphs: int = 8):
        self.dev = torch.device(device)
        self.forward = forward              # forward(meta) -> (logits [B, V] fp32, argmax [B] int32), written to meta["mirror"] too
        self.ops = ops
        self.vocab = int(vocab)
        self.max_graphs = max_graphs
        self.pool = torch.cuda.graph_pool_handle()
        self.graphs: "OrderedDict[tuple, _Graph]" = OrderedDict()
        self.seen: "OrderedDict[tuple, _StepInputs]" = OrderedDict()      # shapes a step of which has run
        self.captures = self.replays = self.eager = 0
        self.generation = -1
        self._down: Optional[torch.Tensor] = None      # pinned: where a step's results go

    def _step(self, inputs: "_StepInputs"):
        """The step's launches, its index arrays' arrival first."""
        self.ops.copy_words(inputs.up, inputs.flat)
        inputs.meta["mirror"] = self.ops.host_rows(inputs.flat[:2].view(torch.int64))
        return self.forward(inputs.meta)

    @classmethod
    def _widened(cls, t: np.ndarray) -> np.ndarray:
        w = np.zeros((t.shape[0], _ceil(t.shape[1], cls.TABLE_BUCKET)), np.int32)
        w[:, :t.shape[1]] = np.maximum(t, 0)
        return w

    def host_meta(self, batch) -> Dict[str, np.ndarray]:
        B = len(batch.rids)
        m = {k: getattr(batch, k) for k in self.KEYS if k not in ("page_table", "want_idx")}
        m["page_table"] = self._widened(batch.page_table)
        for P, t in batch.block_tables.items():
            m[f"block_table_{P}"] = self._widened(t)
        if batch.prev_ids is not None:
            m["prev_ids"] = batch.prev_ids
        m["want_idx"] = np.arange(B, dtype=np.int32)
        return m

    def run(self, batch, generation: int, want: List[int]) -> List[Tuple[np.ndarray, np.ndarray]]:
        """One step, waited for -> (logits [1, V] fp32, argmax [1] int32) of each row of ``want`` on the host, the caller's own."""
        if generation != self.generation:
            self.graphs.clear()
            self.seen.clear()
            self.generation = generation
        B = len(batch.rids)
        host = self.host_meta(batch)
        key = (B,) + tuple(v.shape[1] for v in host.values() if v.ndim == 2)
        n = B * (self.vocab + 1)
        if want and (self._down is None or self._down.numel() < 4 * n):
            self._down = alloc_host(4 * n)
        try:
            self._replay(key, host, B, self._down.data_ptr() if want else 0)
        finally:                                       # (pinned memory of the step is not touched before its kernels are done)
            torch.cuda.current_stream(self.dev).synchronize()
        if not want:
            return []
        words = self._down.numpy()[:4 * n].view(np.int32)
        logits, am = words[:-B].view(np.float32).reshape(B, self.vocab), words[-B:]
        return [(logits[i:i + 1].copy(), am[i:i + 1].copy()) for i in want]

    def _replay(self, key, host, B: int, address: int) -> None:
        g = self.graphs.get(key)
        if g is not None:
            self.graphs.move_to_end(key)
            g.inputs.fill(host, address)
        else:
            first = key not in self.seen
            if first:
                if len(self.seen) >= self.MAX_SEEN:
                    self.seen.popitem(last=False)
                self.seen[key] = _StepInputs(host, B, self.ADDRESS, self.dev)
            inputs = self.seen[key]
            inputs.fill(host, address)
            if first:
                self.eager += 1
                self._step(inputs)
                return
            if len(self.graphs) >= self.max_graphs:
                self.graphs.popitem(last=False)
            g = _Graph(inputs.meta)
            g.inputs = inputs
            s = torch.cuda.Stream(self.dev)
            s.wait_stream(torch.cuda.current_stream(self.dev))
            torch.cuda.synchronize(self.dev)
            with _capturing(g.graph, self.pool, s):
                g.out = self._step(inputs)
            torch.cuda.synchronize(self.dev)
            self.graphs[key] = g
            self.captures += 1
        g.graph.replay()
        g.replays += 1
        self.replays += 1
