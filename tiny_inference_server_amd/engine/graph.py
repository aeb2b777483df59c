"""Captured steps.

A step in which every request brings exactly one token, far enough into its sequence that every stage has
one row per request, always launches the same kernels on arrays of the same shapes. Such a step is
captured once per (number of requests, block-table width) as a HIP graph over a fixed device buffer that
holds the step's integer arrays; later steps of the same shape write their arrays into pinned memory, from where the
graph's first kernel takes them, and replay the graph, which removes the launch cost of several hundred small kernels. Any other step is captured
the same way once its exact shape (row counts, wanted places, attention work) has come three times.

Nothing is cleared inside the graph with a memset, and the first steps of a shape run without a graph (the
library chooses its algorithms for the shape then), so a capture records kernel launches only.
"""
from __future__ import annotations

import gc
import time
from collections import deque

import numpy as np
import torch

from .batch import StepPlan, materialize


class _NoEvent:
    """Stands in for a device event where copies are synchronous (a host-only run)."""

    def record(self):
        pass

    def synchronize(self):
        pass


class HostSets:
    """The sets of a captured step's arrays in host memory: two, written in turn, where the graph itself takes them from there (upload_ring), and
    `done` is where the GPU writes down how many replays each of its workgroups has taken; else one (done: None), which is copied before every replay.
    wait: waits for the last copy out of the one set, or for the device, where it has not taken one of two for seconds."""
    ASK_EVERY = 100000

    def __init__(self, ring: torch.Tensor, done, wait):
        self.ring, self.done, self.wait = ring, done, wait
        self._sets = list(ring.numpy())
        self._read = done.numpy().view(np.uint32) if done is not None else None
        self.at = 0                  # the set that the next replay takes ...
        self.held = 0                # ... and the one that holds what the last step left
        self.replays = 0

    def unread(self) -> int:
        """How many replays have not yet taken their set."""
        return max((self.replays - int(n)) & 0xFFFFFFFF for n in self._read) if self._read is not None else 0      # (32-bit counters)

    def free(self) -> np.ndarray:
        """The set that the next replay takes, once no replay before it still has to read it."""
        if self._read is None:
            self.wait()
        waits = 0
        while self.unread() > 1:
            waits += 1
            if waits > 100:
                time.sleep(0 if waits < 20000 else 5e-5)
            if waits % self.ASK_EVERY == 0:       # seconds: either the GPU has that much to do, or it says here what went wrong
                self.wait()
                if self.unread() > 1:
                    raise RuntimeError("a replayed step never took its arrays")
        return self._sets[self.at]

    def carry(self) -> np.ndarray:
        """The next replay's set, holding what the last step left."""
        if self.held == self.at and self._read is not None:
            return self._sets[self.at]            # (of two sets: free since the call that carried it over, or never launched)
        flat = self.free()
        if self.held != self.at:
            np.copyto(flat, self._sets[self.held])
            self.held = self.at
        return flat

    def replayed(self) -> None:
        """The next replay has been launched, on the set that has been filled."""
        self.held = self.at
        if self._read is not None:
            self.replays = (self.replays + 1) & 0xFFFFFFFF
            self.at ^= 1


# Sets of graphs that were dropped while a replay had still to read them: a kernel reads them, of which the memory's allocator knows nothing, so they stay
# until the counters say that it has. Looked through when a graph is made or dropped; no call of the runtime, because a graph may be dropped while
# another is being captured.
_UNREAD = deque()


def _release_read(sets=None) -> None:
    if sets is not None:
        _UNREAD.append(sets)
    for _ in range(len(_UNREAD)):
        try:
            kept = _UNREAD.popleft()
        except IndexError:           # (another thread looks through them too)
            return
        if kept.unread():
            _UNREAD.append(kept)


class DecodeGraph:
    """One captured step: a fixed buffer of the step's integer arrays, and the graph that runs on it.

    occupants: for every entry of the plan something that names the request itself and not merely its slot
    (the engine passes (slot, admission number)); the quick update below is only right while the buffer's
    lines belong to the very same requests.
    capture=False records nothing: a replay then runs the same calls again on the same buffers. That is how an
    operations object without a device (a test's stand-in) exercises this file's host logic.
    """

    def __init__(self, engine, plan: StepPlan, kv_capacity: int, occupants=None, capture: bool = True, mode=None, heads: bool = False):
        self.layout = plan.layout()
        self.mode = mode
        self.heads = heads       # every stage's logits, as the model's all_logits gives them
        self.engine = engine
        self.capture = capture
        dev = engine.device
        on_gpu = torch.device(dev).type == "cuda"
        total = max(plan.packer.total, 4)
        self.uploads = on_gpu and capture and hasattr(engine.ops, "upload_ring")
        _release_read()
        ring = torch.zeros(2 if self.uploads else 1, total, dtype=torch.int32, pin_memory=on_gpu)
        self.dev = torch.zeros(total, dtype=torch.int32, device=dev)
        self.copied = torch.cuda.Event() if on_gpu and not self.uploads else _NoEvent()      # (of the one set)
        if self.uploads:
            counters = engine.ops.upload_counters(total)
            self._sent = torch.zeros(counters, dtype=torch.int32, device=dev)
            self.sets = HostSets(ring, torch.zeros(counters, dtype=torch.int32, pin_memory=True), lambda: torch.cuda.synchronize(dev))
        else:
            self.sets = HostSets(ring, None, self.copied.synchronize)
        self.step = materialize(plan, dev, ring[0], self.dev)
        for st in self.step.stages:          # later steps of the shape may see more keys than this one
            st.max_kv_len = kv_capacity
        self.graph = None
        if capture:
            self.graph = torch.cuda.CUDAGraph()
            torch.cuda.synchronize(dev)
            # No garbage collection while the stream is capturing: a collection may finalise an engine that is no
            # longer used (engines and their captured steps refer to each other, so only the collector frees them),
            # and destroying its graphs in the middle of a capture aborts the process. The context below collects
            # once before the capture begins.
            collecting = gc.isenabled()
            gc.disable()
            try:
                with torch.cuda.graph(self.graph):
                    self._launch()
            finally:
                if collecting:
                    gc.enable()
        self.copied.record()         # (with two sets: the copy that `materialize` made was waited for before the capture)
        # what the quick update needs: which requests, in which order, the buffer holds, and where their arrays lie
        self.slots = tuple(e.slot for e in plan.entries)
        self.occupants = tuple(occupants) if occupants is not None else None
        self.cache = engine.cache
        self.page_size = engine.page_size
        off = lambda i: plan.packer.offsets[i][0]
        self.table_at = {g: (off(i), plan.packer.offsets[i][1]) for g, i in plan.bt_ids.items()}
        self.stage_at = [dict(lag=pl["lag"], tokens=off(pl["tokens"]), positions=off(pl["positions"]),
                              ws={g: off(i) for g, i in pl["ws"].items()}) for pl in plan.plans]
        # the same for all stages at once: where the requests' positions go [stages, requests], and for each group of pages, of the stages
        # that write to it, where their slots go and where the requests' block tables begin
        line = np.arange(len(self.slots))
        slots = {}
        for g, (t_off, (_, width)) in self.table_at.items():
            stages = [j for j, st in enumerate(self.stage_at) if g in st["ws"]]
            if stages:
                slots[g] = (stages, np.array([self.stage_at[j]["ws"][g] + line for j in stages]), t_off + line * width)
        self._places = (np.array([st["positions"] + line for st in self.stage_at]), np.array([[st["lag"]] for st in self.stage_at]), slots)
        self.pages_held = {g: np.array([len(engine.cache.groups[g].tables[s]) for s in self.slots])
                           for g in self.table_at}
        # what the parts planned for each stage (work lists of their kernels): where each array lies, in the order
        # the planning added them, and the host values that the captured launches were made from
        self.extras_at = [[(off(i), plan.packer.offsets[i][1]) for i in sorted(v[0] for v in pl["extra"].values())]
                          for pl in plan.plans]
        self.extras_host = [tuple(sorted((k, v[1:]) for k, v in pl["extra"].items())) for pl in plan.plans]
        self._ahead = None       # (positions the buffer was filled for ahead of time, requests still to be filled)

    def _launch(self):
        engine, n = self.engine, self.step.n_wanted
        if self.uploads:
            engine.ops.upload_ring(self.sets.ring, self.dev, self._sent, self.sets.done)
        outs = engine.model.forward(self.step, engine.cache)
        self.logits = engine.model.all_logits(outs, n) if self.heads else engine.logits_of(outs, self.step, n)

    @property
    def host(self) -> torch.Tensor:
        """The arrays as they stand for the next step."""
        self.sets.carry()
        return self.sets.ring[self.sets.at]

    def _replay(self):
        """The step, on the set that has been filled."""
        if not self.uploads:
            self.dev.copy_(self.sets.ring[0], non_blocking=True)
            self.copied.record()
        if self.graph is not None:
            self.graph.replay()
        else:
            self._launch()
        self.sets.replayed()

    def __del__(self):
        try:
            if self.sets.unread():
                _release_read(self.sets)
        except Exception:            # not made to the end, or the interpreter is going away
            pass

    def holds(self, occupants) -> bool:
        """Whether the buffer's lines are those of exactly these requests, in this order."""
        return self.occupants is not None and self.occupants == tuple(occupants)

    def run_same_requests(self, entries) -> torch.Tensor:
        """The next step of the very requests whose arrays the buffer already holds, in the same order: only
        tokens, positions, write slots and newly taken pages change, and those are written in place.

        Everything but the tokens depends on the requests' positions alone, and after a step of single tokens the
        likeliest next step is the same requests one position on. So once a step has been launched, while the GPU
        runs it (the caller cannot go on before it has the step's tokens anyway), the buffer is filled for that next
        step; when it comes, only its tokens, and the lines of requests that have taken a page since, are left to
        write before the copy and the replay."""
        flat = self.sets.carry()
        n = len(entries)
        starts = np.fromiter((e.start for e in entries), dtype=np.int64, count=n)
        tokens = np.fromiter((e.tokens[0] for e in entries), dtype=np.int32, count=n)
        ahead, self._ahead = self._ahead, None
        if ahead is not None and len(ahead[0]) == n and np.array_equal(ahead[0], starts):
            if ahead[1]:
                self._fill_late(flat, starts, ahead[1])
        else:
            self._fill_positions(flat, starts)
        return self._run_filled(starts, tokens)

    def run_ahead(self, tokens) -> torch.Tensor:
        """The step that the buffer was filled for ahead of time, with its requests' tokens (lines that fill the step up keep theirs):
        run_same_requests for a caller that knows which step this is."""
        starts, late = self._ahead
        self._ahead = None
        if late:
            self._fill_late(self.sets.carry(), starts, late)
        return self._run_filled(starts, tokens)

    def _run_filled(self, starts, tokens) -> torch.Tensor:
        flat, n = self.sets.carry(), len(tokens)
        for st in self.stage_at:
            flat[st["tokens"]:st["tokens"] + n] = tokens
        self._replay()
        # the arrays of the step after this one, while this one runs
        flat = self.sets.carry()
        nxt = starts + 1
        if self.cache.spare_slot is not None:       # (lines that fill the step up stay where they are)
            nxt = nxt - np.fromiter((s == self.cache.spare_slot for s in self.slots), dtype=np.int64, count=len(starts))
        self._ahead = (nxt, self._fill_positions(flat, nxt, ahead=True))
        return self.logits

    def _table_line(self, flat, g, k, need):
        """Request k's line of a block table, where it holds fewer than `need` pages; False where the request has not got them either."""
        held = self.pages_held[g][k]
        if need <= held:
            return True
        t_off, (_, width) = self.table_at[g]
        t = self.cache.groups[g].tables[self.slots[k]]
        if len(t) < need:
            return False
        if len(t) > width:
            raise RuntimeError("a block table outgrew the captured width")
        at = t_off + k * width
        if self.engine._has_windows:                # (pages that a window has passed are given back: the whole line)
            flat[at:at + len(t)] = [p if p >= 0 else 0 for p in t]
        else:
            flat[at + held:at + len(t)] = t[held:]
        self.pages_held[g][k] = len(t)
        return True

    def _fill_late(self, flat, starts, late):
        """What _fill_positions writes, for the few requests it left out ahead of the step because their positions open pages."""
        ps = self.page_size
        for k in late:
            start = int(starts[k])
            for g in self.table_at:
                if not self._table_line(flat, g, k, start // ps + 1):
                    raise RuntimeError("a request's position lies beyond its pages")
            for st in self.stage_at:
                pos = start - st["lag"]
                flat[st["positions"] + k] = pos
                for g, w_off in st["ws"].items():
                    t_off, (_, width) = self.table_at[g]
                    flat[w_off + k] = flat[t_off + k * width + pos // ps] * ps + pos % ps

    def _fill_positions(self, flat, starts, ahead=False):
        """Positions, write slots, newly taken pages and the parts' work lists for requests that stand at `starts`.
        ahead: the step has not come yet, so a request whose position opens a page may not have that page; such
        requests are skipped and their indices returned, to be filled when the step comes."""
        n = len(starts)
        ps = self.page_size
        late = []
        need = starts // ps + 1
        for g in self.table_at:
            for k in np.nonzero(need > self.pages_held[g])[0].tolist():
                if not self._table_line(flat, g, k, int(need[k])):
                    if not ahead:
                        raise RuntimeError("a request's position lies beyond its pages")
                    if k not in late:
                        late.append(k)
        which = [k for k in range(n) if k not in late] if late else slice(None)
        places, lags, slots = self._places
        pos = starts[which] - lags               # [stages, requests]
        flat[places[:, which]] = pos
        page, at = np.divmod(pos, ps)
        for g, (stages, into, lines) in slots.items():
            flat[into[:, which]] = flat[lines[which] + page[stages]] * ps + at[stages]
        if any(self.extras_at):
            # the parts plan again for the new positions, into the places their arrays have in the buffer
            for at, host_values, st in zip(self.extras_at, self.extras_host, self.stage_at):
                slots_left = list(at)

                def put(arr, shape=None, slots_left=slots_left):
                    a = np.ascontiguousarray(arr, dtype=np.int32).reshape(-1)
                    if not slots_left or int(np.prod(slots_left[0][1])) != a.size:
                        raise RuntimeError("a part planned an array that the captured step has no place for")
                    o, _ = slots_left.pop(0)
                    flat[o:o + a.size] = a
                    return -1

                pos = starts - st["lag"]
                extra = self.engine.model.plan_rows([(k, int(pos[k]), 1) for k in range(n)], put, self.mode)
                if slots_left or tuple(sorted((k, v[1:]) for k, v in extra.items())) != host_values:
                    raise RuntimeError("the parts' planning no longer fits the captured step")
        return late

    def run(self, plan: StepPlan, occupants=None) -> torch.Tensor:
        if plan.layout() != self.layout:
            raise RuntimeError("this step's arrays do not have the captured layout")
        flat = self.sets.free()
        self._ahead = None
        plan.packer.fill(flat)
        self.slots = tuple(e.slot for e in plan.entries)
        self.occupants = tuple(occupants) if occupants is not None else None
        for g in self.table_at:
            self.pages_held[g] = np.array([len(self.cache.groups[g].tables[s]) for s in self.slots])
        self._replay()
        return self.logits
