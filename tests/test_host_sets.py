"""The sets of arrays that a captured step takes from host memory by itself: the host's side, with a thread or the test in the GPU's place."""
from __future__ import annotations

import gc
import threading
import time
import weakref

import pytest
import torch

from tiny_inference_server_amd.engine import graph as G


def sets_of(counters=3, wait=None):
    return G.HostSets(torch.zeros(2, 8, dtype=torch.int32), torch.zeros(counters, dtype=torch.int32), wait)


def test_sets_are_written_in_turn_and_carry_what_the_last_step_left():
    s = sets_of()
    s.free()[:] = range(8)
    s.replayed()
    for k in range(1, 9):
        flat = s.carry()
        assert s.unread() == 1 and flat.tolist() == list(range(k - 1, k + 7))
        assert s.carry() is flat                             # (once a step)
        flat += 1
        s.replayed()
        assert s.ring[(k + 1) % 2].tolist() == list(range(k - 1, k + 7))      # the set before is as its replay may still have to read it
        s.done += 1                                          # the replay before has taken its set
    s.free()[:] = 7                                          # a step that brings everything: nothing is carried
    s.replayed()
    s.done += 1
    assert s.carry().tolist() == [7] * 8


def test_one_set_that_is_copied_is_free_once_it_is():
    waits = []
    s = G.HostSets(torch.zeros(1, 8, dtype=torch.int32), None, lambda: waits.append(1))
    for k in range(3):
        assert s.unread() == 0 and s.carry() is s.free()
        s.replayed()
    assert len(waits) == 6                                   # every time for the copy that may still be under way


@pytest.mark.parametrize("start", [0, 0x7FFFFFFE, 0xFFFFFFFE])
def test_a_set_is_free_once_every_workgroup_has_read_it(start):
    """Counters of 32 bits that go on past their sign and past their end; the slowest workgroup decides."""
    s = sets_of()
    s.replays = start
    s.done[:] = torch.tensor(start, dtype=torch.int64).to(torch.int32)
    turns, seen = 6, []

    def device():
        for k in range(turns):
            while not s.unread():
                time.sleep(1e-4)
            for i in range(3):                               # (the host is two steps ahead long before the last one)
                time.sleep(3e-3)
                if i == 2:
                    seen.append(s.ring[k % 2, 0].item())
                s.done[i] = (s.done[i].item() + 1 + (1 << 31)) % (1 << 32) - (1 << 31)

    t = threading.Thread(target=device, daemon=True)
    t.start()
    for k in range(turns):
        s.free()[:] = 100 + k
        s.replayed()
    t.join(20)
    assert not t.is_alive() and seen == [100 + k for k in range(turns)] and s.unread() == 0


def test_a_step_that_never_takes_its_arrays_is_said_so(monkeypatch):
    monkeypatch.setattr(G.HostSets, "ASK_EVERY", 50)
    asked = []
    s = sets_of(wait=lambda: asked.append(1))
    s.replayed(), s.replayed()
    with pytest.raises(RuntimeError, match="never took"):
        s.free()
    assert asked == [1]
    late = sets_of(wait=lambda: late.done.fill_(2))           # a device with that much to do
    late.replayed(), late.replayed()
    late.free()


def test_sets_that_a_replay_has_still_to_read_outlive_their_graph():
    """However long it takes, and without waiting for it; once they are read they go with the next graph that is made or dropped."""
    def graph(replays, taken):
        g = object.__new__(G.DecodeGraph)
        g.sets = sets_of()
        g.sets.replays = replays
        g.sets.done[:] = taken
        return g, weakref.ref(g.sets), g.sets.done

    G._release_read()
    pending, sets, done = graph(5, 4)
    read, gone, _ = graph(5, 5)
    before = time.monotonic()
    del pending, read
    gc.collect()
    assert time.monotonic() - before < 5 and sets() is not None and gone() is None
    other, others, _ = graph(2, 1)
    del other
    assert sets() is not None and others() is not None
    done[:] = 5
    G._release_read()
    assert sets() is None and others() is not None
    others().done[:] = 2
    G._release_read()
    assert others() is None and not G._UNREAD


def test_a_graph_that_was_never_made_is_dropped_quietly():
    object.__new__(G.DecodeGraph).__del__()
