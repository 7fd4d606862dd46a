"""The engine's ring of pinned regions: a region is written again only behind the event of every upload it overlaps."""
import random

import pytest
import torch

from llm_weighted_consensus_amd.engine import engine


@pytest.mark.parametrize("sizes", [
    # a small region at the arena's end that the next round passes over: what lies at its start is still waited for
    [250, 250, 250, 200, 50, 250, 250, 250, 150, 150, 250],
    [random.Random(3).randint(1, 250) for _ in range(400)]])
def test_regions_wait_for_what_they_overlap(monkeypatch, sizes):
    made = []

    class Event:
        def record(self):
            made.append(self)
            self.done = False

        def synchronize(self):
            self.done = True

    empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **kw: empty(*a, **kw))
    monkeypatch.setattr(torch.cuda, "Event", Event)
    ring = engine._PinnedRing(1000 * 256)
    regions = []
    for n in sizes:
        before = len(made)
        ring.upload(torch.zeros(n * 256, dtype=torch.uint8), "cpu")
        start, end, ev = ring.live[-1]
        assert ev is made[before] and end - start == n * 256 and end <= ring.n
        for a, b, other in regions:
            assert other.done or b <= start or end <= a
        regions.append((start, end, ev))
