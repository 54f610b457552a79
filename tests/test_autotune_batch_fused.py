"""CPU test of the batch autotuner's search on a batch whose members take the
fused sweep: it is not searched for an x chunk length that no member uses."""
import time

import pytest

from test_autotune import Clock, FakeBatch, load_autotune


class FakeFusedBatch(FakeBatch):
    """All of four members take the fused sweep: the x chunk length changes nothing."""

    members = dict.fromkeys(range(4))

    def fused_members(self):
        return self.fused

    def cost(self):
        lx, self.tiles = self.tiles[0], (8,) + tuple(self.tiles[1:])
        c = super().cost()
        self.tiles = (lx,) + tuple(self.tiles[1:])
        return c


@pytest.mark.parametrize("fused", [4, 3])
def test_batch_finalists_differ_in_shapes_that_are_used(monkeypatch, fused):
    at = load_autotune()
    clock = Clock()
    monkeypatch.setattr(time, "perf_counter", clock)
    b = FakeFusedBatch(clock)
    b.fused = fused
    res = at.autotune_batch(b, 0.01, steps=4)
    assert res["tiles"][1] == 16 and res["col_threads"] == 768 and res["streams"] == 2
    assert {t[0] for t, _, _ in b.timed} == ({8} if fused == 4 else {8, 16})
    if fused == 4:
        assert len({(t[1], thr) for t, thr, g in b.timed if g > 1}) == 3
