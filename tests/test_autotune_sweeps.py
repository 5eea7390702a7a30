"""Tile choice of the autotuner where one sweep takes several steps: the steps inside it take the sweep's tile (their own
times are 0 whatever the tile, which says nothing about it).  A stand-in batch; no device calls."""
import time
import types

import numpy as np
import pytest

from _pkg import egs

at = egs.autotune


class Batch:
    """Steps 0 .. 2 are one sweep, fastest with tiles of 2^12; step 3 is one of its own, fastest with 2^10."""

    maxns, lanes, storage = 4, [64], 0

    def __init__(self):
        self.plans = [types.SimpleNamespace(ns=4, digest="d")]
        self.tile = [9] * 4
        self.graph = False

    def set_tile(self, i, lg, k):
        self.tile[k] = lg

    def set_unroll(self, lu):
        pass

    def use_graph(self, on):
        self.graph = on

    def score(self, bits, **_):
        if self.graph:
            time.sleep(1e-3 * (abs(self.tile[0] - 12) + abs(self.tile[3] - 10)))

    def last_ms(self):
        a = 1.0 + abs(self.tile[0] - 12)
        b = a + 1.0 + abs(self.tile[3] - 10)
        return b, np.array([a, a, a, b])


@pytest.mark.parametrize("cache", [False, True])
def test_steps_inside_a_sweep_take_its_tile(cache, tmp_path):
    bt = Batch()
    path = str(tmp_path / "tiles.json") if cache else None
    got = at.tune_tiles(bt, None, cache=path)
    assert got["choice"] == "per_step" and got["lg"] == [12, 12, 12, 10] and bt.tile == [12, 12, 12, 10]
    if cache:
        bt.tile = [9] * 4
        again = at.tune_tiles(bt, None, cache=path)
        assert again["cached"] and again["lg"] == got["lg"] and bt.tile == got["lg"]
