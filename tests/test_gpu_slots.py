"""Strings of one call when the device has no room for as many arenas as the call would take: it takes fewer per launch, and
an engine keeps the ones it has.  The results are those of one string per launch to the last bit."""
import numpy as np
import pytest
import torch

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu


def test_fewer_arenas_where_memory_is_short(tmp_path):
    inst = egs.instances.Instance(60, 24, 4, R=22)            # complex64 arenas of 32 MiB
    plan = str(tmp_path / "p.txt")
    inst.write_plan(plan)
    given = np.random.default_rng(3).integers(0, 2, size=(40, inst.N)).astype(np.int8)
    room = 400 << 20                                          # eight to eleven more arenas, not the forty asked for
    with gs.Engine(plan, gs.C64) as one:
        ref = np.concatenate([one.chain(g)[0] for g in given])
    with gs.Engine(plan, gs.C64) as e:
        assert np.array_equal(e.chain(given[:2])[0], ref[:2])
        torch.cuda.synchronize()
        fill, block = [], 16 << 30
        while block >= 64 << 20:                              # leaves between `room` and a little more
            while torch.cuda.mem_get_info()[0] > room + block:
                fill.append(torch.empty(block, dtype=torch.uint8, device="cuda"))
            block //= 2
        free = torch.cuda.mem_get_info()[0]
        print("free MiB", free >> 20, flush=True)
        assert room < free < 2 * room
        got = e.chain(given)[0]
        left = torch.cuda.mem_get_info()[0]
        again = e.chain(given)[0]
        same = torch.cuda.mem_get_info()[0]
        fill.clear()
        torch.cuda.empty_cache()
    print("left MiB", left >> 20, same >> 20, flush=True)
    assert np.array_equal(got, ref) and np.array_equal(again, ref)
    assert left < free and same == left                       # more arenas than the two before, and kept
