"""Gradients of batches whose strings are scored in LDS: the sweeps of several steps are made when a gradient first asks, in
whatever order scores, gradients and the setting for several steps come.  FP64 sums in another order: 1e-11."""
import numpy as np
import pytest

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
def test_gradients_before_and_after_scores(storage, tmp_path):
    plans, bits = [], []
    rng = np.random.default_rng(31)
    for i, shape in enumerate([(24, 10, 1), (33, 13, 2)]):
        inst = egs.instances.Instance(*shape)
        plans.append(str(tmp_path / f"p{i}.txt"))
        inst.write_plan(plans[-1])
        bits.append(rng.integers(0, 2, size=(64, inst.N)).astype(np.int8))
    print(storage, flush=True)

    def values(order):
        with gs.BatchEngine(plans, [64, 64], storage=storage) as bt:
            out = {}
            for what in order:
                if what in ("on", "off"):
                    bt.set_pairs(what == "on")
                elif what == "graph":
                    bt.use_graph(True)
                elif what == "score":
                    out["score"] = bt.score(bits)
                else:
                    out["grad"] = bt.grad(bits)[0]
            return out

    first = values(("grad", "score"))
    others = [values(o) for o in (("score", "grad", "score"), ("off", "grad", "score", "on", "score", "grad", "grad"),
                                  ("graph", "score", "grad", "score"), ("off", "score", "grad"))]
    for j, other in enumerate(others):
        for i in range(2):
            a, b = first["grad"][i], other["grad"][i]
            assert np.array_equal(first["score"][2][i], other["score"][2][i])
            assert np.max(np.abs(first["score"][0][i] - other["score"][0][i])) < 1e-11
            if j < 3:                                         # the same sweeps: the same sums
                assert all(np.array_equal(x, y) for x, y in zip(a, b))
            assert np.array_equal(a[1], b[1]) and np.max(np.abs(a[0] - b[0])) < 1e-11
            assert np.max(np.abs(a[2] - b[2])) < 1e-11 * np.max(np.abs(a[2]))
