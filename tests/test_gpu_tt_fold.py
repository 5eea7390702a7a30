"""Two-table engine with the next step's norms folded into each write, against the in-place engine on the same instance:
identical bits, log2 Pr and conditionals to the storage's rounding (the two engines round different intermediate tables:
1e-5 in complex64, 1e-11 in complex128)."""
import numpy as np
import pytest

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu

# tables below a block; with and without partner directions; gadget plans (kernels holding the bare x bit)
PLANS = [(20, 6, 1, 0), (34, 14, 3, 0), (40, 17, 3, 9), (45, 18, 11, 0), (52, 21, 8, 0)]


@pytest.mark.parametrize("storage,tol", [(gs.C64, 1e-5), (gs.C128, 1e-11)])
@pytest.mark.parametrize("shape", PLANS)
@pytest.mark.parametrize("grid", [1, 4, 0])
def test_two_table_equals_in_place(shape, storage, tol, grid, tmp_path):
    n, band, seed, gadgets = shape
    inst = egs.instances.Instance(n, band, seed, gadgets_count=gadgets)
    plan, ttplan = str(tmp_path / "p.txt"), str(tmp_path / "tt.txt")
    inst.write_plan(plan)
    egs.engine.write_sampler_plan(ttplan, inst.am)
    rng = np.random.default_rng(4)
    given = rng.integers(0, 2, size=(2, inst.N)).astype(np.int8)
    given[:, :gadgets] = 0
    part = given.copy()
    part[:, inst.N // 2:] = -1
    part[:, inst.N // 2 + 3] = 1
    print(shape, storage, grid, flush=True)
    with gs.Engine(plan, storage) as e, gs.TwoTableEngine(ttplan, storage=storage) as t:
        t.set_grid_log2(grid)
        # a gadget plan's ancillas are projected on 0, so whole strings are only sampled from plans without
        if not gadgets:
            bits, lp = t.sample(3, 21)
            rb, rl = e.sample(3, 21)
            assert np.array_equal(bits, rb) and np.max(np.abs(lp - rl)) < tol
        assert np.max(np.abs(t.prob(given) - e.prob(given))) < tol
        tb, tl, tc = t.hybrid(part, 3)
        rb, rl, rc = e.hybrid(part, 3)
        assert np.array_equal(tb, rb) and np.max(np.abs(tl - rl)) < tol and np.max(np.abs(tc - rc)) < tol
        again = t.hybrid(part, 3)
        assert np.array_equal(again[1], tl) and np.array_equal(again[2], tc)
