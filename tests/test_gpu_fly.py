"""Butterfly sweeps (two steps per write, the second one's decision from a read-only pass) against one step per sweep, on
plans whose steps are large enough to take them: identical bits; log2 Pr and conditionals to the order of their FP64
sums, which moves a decision's scale by 1e-16 and so now and then the rounding of a stored value (1e-9 in complex64
tables of 2^20 entries and more, 1e-12 in complex128)."""
import numpy as np
import pytest

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,tol", [(gs.C64, 1e-9), (gs.C128, 1e-12)])
@pytest.mark.parametrize("shape", [(70, 26, 3, 0), (66, 26, 8, 0), (48, 24, 5, 16)])
@pytest.mark.parametrize("grid", [5, 0])
def test_butterflies_equal_single_steps(shape, storage, tol, grid, tmp_path):
    n, band, seed, gadgets = shape
    inst = egs.instances.Instance(n, band, seed, gadgets_count=gadgets)
    plan = str(tmp_path / "p.txt")
    inst.write_plan(plan)
    given = np.random.default_rng(6).integers(0, 2, size=(2, inst.N)).astype(np.int8)
    given[:, :gadgets] = 0
    part = given.copy()
    part[:, inst.N // 3:] = -1
    part[1, inst.N // 2:inst.N // 2 + 3] = 0                # forced steps inside the run
    print(shape, storage, grid, flush=True)
    got = []
    with gs.Engine(plan, storage) as e:
        e.set_grid_log2(grid)
        for on in (True, False):
            e.set_pairs(on)
            got.append((*e.sample(2, 31), e.prob(given), *e.hybrid(part, 4), *e.chain(given)))
    for a, b in zip(*got):
        if a.dtype == np.int8:
            assert np.array_equal(a, b)
        elif a.dtype == complex:
            assert np.array_equal(a, b)                     # chain mode: the same tables
        else:
            assert np.allclose(a, b, rtol=tol, atol=tol), np.max(np.abs(a - b))
