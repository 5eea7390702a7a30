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


# plateaus of 24 and 20 steps; gadgets; two instances whose plateaus overlap in part
BATCHES = [[((40, 8, 1, 0), 64)], [((52, 16, 4, 0), 128)], [((40, 12, 3, 6), 64)],
           [((40, 8, 1, 0), 64), ((44, 10, 2, 0), 64)]]


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
@pytest.mark.parametrize("batch", BATCHES)
def test_batched_butterflies_equal_single_steps(batch, storage, tmp_path):
    """The tables are the same bit for bit; norms and gradients are FP64 sums over up to 2^16 cosets in another order
    (2^16 terms x 2^-53, with room: 1e-11)."""
    plans, bits = [], []
    rng = np.random.default_rng(19)
    for i, ((n, band, seed, gadgets), lanes) in enumerate(batch):
        inst = egs.instances.Instance(n, band, seed, gadgets_count=gadgets)
        plans.append(str(tmp_path / f"p{i}.txt"))
        inst.write_plan(plans[-1])
        bits.append(rng.integers(0, 2, size=(lanes, inst.N)).astype(np.int8))
    print(batch, storage, flush=True)
    with gs.BatchEngine(plans, [lanes for _, lanes in batch], storage=storage) as bt:
        many = bt.score(bits)
        gmany, _ = bt.grad(bits)
        gseg, _ = bt.grad(bits, seg=5)
        bt.set_pairs(False)
        one = bt.score(bits)
        gone, _ = bt.grad(bits)
    for i in range(len(batch)):
        assert np.array_equal(many[2][i], one[2][i])
        assert np.max(np.abs(many[0][i] - one[0][i])) < 1e-11
        assert np.allclose(many[1][i], one[1][i], rtol=1e-11, atol=0)
        assert np.max(np.abs(gmany[i][2] - gone[i][2])) < 1e-11 * np.max(np.abs(gone[i][2]))
        assert np.array_equal(gmany[i][2], gseg[i][2]) and np.array_equal(gmany[i][1], gseg[i][1])
