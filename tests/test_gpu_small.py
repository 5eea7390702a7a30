"""Runs of small steps (one block per string, table in LDS) and chain-mode pairs of steps against one sweep per step: the
same bits and amplitudes, and log2 Pr and conditionals to the order of their FP64 sums (at most 2^14 terms: 1e-12)."""
import numpy as np
import pytest

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu

# one-wave steps only; whole plan in one run; head and tail runs; gadget plans (one-output steps); more steps than a run
# holds (64)
PLANS = [(7, 3, 2, 0), (24, 10, 1, 0), (34, 14, 3, 0), (40, 18, 3, 12), (22, 9, 5, 8), (75, 6, 4, 0)]


def _inst(shape, tmp_path):
    n, band, seed, gadgets = shape
    inst = egs.instances.Instance(n, band, seed, gadgets_count=gadgets)
    plan = str(tmp_path / "p.txt")
    inst.write_plan(plan)
    return inst, plan


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
@pytest.mark.parametrize("limit", [3, 6, 10, 12])
@pytest.mark.parametrize("shape", PLANS)
def test_small_runs_equal_single_sweeps(shape, limit, storage, tmp_path):
    inst, plan = _inst(shape, tmp_path)
    rng = np.random.default_rng(5)
    given = rng.integers(0, 2, size=(3, inst.N)).astype(np.int8)
    part = given.copy()
    part[:, inst.N // 3:] = -1
    K = inst.N // 2
    print(shape, limit, storage, flush=True)
    with gs.Engine(plan, storage) as e:
        e.set_pairs(False)
        got = []
        for nk in (limit, -1):
            e.set_small_steps(nk)
            bits, lp = e.sample(3, 9)
            pre = e.prefix(given[0], K)
            res = e.resume(np.concatenate([given[0][:K], np.full(inst.N - K, -1, np.int8)]), K, [pre[0]], [pre[3]], 4)
            got.append((bits, lp, e.prob(given), *e.chain(given), *e.hybrid(part, 2), pre[0], np.array(pre[3:]), *res))
    tol = 1e-12 if storage == gs.C128 else 2e-6
    for a, b in zip(*got):
        a, b = np.asarray(a), np.asarray(b)
        if a.dtype == np.int8:
            assert np.array_equal(a, b)
        else:
            assert np.allclose(a, b, rtol=tol, atol=tol * 1e-3), np.max(np.abs(a - b))


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
@pytest.mark.parametrize("shape", [(34, 14, 3, 0), (40, 18, 3, 12), (60, 24, 4, 0), (52, 21, 8, 0)])
@pytest.mark.parametrize("grid", [2, 0])
def test_chain_pairs_equal_single_steps(shape, storage, grid, tmp_path):
    inst, plan = _inst(shape, tmp_path)
    given = np.random.default_rng(6).integers(0, 2, size=(3, inst.N)).astype(np.int8)
    print(shape, storage, grid, flush=True)
    with gs.Engine(plan, storage) as e:
        e.set_grid_log2(grid)
        two = e.chain(given)
        one_by_one = [e.chain(g) for g in given]
        e.set_pairs(False)
        one = e.chain(given)
    assert np.array_equal(two[2], one[2])                   # the tables are the same, bit for bit
    assert np.max(np.abs(two[0] - one[0])) < 1e-11
    assert np.allclose(two[1], one[1], rtol=1e-12, atol=0)
    for j in range(3):
        assert np.array_equal(two[j], np.concatenate([r[j] for r in one_by_one]))
