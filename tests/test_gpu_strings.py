"""Several strings per launch: every mode gives, string by string, bitwise what the same call gives one string at a
time.  The plans cover a string's sweeps of one block (n = 24), of a few blocks that finish in the kernel (n = 34), of
many blocks followed by a reduction (n = 60, 2^20 slots), and a gadget plan; the counts cover one launch, its edges and a
second chunk of strings."""
import numpy as np
import pytest

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu

PLANS = [((24, 10, 1, 0), (1, 2, 63, 65)), ((34, 13, 6, 0), (3, 33)), ((30, 12, 5, 7), (9,)), ((60, 24, 4, 0), (2, 5))]


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
@pytest.mark.parametrize("shape,counts", PLANS)
def test_strings_of_one_call_equal_one_string_calls(shape, counts, storage, tmp_path):
    n, band, seed, gadgets = shape
    inst = egs.instances.Instance(n, band, seed, gadgets_count=gadgets)
    plan = str(tmp_path / "p.txt")
    inst.write_plan(plan)
    rng = np.random.default_rng(8)
    with gs.Engine(plan, storage) as many, gs.Engine(plan, storage) as one:
        for count in counts:
            print(shape, storage, count, flush=True)
            bits, lp = many.sample(count, 11)
            ref = [one.sample(1, 11, first=i) for i in range(count)]
            assert np.array_equal(bits, np.concatenate([r[0] for r in ref]))
            assert np.array_equal(lp, np.concatenate([r[1] for r in ref]))
            given = rng.integers(0, 2, size=(count, inst.N)).astype(np.int8)
            assert np.array_equal(many.prob(given), np.concatenate([one.prob(g) for g in given]))
            lp, cond, amp = many.chain(given)
            ref = [one.chain(g) for g in given]
            for got, j in ((lp, 0), (cond, 1), (amp, 2)):
                assert np.array_equal(got, np.concatenate([r[j] for r in ref]))
            # '?' steps that change from string to string split the call into launches of like strings
            free = rng.integers(0, 4, size=count)
            for i in range(count):
                given[i, inst.N - 2 * free[i]:] = -1
            ob, lp, cond = many.hybrid(given, 5)
            ref = [one.hybrid(given[i], 5, first_line=i) for i in range(count)]
            for got, j in ((ob, 0), (lp, 1), (cond, 2)):
                assert np.array_equal(got, np.concatenate([r[j] for r in ref]))


def test_dead_strings_beside_live_ones(golden):
    """Zero-probability branches (the golden plan with a zeroed M row) among strings that are not."""
    plan = f"{golden}/zero/plan.txt"
    with gs.Engine(plan, gs.C64) as many, gs.Engine(plan, gs.C64) as one:
        given = np.random.default_rng(3).integers(0, 2, size=(40, many.ns)).astype(np.int8)
        lp, cond, amp = many.chain(given)
        ref = [one.chain(g) for g in given]
        assert np.isinf(lp).any() and np.isfinite(lp).any()
        assert np.array_equal(lp, np.concatenate([r[0] for r in ref]))
        assert np.array_equal(cond, np.concatenate([r[1] for r in ref]))
        assert np.array_equal(amp, np.concatenate([r[2] for r in ref]))
        assert np.array_equal(many.prob(given), np.concatenate([one.prob(g) for g in given]))
