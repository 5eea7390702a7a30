"""Two-table engine, strings that meet a branch of probability zero: the table of such a prefix is zero and so is the
amplitude, whatever the two tables held before (the steps behind the branch do not run)."""
import numpy as np
import pytest

from _pkg import egs
from test_gpu_dead_prefix import zeroed

gs = egs.gsamp
pytestmark = pytest.mark.gpu

PLANS = [(24, 10, 1), (52, 21, 8)]
STEPS = [2, 3]              # an even and an odd number of steps behind the branch: either table is the last one's


def strings(inst, d):
    bits = np.random.default_rng(12).integers(0, 2, size=inst.N).astype(np.int8)
    bits[d] = 1
    other = bits.copy()
    other[d] = 0
    return bits, other


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
@pytest.mark.parametrize("shape", PLANS)
@pytest.mark.parametrize("step", STEPS)
def test_dead_prefix_is_a_zero_table(shape, step, storage, tmp_path):
    inst, d, _, dead = zeroed(shape, tmp_path, two_table=True, step=step)
    bits, other = strings(inst, d)
    with gs.TwoTableEngine(dead, storage=storage) as e:
        for K in (d + 1, d + 2, d + 3, inst.N):
            print(shape, step, storage, K, flush=True)
            assert np.any(e.prefix(other, K)[0])
            tab, _, ls, lp = e.prefix(bits, K)
            assert not np.any(tab) and lp == -np.inf and np.isfinite(ls)


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
@pytest.mark.parametrize("shape", PLANS)
@pytest.mark.parametrize("step", STEPS)
def test_dead_string_has_no_amplitude(shape, step, storage, tmp_path):
    inst, d, _, dead = zeroed(shape, tmp_path, two_table=True, step=step)
    bits, other = strings(inst, d)
    print(shape, step, storage, flush=True)
    with gs.TwoTableEngine(dead, storage=storage) as e:
        lp, cond, amp = e.chain(np.array([other, bits, other]))
    assert np.isfinite(lp[0]) and lp[1] == -np.inf and lp[2] == lp[0]
    assert np.all(cond[1, d:] == 0)
    assert amp[1] == 0 and amp[0] != 0 and amp[0] == amp[2]
