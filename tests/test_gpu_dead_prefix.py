"""The table of a prefix of probability zero is zero, whatever earlier calls left on the device, and adds nothing to a sum
of slices.

The plans are one small run (width 7) and one with a plateau of wide steps (width 24, complex128 strings taking two steps
per write there); the branch is a step of the plateau whose row of M is zeroed.  The logscale of a dead prefix is that of
the steps before it, half the log2 of the norms 2 cond.  A sum with a live slice differs from the live slice alone by the
weight 2^(logscale - the larger one), one more rounding of every stored entry: 2^-24 or 2^-53 of its size, so 1e-6 and 1e-12
on log2 Pr and on conditionals."""
import numpy as np
import pytest

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu

PLANS = [(24, 10, 1), (70, 26, 3)]


def zeroed(shape, tmp_path, two_table=False, step=2):
    """Instance, dead step, its plan as it is and with bit 1 of the dead step impossible."""
    n, band, seed = shape
    inst = egs.instances.Instance(n, band, seed)
    d = int(np.argmax([s["r"] for s in inst.steps])) + step
    write = (lambda p: egs.engine.write_sampler_plan(p, inst.am)) if two_table else inst.write_plan
    live, dead = str(tmp_path / "live.txt"), str(tmp_path / "dead.txt")
    write(live)
    v = inst.step_vertices[d]
    inst.am.M[v] = np.array(inst.am.M[v])
    inst.am.M[v][1] = 0
    write(dead)
    return inst, d, live, dead


@pytest.mark.parametrize("storage,tol", [(gs.C64, 1e-6), (gs.C128, 1e-12)])
@pytest.mark.parametrize("shape", PLANS)
def test_dead_prefix_is_a_zero_table(shape, storage, tol, tmp_path):
    inst, d, live, dead = zeroed(shape, tmp_path)
    rng = np.random.default_rng(12)
    bits = rng.integers(0, 2, size=inst.N).astype(np.int8)
    bits[d] = 1
    other = bits.copy()
    other[d] = 0
    last = None
    with gs.Engine(dead, storage) as e:
        cond = e.hybrid(bits, 0)[2][0]
        assert np.all(cond[:d] > 0) and np.all(cond[d:] == 0)
        scale = 0.5 * np.sum(np.log2(2 * cond[:d]))
        for K in (d + 1, d + 2, d + 3, d + 6, inst.N):
            print(shape, storage, K, flush=True)
            assert np.any(e.prefix(other, K)[0])              # fills the arena
            tab, _, _, ls, lp = e.prefix(bits, K)
            assert not np.any(tab) and lp == -np.inf and abs(ls - scale) < 1e-9
            if K == d + 3:
                last = tab, ls
    K = d + 3
    with gs.Engine(live, storage) as e:
        tab, _, _, ls, _ = e.prefix(bits, K)
        alone = e.resume(bits, K, [tab], [ls], 1)
        both = e.resume(bits, K, [last[0], tab], [last[1], ls], 1)
    assert abs(alone[1] - both[1]) < tol and abs(alone[2] - both[2]) < tol
    assert np.max(np.abs(alone[3] - both[3])) < tol
