"""Plans of 2^12 to 2^14 slots on an engine as it is made, which runs them as one small run with steps of up to 2^13 cosets,
against one sweep per step: the same bits and chain-mode amplitudes, and log2 Pr and conditionals to the order of their FP64
sums (a scale's last bit now and then moves the rounding of a stored value: 2e-6 in complex64, 1e-12 in complex128, as for
runs of fewer cosets).  A limit of 10 is the setting an engine is made with."""
import numpy as np
import pytest

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu

PLANS = [(34, 14, 3), (36, 15, 2), (40, 16, 7)]               # widths 12, 13 and 14


def _plan(shape, tmp_path):
    inst = egs.instances.Instance(*shape)
    path = str(tmp_path / "p.txt")
    inst.write_plan(path)
    return inst, path


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
@pytest.mark.parametrize("shape", PLANS)
def test_default_engine_equals_single_sweeps(shape, storage, tmp_path):
    inst, plan = _plan(shape, tmp_path)
    rng = np.random.default_rng(5)
    given = rng.integers(0, 2, size=(5, inst.N)).astype(np.int8)
    part = given.copy()
    part[:, inst.N // 3:] = -1
    K = inst.N // 2
    rest = np.concatenate([given[0][:K], np.full(inst.N - K, -1, np.int8)])
    print(shape, storage, flush=True)
    got = []
    with gs.Engine(plan, storage) as made, gs.Engine(plan, storage) as sweeps:
        sweeps.set_small_steps(-1)
        sweeps.set_pairs(False)
        for e in (made, sweeps):
            pre = e.prefix(given[0], K)
            got.append((*e.sample(3, 9), e.prob(given), *e.chain(given), *e.hybrid(part, 2), pre[0], np.array(pre[3:]),
                        *e.resume(rest, K, [pre[0]], [pre[3]], 4)))
    tol = 1e-12 if storage == gs.C128 else 2e-6
    for a, b in zip(*got):
        a, b = np.asarray(a), np.asarray(b)
        if a.dtype == np.int8:
            assert np.array_equal(a, b)
        else:
            assert np.allclose(a, b, rtol=tol, atol=tol * 1e-3), np.max(np.abs(a - b))
    assert np.array_equal(got[0][5], got[1][5])


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
def test_limit_ten_restores_the_default(storage, tmp_path):
    inst, plan = _plan((34, 14, 3), tmp_path)
    given = np.random.default_rng(7).integers(0, 2, size=(2, inst.N)).astype(np.int8)
    print(storage, flush=True)

    def sweeps_and_results(e):
        e.profile(True)
        got = e.prob(given)
        return int(e.profile_read()[1].sum()), got

    with gs.Engine(plan, storage) as e:
        made = sweeps_and_results(e)
        e.set_small_steps(-1)
        off = sweeps_and_results(e)
        e.set_small_steps(10)
        again = sweeps_and_results(e)
    assert made[0] == 0 and off[0] > 0
    assert again[0] == made[0] and np.array_equal(again[1], made[1])
