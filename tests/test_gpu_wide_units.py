"""Sweeps of several steps where no small run and no LDS score takes their place: batches of plans of at least 2^16 slots, and
engines with small runs off.  Each batch has strings of probability zero (a row of M is zeroed, in the plateau, after the
first comparison), whose bookkeeping the sweeps do themselves.

Tables between the steps are rounded as single steps round them, so amplitudes are equal bit for bit; norms and gradients are
FP64 sums over up to 2^20 terms in another order: 2^20 x 2^-53 = 1.2e-10 relative at worst, far less for sums taken in trees,
so 1e-11 as in the tests of the narrower plans.  Sampled and forced complex64 strings of 2^20 entries and more keep 1e-9."""
import numpy as np
import pytest

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu

# (n, band, seed, gadgets), lanes: widths 16 to 19; a plateau alone, one-output steps, like and unlike plans side by side
BATCHES = [
    [((44, 18, 1, 0), 64)],
    [((40, 19, 6, 10), 64)],
    [((46, 18, 2, 0), 64), ((46, 18, 2, 0), 128)],
    [((46, 19, 5, 0), 128), ((43, 18, 9, 0), 64), ((24, 10, 1, 0), 64)],
]


def _close(a, b, tol):
    fin = np.isfinite(a)
    return np.array_equal(fin, np.isfinite(b)) and np.allclose(np.asarray(a)[fin], np.asarray(b)[fin], rtol=tol, atol=tol)


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
@pytest.mark.parametrize("batch", BATCHES, ids=range(len(BATCHES)))
def test_wide_batches_equal_single_steps(batch, storage, tmp_path):
    plans, bits, dead = [], [], []
    rng = np.random.default_rng(29)
    for i, ((n, band, seed, gadgets), lanes) in enumerate(batch):
        inst = egs.instances.Instance(n, band, seed, gadgets_count=gadgets)
        plans.append(str(tmp_path / f"p{i}.txt"))
        inst.write_plan(plans[-1])
        bits.append(rng.integers(0, 2, size=(lanes, inst.N)).astype(np.int8))
        M = np.array([inst.am.M[v] for v in inst.step_vertices])
        M[inst.N // 2, 1] = 0                               # bit 1 there: probability zero from that step on
        dead.append(M)
    print(batch, storage, flush=True)
    with gs.BatchEngine(plans, [lanes for _, lanes in batch], storage=storage) as bt:
        got = []
        for zero in (False, True):
            for i, M in enumerate(dead if zero else []):
                bt.set_matrices(i, M)
            for on in (True, False):
                bt.set_pairs(on)
                got.append((bt.score(bits), bt.grad(bits)[0]))
    for (many, gmany), (one, gone) in ((got[0], got[1]), (got[2], got[3])):
        for i in range(len(batch)):
            assert np.array_equal(many[2][i], one[2][i])
            assert _close(many[0][i], one[0][i], 1e-11) and _close(gmany[i][0], gone[i][0], 1e-11)
            assert np.allclose(many[1][i], one[1][i], rtol=1e-11, atol=0)
            assert np.array_equal(gmany[i][1], gone[i][1])
            assert np.max(np.abs(gmany[i][2] - gone[i][2])) <= 1e-11 * np.max(np.abs(gone[i][2]))
    for i, b in enumerate(bits):
        at = batch[i][0][0] + batch[i][0][3]
        gone_at = b[:, at // 2] == 1
        assert np.array_equal(np.isneginf(got[2][0][0][i]), gone_at)
        assert np.all(got[2][0][2][i][gone_at] == 0) and np.all(got[2][0][1][i][gone_at, at // 2:] == 0)


# one string's steps of a few blocks and of many, gadget plans; width 24 takes two steps per write in complex128
ENGINES = [(34, 14, 3, 0), (40, 18, 3, 12), (60, 24, 4, 0), (70, 26, 3, 0)]


@pytest.mark.parametrize("storage,tol", [(gs.C64, 1e-9), (gs.C128, 1e-12)])
@pytest.mark.parametrize("shape", ENGINES)
def test_dead_strings_on_wide_sweeps(shape, storage, tol, tmp_path):
    """Strings that die in the plateau beside strings that do not, small runs off: several strings per launch and several
    steps per sweep against one string and one step at a time."""
    n, band, seed, gadgets = shape
    inst = egs.instances.Instance(n, band, seed, gadgets_count=gadgets)
    d = int(np.argmax([s["r"] for s in inst.steps])) + 2
    v = inst.step_vertices[d]
    inst.am.M[v] = np.array(inst.am.M[v])
    inst.am.M[v][1] = 0
    plan = str(tmp_path / "p.txt")
    inst.write_plan(plan)
    given = np.random.default_rng(41).integers(0, 2, size=(6, inst.N)).astype(np.int8)
    given[:, :gadgets] = 0
    given[:, d] = [1, 0, 1, 0, 0, 1]
    part = given.copy()
    part[:, d + 1:] = -1
    free = given.copy()
    free[:, :d] = -1                                          # the steps up to the dead one sampled, then forced
    print(shape, storage, flush=True)
    with gs.Engine(plan, storage) as e, gs.Engine(plan, storage) as one:
        for x in (e, one):
            x.set_small_steps(-1)
        one.set_pairs(False)
        many = (e.prob(given), *e.chain(given), *e.hybrid(part, 2), *e.hybrid(free, 2))
        each = [(one.prob(g), *one.chain(g), *one.hybrid(p, 2, i), *one.hybrid(f, 2, i))
                for i, (g, p, f) in enumerate(zip(given, part, free))]
    gone = given[:, d] == 1
    for j, a in enumerate(many):
        b = np.concatenate([r[j] for r in each])
        if a.dtype == np.int8:
            assert np.array_equal(a, b), j
        elif a.dtype == complex:
            assert np.array_equal(a, b) and np.all(a[gone] == 0) and np.all(a[~gone] != 0)
        else:
            assert _close(a, b, tol), j
            assert np.all(np.isneginf(a[gone]) if a.ndim == 1 else a[gone, d:] == 0), j


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
def test_strings_of_one_call_on_sweeps(storage, tmp_path):
    """Plans that run as one small run by themselves, with small runs off: strings in one call are bitwise those one by one."""
    inst = egs.instances.Instance(34, 14, 3)
    plan = str(tmp_path / "p.txt")
    inst.write_plan(plan)
    given = np.random.default_rng(8).integers(0, 2, size=(33, inst.N)).astype(np.int8)
    part = given.copy()
    part[:, inst.N // 2:] = -1
    print(storage, flush=True)
    with gs.Engine(plan, storage) as e:
        e.set_small_steps(-1)
        many = (*e.sample(33, 11), e.prob(given), *e.chain(given), *e.hybrid(part, 5))
        each = [(*e.sample(1, 11, first=i), e.prob(g), *e.chain(g), *e.hybrid(p, 5, i))
                for i, (g, p) in enumerate(zip(given, part))]
    for j, a in enumerate(many):
        assert np.array_equal(a, np.concatenate([r[j] for r in each])), j
