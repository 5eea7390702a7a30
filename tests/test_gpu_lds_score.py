"""Batched scores with whole strings in LDS against one step per sweep: the same amplitudes bit for bit; log2 Pr and
conditionals to the order of FP64 sums over at most 2^14 values (1e-12).  Plans of one wave, four and eight waves a
string, the largest table that fits and the first that does not, batches of unlike plans, matrices that change, strings
of probability zero."""
import numpy as np
import pytest

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu

BATCHES = [[((6, 2, 1, 0), 64)], [((26, 9, 2, 0), 64)], [((30, 11, 3, 5), 320)], [((40, 14, 3, 0), 64)],
           [((44, 16, 5, 0), 64)], [((50, 18, 7, 0), 64)], [((24, 10, 1, 0), 64), ((9, 4, 1, 0), 192), ((33, 13, 2, 6), 128)]]


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
@pytest.mark.parametrize("batch", BATCHES)
def test_lds_scores_equal_sweeps(batch, storage, tmp_path):
    plans, bits, Ms = [], [], []
    rng = np.random.default_rng(23)
    for i, ((n, band, seed, gadgets), lanes) in enumerate(batch):
        inst = egs.instances.Instance(n, band, seed, gadgets_count=gadgets)
        plans.append(str(tmp_path / f"p{i}.txt"))
        inst.write_plan(plans[-1])
        bits.append(rng.integers(0, 2, size=(lanes, inst.N)).astype(np.int8))
        M = rng.normal(size=(inst.N, 2, 2)) + 1j * rng.normal(size=(inst.N, 2, 2))
        M[inst.N // 2, 1] = 0                               # bit 1 there: probability zero from that step on
        Ms.append(M)
    print(batch, storage, flush=True)
    with gs.BatchEngine(plans, [lanes for _, lanes in batch], storage=storage) as bt:
        got = []
        for on in (True, False):
            bt.set_pairs(on)
            got.append(bt.score(bits))
        one = got[1]
        for i, M in enumerate(Ms):
            bt.set_matrices(i, M)
        bt.set_pairs(True)
        new = bt.score(bits)
        bt.use_graph(True)
        replays = [bt.score(bits) for _ in range(3)]
        bt.use_graph(False)
        bt.set_pairs(False)
        new1 = bt.score(bits)
    for many, single in ((got[0], one), (new, new1)):
        for i in range(len(batch)):
            assert np.array_equal(many[2][i], single[2][i])
            fin = np.isfinite(single[0][i])
            assert np.array_equal(fin, np.isfinite(many[0][i]))
            assert np.allclose(many[0][i][fin], single[0][i][fin], rtol=1e-12, atol=1e-12)
            assert np.allclose(many[1][i], single[1][i], rtol=1e-12, atol=0)
    for r in replays:
        assert all(np.array_equal(r[j][i], new[j][i]) for j in range(3) for i in range(len(batch)))
    assert not all(np.isfinite(x).all() for x in new[0])
