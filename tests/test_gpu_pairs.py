"""Two steps per sweep in the batched engine against one step per sweep: scores, conditionals, amplitudes and gradients.
Amplitudes are equal bitwise in the forward pass (the table between the steps is rounded in registers as it would be
in memory); norms and gradients are FP64 sums over up to 2^(width) cosets in another order, so they agree to 1e-12
relative (2^14 terms x 2^-53, with room)."""
import numpy as np
import pytest

from _pkg import egs

gs = egs.gsamp
pytestmark = pytest.mark.gpu

BATCHES = [
    [((9, 4, 1, 0), 64)],                                   # a few cosets: ranges shorter than a wave's
    [((24, 10, 1, 0), 128)],
    [((30, 12, 5, 7), 64)],                                 # gadget plan: one-output steps
    [((40, 18, 3, 12), 64)],                                # gadget plan, all slot counts on both sides
    [((37, 15, 9, 0), 192)],
    [((24, 10, 1, 0), 64), ((24, 10, 1, 0), 128)],          # like steps in both instances
    [((24, 10, 1, 0), 64), ((29, 9, 4, 0), 64), ((13, 5, 2, 3), 64)],   # unlike ones, of different lengths
]


@pytest.mark.parametrize("storage", [gs.C64, gs.C128])
@pytest.mark.parametrize("batch", BATCHES)
def test_pairs_equal_single_steps(batch, storage, tmp_path):
    plans, bits = [], []
    rng = np.random.default_rng(17)
    for i, ((n, band, seed, gadgets), lanes) in enumerate(batch):
        inst = egs.instances.Instance(n, band, seed, gadgets_count=gadgets)
        plans.append(str(tmp_path / f"p{i}.txt"))
        inst.write_plan(plans[-1])
        bits.append(rng.integers(0, 2, size=(lanes, inst.N)).astype(np.int8))
    print(batch, storage, flush=True)
    with gs.BatchEngine(plans, [lanes for _, lanes in batch], storage=storage) as bt:
        two = bt.score(bits)
        gtwo, _ = bt.grad(bits)
        gseg, _ = bt.grad(bits, seg=3)
        bt.set_pairs(False)
        one = bt.score(bits)
        gone, _ = bt.grad(bits)
        bt.set_pairs(True)
        bt.use_graph(True)
        again = [bt.score(bits) for _ in range(3)]
    for i in range(len(batch)):
        assert np.array_equal(two[2][i], one[2][i])
        assert np.max(np.abs(two[0][i] - one[0][i])) < 1e-11
        assert np.allclose(two[1][i], one[1][i], rtol=1e-12, atol=0)
        for g in again:
            assert all(np.array_equal(g[j][i], two[j][i]) for j in range(3))
        scale = np.max(np.abs(gone[i][2]))
        assert np.max(np.abs(gtwo[i][2] - gone[i][2])) < 1e-12 * scale
        assert np.array_equal(gtwo[i][2], gseg[i][2]) and np.array_equal(gtwo[i][1], gseg[i][1])
