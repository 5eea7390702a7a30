"""Batches of plans of different shapes, whose instances may take sweeps of their own (widest first).

Every table between sweeps is rounded as single steps round it, so the amplitudes are those of single steps bit for bit;
the norms are sums of up to 2^14 squares in another order: 2^14 x 2^-53 = 2e-12 relative at worst, far less for sums taken
in trees, so 1e-11 on log2 Pr and 1e-11 on conditionals.
"""
import numpy as np
import pytest

from _pkg import egs

pytestmark = pytest.mark.gpu

# (n, band, seed) and lanes: widths 4 to 14; shapes that share launches, single plans that leave, lanes that differ
BATCHES = [
    [((40, 16, 7), 512), ((37, 15, 8), 512), ((43, 14, 9), 512)],
    [((40, 16, 7), 256), ((40, 16, 7), 64), ((12, 4, 1), 64), ((30, 11, 3), 1024), ((24, 16, 5), 512)],
    [((44, 17, 2), 128)] + [((20 + i, 7, i), 64) for i in range(12)],
]


@pytest.mark.parametrize("storage", (0, 1), ids=("c64", "c128"))
@pytest.mark.parametrize("batch", BATCHES, ids=range(len(BATCHES)))
def test_mixed_batch_equals_single_steps(batch, storage, tmp_path):
    plans, bits = [], []
    rng = np.random.default_rng(23)
    for i, ((n, band, seed), lanes) in enumerate(batch):
        inst = egs.instances.Instance(n, band, seed)
        plans.append(str(tmp_path / f"p{i}.txt"))
        inst.write_plan(plans[-1])
        bits.append(rng.integers(0, 2, size=(lanes, inst.N)).astype(np.int8))
    print(batch, storage, flush=True)
    with egs.gsamp.BatchEngine(plans, [lanes for _, lanes in batch], storage=storage) as bt:
        own = bt.score(bits)
        bt.use_graph(True)
        again = [bt.score(bits) for _ in range(3)]
        bt.use_graph(False)
        bt.set_pairs(False)
        one = bt.score(bits)
    for i in range(len(batch)):
        assert np.array_equal(own[2][i], one[2][i])
        assert np.max(np.abs(own[0][i] - one[0][i])) < 1e-11
        assert np.allclose(own[1][i], one[1][i], rtol=1e-11, atol=0)
        for g in again:
            assert all(np.array_equal(g[j][i], own[j][i]) for j in range(3))
