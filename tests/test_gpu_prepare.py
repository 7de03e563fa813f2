"""set_bin_grid at the sizes where its passes change shape, against the
oracle's sort: one particle, segment edges (64 particles, 256 segments), a
remainder, one bin, more lists than the LDS counters hold, two classes, and
discards from none of the particles to all of them.  Lists, order, forward
bins and the particles kept are whole numbers and equal; edges are within
the two roundings of an exp."""
import numpy as np
import pytest

import oracle
from partmc_amd import CoagGPU, MAX_COMP

pytestmark = pytest.mark.gpu

WEIGHTS = ([[1, 1]], [[2.0, 3.0]], [[0.0, 0.0]])


@pytest.mark.parametrize("n,grid,max_bin", [
    (1, (10, 1e-9, 1e-5), 256), (63, (40, 1e-9, 1e-5), 256), (65, (1, 1e-9, 1e-5), 256),
    (16384, (150, 1e-9, 1e-5), 256), (16385, (150, 2e-8, 4e-7), 256),
    (40001, (100, 3e-8, 1e-7), 256), (3000, (60, 1e-4, 1e-3), 256),
    (5000, (900, 1e-9, 1e-5), 900), (5000, (900, 1e-9, 1e-5), 1600)])
def test_set_bin_grid_matches_oracle_sort(n, grid, max_bin):
    rng = np.random.default_rng(n)
    vol = 10 ** rng.uniform(-24, -19.5, size=(n, 1)) * rng.dirichlet([1, 1], size=n)
    klass = rng.integers(1, 3, size=n).astype(np.int32)
    dens = np.array([1800.0, 1000.0])
    g = CoagGPU(1, dens, max_bin=max_bin)
    g.set_weights(0, *WEIGHTS)
    g.upload(0, vol, np.arange(1, n + 1), np.ones(n), klass, capacity=n + 10)
    g.set_bin_grid(0, *grid)
    ob = oracle.Box(dens, oracle.Weights(*WEIGHTS), seed=1)
    ob.add_particles(vol, np.arange(1, n + 1), np.ones(n), klass)
    ob.sort_with_grid(*grid)
    o, d = ob.particles(), g.download(0)
    np.testing.assert_array_equal(d["id"], o["id"])
    np.testing.assert_array_equal(d["vol"], o["vol"])
    np.testing.assert_array_equal(d["klass"], o["klass"])
    np.testing.assert_array_equal(d["comp_source"], np.zeros((len(d["id"]), MAX_COMP)))
    for a, b in zip(ob.lists(), g.lists(0, 2)):
        np.testing.assert_array_equal(a, b)
    e, _, _ = g.grid(0)
    np.testing.assert_allclose(e, oracle.bin_grid_make_log(*grid)[0], rtol=1e-14, atol=0)
    assert len(g.removed(0)[0]) == 0  # discards are not logged
