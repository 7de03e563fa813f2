"""The exact sweep where its speculation takes its rarer turns, against the
oracle: lists too many for LDS, a row of bins emptied while it is walked,
bins that become occupied, fewer and more pairs than a pass takes, targets
that remove sources, grow a bin or leave copies, component resampling, two
classes and two groups.  Whole numbers and list order are equal, volumes are
sums of the same doubles (relative 1e-12)."""
import numpy as np
import pytest

import oracle
from helpers import compare_state
from partmc_amd import CoagGPU, populations as P

pytestmark = pytest.mark.gpu


def boxes(n, weights, grid, seed, max_bin, n_class, decades=(-24.0, -21.0), n_primary=None):
    rng = np.random.default_rng(seed)
    vol = 10 ** rng.uniform(*decades, size=(n, 1)) * rng.dirichlet([1, 2, 1], size=n)
    klass = rng.integers(1, n_class + 1, size=n).astype(np.int32)
    group = rng.integers(1, len(weights[0]) + 1, size=n).astype(np.int32)
    dens = np.array([1800.0, 1000.0, 1400.0])
    ids = np.arange(1, n + 1)
    g = CoagGPU(1, dens, max_bin=max_bin)
    g.set_rng(seed, 0)
    g.set_weights(0, *weights)
    g.upload(0, vol, ids, group, klass, n_primary=n_primary, capacity=4 * n + 64)
    g.set_next_id(0, n + 1)
    ob = oracle.Box(dens, oracle.Weights(*weights), seed=seed)
    ob.add_particles(vol, ids, group, klass, n_primary)
    ob.next_id = n + 1
    if grid:
        g.set_bin_grid(0, *grid)
        ob.sort_with_grid(*grid)
    return ob, g


FLAT1 = ([[1]], [[4e9]], [[0.0]])
POWER1 = ([[2]], [[3e-14]], [[-3.0]])
FLAT22 = ([[1, 1], [1, 1]], [[2e9, 1e9], [1e9, 3e9]], [[0.0, 0.0], [0.0, 0.0]])


@pytest.mark.parametrize("n,weights,n_class,grid,max_bin,dt,steps", [
    (2, FLAT1, 1, (40, 1e-10, 1e-5), 256, 3000.0, 6),        # ends with one particle
    (9, FLAT1, 1, (40, 1e-10, 1e-5), 256, 800.0, 8),         # rows emptied as they are walked
    (300, FLAT1, 1, (200, 1e-10, 1e-5), 256, 60.0, 6),       # every pair of sparse bins
    (3000, FLAT1, 1, None, 256, 3.0, 5),                     # automatic grid, remade
    (400, FLAT22, 2, (60, 1e-10, 1e-5), 256, 20.0, 6),       # classes and groups
    (300, FLAT22, 2, (900, 1e-10, 1e-5), 1100, 60.0, 3),     # lists in global memory
    (3000, POWER1, 1, (150, 1e-10, 1e-5), 256, 60.0, 6),     # targets
    (3000, POWER1, 1, (30, 1e-10, 1e-5), 256, 600.0, 4)])
def test_sweep_matches_oracle(n, weights, n_class, grid, max_bin, dt, steps):
    ob, g = boxes(n, weights, grid, n, max_bin, n_class)
    total = 0
    for s in range(steps):
        os_, oc = ob.mc_coag(P.KERNEL_BROWN, dt, s)
        gs, gc = g.mc_coag(P.KERNEL_BROWN, dt)
        assert (os_, oc) == (int(gs[0]), int(gc[0])), s
        total += oc
    assert total > 0
    compare_state(ob, g, n_class=n_class)
    assert int(g.path_stats()["n_accel_pairs"][0]) == ob.n_accel


@pytest.mark.parametrize("counts", [(0, 300, 200), (300, 0, 200), (300, 200, 0), (0, 0, 400),
                                    (400, 0, 0), (0, 1, 0)])
def test_classes_without_particles_match_oracle(counts):
    """Pairs of classes of which the first, the second or both have no
    particle."""
    weights = ([[1, 1, 1]], [[2e9, 1e9, 3e9]], [[0.0, 0.0, 0.0]])
    grid = (60, 1e-10, 1e-5)
    n = sum(counts)
    rng = np.random.default_rng(n)
    vol = 10 ** rng.uniform(-24, -21, size=(n, 1)) * rng.dirichlet([1, 2, 1], size=n)
    klass = np.repeat(np.arange(1, 4), counts).astype(np.int32)
    ids, one = np.arange(1, n + 1), np.ones(n, np.int32)
    dens = np.array([1800.0, 1000.0, 1400.0])
    g = CoagGPU(1, dens)
    g.set_rng(n, 0)
    g.set_weights(0, *weights)
    g.upload(0, vol, ids, one, klass, capacity=4 * n + 64)
    g.set_next_id(0, n + 1)
    g.set_bin_grid(0, *grid)
    ob = oracle.Box(dens, oracle.Weights(*weights), seed=n)
    ob.add_particles(vol, ids, one, klass)
    ob.next_id = n + 1
    ob.sort_with_grid(*grid)
    total = 0
    for s in range(4):
        want = ob.mc_coag(P.KERNEL_BROWN, 30.0, s)
        got = g.mc_coag(P.KERNEL_BROWN, 30.0)
        assert want == (int(got[0][0]), int(got[1][0])), s
        total += want[1]
    assert total > 0 or n == 1
    compare_state(ob, g, n_class=3)
    g.close()
