"""Size distributions at the sizes where their passes change shape: one
particle, fewer particles than workgroups, a slice's remainder, every
particle in one bin, one bin, the largest histogram of each workgroup size
and more bins than one window.

A bin is a sum of at most n positive terms, each a few roundings from the
oracle's: the relative difference is at most (n + 32) 2^-52."""
import numpy as np
import pytest

import oracle
from helpers import gpu_boxes, radius
from partmc_amd import populations as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_part,n_bin,spread", [
    (1, 1, 1.0), (63, 16, 1.0), (513, 17, 1.0), (4000, 60, 0.0), (20011, 1, 1.0),
    (3001, 1024, 1.0), (3001, 1025, 1.0), (3001, 2048, 1.0), (3001, 2049, 1.0), (3001, 4500, 1.0)])
def test_size_dist_edges(n_part, n_bin, spread):
    rng = np.random.default_rng(n_part + n_bin)
    vol = 10 ** (-20.0 + spread * rng.uniform(-3, 3, size=(n_part, 1)))
    vol = vol * rng.dirichlet([2, 1, 1], size=n_part)
    pop = P.Population(vol=vol, density=np.array([1000.0, 1800.0, 1400.0]),
                       weight_type=P.WEIGHT_POWER, weight_magnitude=1e-12, weight_exponent=-3.0)
    g = gpu_boxes([pop], 1)
    d_min, d_max = 3e-8, 2e-6  # particles outside at both ends
    e, _, wd = oracle.bin_grid_make_log(n_bin, d_min, d_max)
    r = radius(vol)
    ref = oracle.histogram_1d(e, wd, 2.0 * r, 1e-12 * r ** -3.0)
    got = g.size_dist(0, n_bin, d_min, d_max)
    np.testing.assert_allclose(got, ref, rtol=(n_part + 32) * 2.0 ** -52, atol=0)
