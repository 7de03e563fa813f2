"""A particle's radius over the exponent range of its volume, where it is
formed without a general pow.

Under a weight r**1 and with one particle in one bin, a size distribution is
the radius over the bin's width: the radius's 1/2 ulp (a little more at
subnormal volumes) and five roundings after it, 8 * 2^-53 in all, against the
power in 80-bit arithmetic."""
import numpy as np
import pytest

from partmc_amd import CoagGPU, populations as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lo,hi", [(-307, -280), (-280, -40), (-40, -26), (-26, -18), (-18, 6),
                                   (6, 200)])
def test_radius_is_the_power(lo, hi):
    n = 24
    rng = np.random.default_rng(hi - lo)
    vol = 10.0 ** rng.uniform(lo, hi, size=n)
    d_min, d_max = 1e-110, 1e80
    width = np.longdouble(np.log(d_max)) - np.longdouble(np.log(d_min))
    g = CoagGPU(n, np.array([1000.0]))
    g.reserve([16] * n)
    got = np.zeros(n)
    for b in range(n):
        g.set_weights(b, [[P.WEIGHT_POWER]], [[1.0]], [[1.0]])
        g.upload(b, vol[b:b + 1, None], [1], [1], [1])
        got[b] = g.size_dist(b, 1, d_min, d_max)[0]
    x = 3.0 * vol / 4.0 / np.pi
    ref = x.astype(np.longdouble) ** np.longdouble(1.0 / 3.0) / width
    np.testing.assert_allclose(got.astype(np.longdouble), ref, rtol=8 * 2.0 ** -53, atol=0)


@pytest.mark.parametrize("volume", [np.inf, -np.inf])
def test_an_infinite_volume_lies_outside_every_grid(volume):
    """As its radius by pow does: the distribution is that of a box with a
    volume beyond the grid in its place, bit for bit, and a sort on an
    explicit grid discards it."""
    n = 40
    vol = 10.0 ** np.random.default_rng(3).uniform(-22, -18, size=(n, 1))
    one = np.ones(n, np.int32)
    ends = []
    for last in (1e10, volume):
        vol[-1] = last
        g = CoagGPU(1, np.array([1000.0]))
        g.set_weights(0, [[P.WEIGHT_POWER]], [[1e-12]], [[-3.0]])
        g.upload(0, vol, np.arange(1, n + 1), one, one)
        hist = g.size_dist(0, 50, 1e-9, 1e-3)
        g.set_bin_grid(0, 50, 1e-9, 1e-3)
        ends.append((hist, g.download(0)["id"]))
        g.close()
    np.testing.assert_array_equal(ends[1][0], ends[0][0])
    assert ends[0][0].sum() > 0
    np.testing.assert_array_equal(ends[1][1], ends[0][1])
    np.testing.assert_array_equal(ends[1][1], np.arange(1, n))


def test_radii_that_are_no_numbers():
    """A zero volume has radius 0 (under a weight r**1 its size distribution
    is 0, outside the grid), a negative one and a NaN the power's NaN: each is
    the only particle of its box."""
    g = CoagGPU(3, np.array([1000.0]))
    got = []
    for b, volume in enumerate((0.0, -1e-20, np.nan)):
        g.set_weights(b, [[P.WEIGHT_POWER]], [[1.0]], [[1.0]])
        g.upload(b, np.array([[volume]]), [1], [1], [1])
        got.append(g.size_dist(b, 1, 1e-9, 1e-3)[0])
    g.close()
    assert got[0] == 0.0 and np.isnan(got[1]) and np.isnan(got[2])
