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
