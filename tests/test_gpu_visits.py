"""Target visits at the species counts where their records change form: up to
four species in registers, more in private memory.  The parallel mode's box
with one species more of zero volume is the same box, so every whole number
is equal and the volumes are too."""
import numpy as np
import pytest

from partmc_amd import CoagGPU, MODE_PARALLEL, PREC_FP32_RECHECK, populations as P

pytestmark = pytest.mark.gpu


def run(n_spec, base, dens):
    pop = P.config_c2(seed=3, n_part=6000)
    vol = np.zeros((pop.n_part, n_spec))
    vol[:, :base] = pop.vol[:, :base]
    g = CoagGPU(1, np.concatenate([dens[:base], np.full(n_spec - base, 1234.0)]))
    g.set_rng(11, 0)
    g.set_weights(0, [[2]], [[pop.weight_magnitude * 30]], [[-3.0]])
    g.upload(0, vol, pop.ids(), np.ones(pop.n_part), np.ones(pop.n_part), capacity=4 * pop.n_part)
    g.set_next_id(0, pop.n_part + 1)
    g.set_bin_grid(0, *pop.grid)
    g.set_mode(MODE_PARALLEL, PREC_FP32_RECHECK, 1e-5)
    counts = [tuple(int(x[0]) for x in g.mc_coag(P.KERNEL_BROWN, 60.0)) for _ in range(4)]
    assert int(g.accel_counts()["n_coag"][0]) > 0
    return counts, g.download(0), g.removed(0)


@pytest.mark.parametrize("base", [2, 3, 4])
def test_zero_species_changes_nothing(base):
    # the added species' density lies inside the others' range, so the
    # Brownian bounds stay
    dens = np.array([1800.0, 1000.0, 1400.0, 1500.0])
    c0, d0, r0 = run(base, base, dens)
    for n_spec in (base + 1, 5, 9):
        c1, d1, r1 = run(n_spec, base, dens)
        assert c1 == c0
        for k in ("id", "group", "n_primary", "n_comp"):
            np.testing.assert_array_equal(d1[k], d0[k])
        np.testing.assert_array_equal(d1["vol"][:, :base], d0["vol"])
        for a, b in zip(r1, r0):
            np.testing.assert_array_equal(a, b)
