"""Components through the parallel mode's merges.  Under flat weights no
particle is copied, so a component (its source and time) is in at most one
particle; a particle of at most MAX_COMP primaries holds all of them, and a
larger one MAX_COMP.  Few merges of a wavefront join their components
together, many a lane each: the cases reach both, and the resampling."""
import numpy as np
import pytest

from helpers import small
from partmc_amd import CoagGPU, MAX_COMP, MODE_PARALLEL, PREC_FP32_RECHECK, populations as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,n,dt,steps", [
    (P.KERNEL_ADDITIVE, 200, 100.0, 6), (P.KERNEL_ADDITIVE, 6000, 20.0, 4),
    (P.KERNEL_ADDITIVE, 6000, 200.0, 5), (P.KERNEL_SEDI, 20000, 30.0, 6)])
def test_components_are_conserved(kernel, n, dt, steps):
    if kernel == P.KERNEL_ADDITIVE:
        pop = P.config_c1prime(n_part=n)
    else:
        pop = small(P.config_c5(n_box=1, n_part=50000)[0], n)
        pop.weight_magnitude *= 30.0
    g = CoagGPU(1, pop.density)
    g.set_rng(5, 0)
    g.set_env(0, pop.temp, pop.pressure, pop.beta)
    g.set_weights(0, [[pop.weight_type]], [[pop.weight_magnitude]], [[pop.weight_exponent]])
    source = np.zeros((n, MAX_COMP), np.int32)
    time = np.zeros((n, MAX_COMP))
    source[:, 0] = np.arange(1, n + 1)
    time[:, 0] = 0.5 * source[:, 0]
    one = np.ones(n, np.int32)
    g.upload(0, pop.vol, pop.ids(), one, one, one, 2 * n, one, source, time)
    g.set_next_id(0, n + 1)
    g.set_mode(MODE_PARALLEL, PREC_FP32_RECHECK, 1e-5)
    coag = sum(int(g.mc_coag(kernel, dt)[1][0]) for _ in range(steps))
    d = g.download(0)
    g.close()
    assert coag > n // 50 and d["n_primary"].sum() == n
    np.testing.assert_array_equal(d["n_comp"], np.minimum(d["n_primary"], MAX_COMP))
    held = np.arange(MAX_COMP) < d["n_comp"][:, None]
    src = d["comp_source"][held]
    assert len(np.unique(src)) == len(src) and src.min() >= 1
    np.testing.assert_array_equal(d["comp_time"][held], 0.5 * src)
    assert not d["comp_source"][~held].any()
