"""A box after a call that failed: once its particles are replaced, it steps
as a box that never saw the failing call.  Whole numbers and list order are
the oracle's (the parallel mode's: a fresh handle's, bit for bit), volumes are
sums of the same doubles (relative 1e-12)."""
import numpy as np
import pytest

from helpers import compare_state, oracle_box, small
from partmc_amd import (CoagError, CoagGPU, MODE_PARALLEL, PREC_FP32_RECHECK, PREC_FP64,
                        populations as P)

pytestmark = pytest.mark.gpu

BAD_CLASS = 233133947  # weight class out of range


def make_pop():
    """5000 Brownian particles without a grid of their own."""
    pop = small(P.config_c2(), 5000)
    pop.grid = None
    return pop


def make_gpu(pop):
    n = pop.n_part
    g = CoagGPU(1, pop.density)
    g.reserve([3 * n])
    g.set_rng(11, 0)
    g.set_env(0, pop.temp, pop.pressure, pop.beta)
    g.set_weights(0, [[pop.weight_type]], [[pop.weight_magnitude]], [[pop.weight_exponent]])
    return g


def put(g, pop, klass):
    n = pop.n_part
    one = np.ones(n, np.int32)
    g.upload(0, pop.vol, pop.ids(), one, np.full(n, klass, np.int32))
    g.set_next_id(0, n + 1)


def steps_as_the_oracle(g, pop, steps=3, dt=60.0):
    ob = oracle_box(pop, 11)
    total = 0
    for s in range(steps):
        want = ob.mc_coag(P.KERNEL_BROWN, dt, s)
        got = g.mc_coag(P.KERNEL_BROWN, dt)
        assert want == (int(got[0][0]), int(got[1][0])), s
        total += want[1]
    assert total > 0
    compare_state(ob, g)


# the population's radii span 8e-9 to 4e-5 m: grids that leave particles
# outside below, above, on both sides, and all of them
@pytest.mark.parametrize("grid", [(40, 5e-8, 1e-3), (40, 1e-10, 5e-8), (10, 4e-8, 6e-8),
                                  (10, 1e-3, 1e-2)])
def test_a_failed_set_bin_grid_leaves_no_request(grid):
    pop = make_pop()
    g = make_gpu(pop)
    put(g, pop, 2)  # one class is set
    with pytest.raises(CoagError) as e:
        g.set_bin_grid(0, 10, 4e-8, 6e-3)  # fails on the class
    assert e.value.code == BAD_CLASS
    with pytest.raises(CoagError) as e:
        g.set_bin_grid(0, *grid)  # the box holds that error
    assert e.value.code == BAD_CLASS
    put(g, pop, 1)
    steps_as_the_oracle(g, pop)
    g.close()


def fail_a_step(g, pop):
    """A step that makes the box's grid and then fails on the class, so that
    the majorants and pair tables of the new grid are not computed."""
    put(g, pop, 2)
    with pytest.raises(CoagError) as e:
        g.mc_coag(P.KERNEL_BROWN, 60.0)
    assert e.value.code == BAD_CLASS


def test_a_failed_exact_step_leaves_no_tables():
    pop = make_pop()
    g = make_gpu(pop)
    fail_a_step(g, pop)
    put(g, pop, 1)
    g.set_rng(11, 0)
    steps_as_the_oracle(g, pop)
    g.close()


@pytest.mark.parametrize("precision", [PREC_FP64, PREC_FP32_RECHECK])
def test_a_failed_parallel_step_leaves_no_tables(precision):
    pop = make_pop()
    ends = []
    for fail in (False, True):
        g = make_gpu(pop)
        g.set_mode(MODE_PARALLEL, precision, 1e-5)
        if fail:
            fail_a_step(g, pop)
        put(g, pop, 1)
        g.set_rng(11, 0)
        counts = [tuple(int(x[0]) for x in g.mc_coag(P.KERNEL_BROWN, 60.0)) for _ in range(3)]
        ends.append((counts, g.download(0)))
        g.close()
    assert ends[0][0] == ends[1][0] and ends[0][0][0][1] > 0
    for k, v in ends[0][1].items():
        np.testing.assert_array_equal(ends[1][1][k], v, err_msg=k)


CAPACITY = 3  # particle, list or grid capacity exceeded


def power_pop(n, seed):
    """Particles whose weights make merges keep their parents, so that a step
    appends many."""
    rng = np.random.default_rng(seed)
    vol = 10 ** rng.uniform(-24, -20, size=(n, 1)) * rng.dirichlet([1, 1], size=n)
    return P.Population(vol=vol, density=np.array([1800.0, 1000.0]), weight_type=P.WEIGHT_POWER,
                        weight_magnitude=1e-14, weight_exponent=-3.0)


def flat_pop(n, seed, weight):
    """Larger particles under a flat weight: each merge is one particle less."""
    pop = power_pop(n, seed)
    pop.vol = pop.vol * 1e6
    pop.weight_type, pop.weight_magnitude, pop.weight_exponent = P.WEIGHT_NONE, weight, 0.0
    return pop


def parallel_boxes(pops, room):
    g = CoagGPU(len(pops), pops[0].density)
    g.reserve([p.n_part + r for p, r in zip(pops, room)])
    g.set_rng(3, 0)
    for b, p in enumerate(pops):
        g.load_population(b, p)
    g.set_mode(MODE_PARALLEL, PREC_FP32_RECHECK, 1e-5)
    return g


@pytest.mark.parametrize("n,kernel,dt,flat", [(300, P.KERNEL_CONSTANT, 60.0, 2e6),
                                              (3000, P.KERNEL_BROWN, 600.0, 5e7)])
@pytest.mark.parametrize("room", [0, 1, 40])
def test_a_parallel_step_beyond_the_capacity(n, kernel, dt, flat, room):
    """A box that runs out of slots ends with its error, within its slots.  The
    box whose slots follow conserves its particles (volumes in sums of n
    terms, n 2^-52), and the full one is as a new handle's with its next
    particles, which are larger, so that both make their grid anew."""
    full, other = power_pop(n, 1), flat_pop(n, 2, flat)
    g = parallel_boxes([full, other], [room, 0])
    with pytest.raises(CoagError) as e:
        g.mc_coag(kernel, dt)
    assert e.value.code == CAPACITY
    assert g.n_part(0) <= n + room
    assert np.isfinite(g.download(0)["vol"]).all()
    d, merges = g.download(1), int(g.counters()["n_coag"][1])
    assert merges > 0 and len(d["id"]) == n - merges == len(np.unique(d["id"]))
    assert d["n_primary"].sum() == n
    np.testing.assert_allclose(d["vol"].sum(axis=0), other.vol.sum(axis=0), rtol=n * 2.0 ** -52,
                               atol=0)
    new = parallel_boxes([flat_pop(n, 5, flat), other], [room, 0])
    g.load_population(0, flat_pop(n, 5, flat))
    ends = []
    for h in (g, new):
        h.set_rng(7, 0)
        ends.append(([int(x[0]) for x in h.mc_coag(kernel, dt)], h.download(0)))
        h.close()
    assert ends[0][0] == ends[1][0] and ends[0][0][1] > 0
    for k, v in ends[0][1].items():
        np.testing.assert_array_equal(ends[1][1][k], v, err_msg=k)


# a parent with fewer primaries than components
BAD_PRIMARIES = (465791384, 465791385)


@pytest.mark.parametrize("share", [0.002, 0.02, 0.3])
def test_a_target_event_that_fails_leaves_no_claims(share):
    """Power weights, where targets sample sources and remove some of them: an
    event that meets a particle without primaries fails with claims on the
    sources it took before.  The box goes on with larger particles (a new
    grid) as a new handle does."""
    pop = small(P.config_c2(), 3000)
    pop.weight_magnitude *= 30.0
    pop.grid = None
    n = pop.n_part
    one = np.ones(n, np.int32)

    def new_handle():
        g = make_gpu(pop)
        g.reserve([60 * n])
        g.set_mode(MODE_PARALLEL, PREC_FP32_RECHECK, 1e-5)
        return g

    g = new_handle()
    primaries = np.where(np.random.default_rng(4).uniform(size=n) < share, 0, 1).astype(np.int32)
    g.upload(0, pop.vol, pop.ids(), one, one, n_primary=primaries)
    g.set_next_id(0, n + 1)
    with pytest.raises(CoagError) as e:
        for _ in range(4):
            g.mc_coag(P.KERNEL_BROWN, 60.0)
    assert e.value.code in BAD_PRIMARIES
    ends = []
    for h in (g, new_handle()):
        h.set_weights(0, [[pop.weight_type]], [[pop.weight_magnitude * 1e3]],
                      [[pop.weight_exponent]])
        h.upload(0, pop.vol * 1e3, pop.ids(), one, one)
        h.set_next_id(0, n + 1)
        h.set_rng(7, 0)
        counts = [tuple(int(x[0]) for x in h.mc_coag(P.KERNEL_BROWN, 100.0)) for _ in range(3)]
        ends.append((counts, h.download(0)))
        assert int(h.accel_counts()["n_coag"][0]) > 0
        h.close()
    assert ends[0][0] == ends[1][0]
    for k, v in ends[0][1].items():
        np.testing.assert_array_equal(ends[1][1][k], v, err_msg=k)


@pytest.mark.parametrize("n_box,mean", [(1, 5e9), (3, 1.9e9)])
def test_more_tests_than_a_step_can_number(n_box, mean):
    """All particles in the middle one of three bins: more tests than a pair's
    draw holds, and pairs of which each can be drawn but whose sum passes 32
    bits.  Neither makes a test; the boxes then step as a new handle's with
    other particles."""
    n, flat = 2000, 2e6
    k_max = 2.0 * 0.25 / (60.0 * 2e8)  # the constant kernel's majorant, over-estimated by 2
    dt = mean / (k_max * flat * n * (n - 1) / 2)
    pops = [flat_pop(n, 20 + b, flat) for b in range(n_box)]
    g = parallel_boxes(pops, [64] * n_box)
    for b in range(n_box):
        g.set_bin_grid(b, 3, 1e-10, 1e-1)
    with pytest.raises(CoagError) as e:
        g.mc_coag(P.KERNEL_CONSTANT, dt)
    assert e.value.code == CAPACITY
    # smaller particles, so that both make their grid anew
    new = parallel_boxes(pops, [64] * n_box)
    ends = []
    for h in (g, new):
        for b, p in enumerate(pops):
            p.vol = flat_pop(n, 20 + b, flat).vol * 1e-12
            h.load_population(b, p)
        h.set_rng(7, 0)
        ends.append(([x.tolist() for x in h.mc_coag(P.KERNEL_CONSTANT, 6.0)],
                     [h.download(b) for b in range(n_box)]))
        h.close()
    assert ends[0][0] == ends[1][0] and min(ends[0][0][1]) > 0
    for x, y in zip(ends[0][1], ends[1][1]):
        for k, v in x.items():
            np.testing.assert_array_equal(y[k], v, err_msg=k)


def test_step_lists_across_a_new_class_count():
    """The lists of the last step end with the class count they were made for:
    asking for them before the next step is an error, and the next step's are
    the particles' counts."""
    pops = [flat_pop(400, 30 + b, 2e6) for b in range(3)]
    g = parallel_boxes(pops, [64] * 3)
    g.mc_coag(P.KERNEL_CONSTANT, 6.0)
    assert g.step_lists(2).sum() == 400
    for b in range(3):
        g.set_weights(b, [[1, 1, 1]], [[2e6, 2e6, 2e6]], [[0.0, 0.0, 0.0]])
    for b in range(3):
        with pytest.raises(CoagError):
            g.step_lists(b, 3)
    left = [g.n_part(b) for b in range(3)]
    g.mc_coag(P.KERNEL_CONSTANT, 6.0)
    for b in range(3):
        counts = g.step_lists(b, 3)
        assert counts.sum() == left[b]
    g.close()
