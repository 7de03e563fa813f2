"""Parallel steps with a call between them that changes a box.  A step that
follows another takes over its keys, terms and tables, so each such call has
to send the next step back to them: the steps are those of a run in which
every step is preceded by a call that does so and changes nothing, bit for
bit.  A step on what the change made stale would differ: the change is large
enough to move the counts, which is asserted against a run without it."""
import numpy as np
import pytest

from helpers import gpu_boxes, small
from partmc_amd import (MODE_EXACT, MODE_PARALLEL, PREC_FP32_RECHECK, PREC_FP64, populations as P)

pytestmark = pytest.mark.gpu

N_BOX = 2


def pops():
    return [small(P.config_c2(seed=70 + b), 3000 + 500 * b) for b in range(N_BOX)]


def other_weights(g):
    t, m, e = g.weights(1)
    g.set_weights(1, t, m * 5.0, e)


def more_classes(g):
    t, m, e = g.weights(1)
    g.set_weights(1, np.tile(t, (1, 2)), np.tile(m, (1, 2)) * 3.0, np.tile(e, (1, 2)))


def new_particles(g):
    pop = small(P.config_c2(seed=99), 2000)
    one = np.ones(2000, np.int32)
    g.upload(1, pop.vol, np.arange(1, 2001), one, one)


def appended(g):
    vol = small(P.config_c2(seed=98), 900).vol
    one = np.ones(900, np.int32)
    g.append(1, vol, one, one)


def halved(g):
    for b in range(N_BOX):
        g.set_n_part_ideal(b, 900.0)
    g.rebalance()


def exact_step(g):
    g.set_mode(MODE_EXACT, PREC_FP64, 1e-5)
    g.mc_coag(P.KERNEL_BROWN, 60.0)
    g.set_mode(MODE_PARALLEL, PREC_FP32_RECHECK, 1e-5)


def precision(g):
    g.set_mode(MODE_PARALLEL, PREC_FP64, 1e-5)
    g.mc_coag(P.KERNEL_BROWN, 60.0)
    g.set_mode(MODE_PARALLEL, PREC_FP32_RECHECK, 1e-5)


def kernel_type(g):
    g.mc_coag(P.KERNEL_SEDI, 1.0)


def bigger_store(g):
    g.reserve([20000] * N_BOX)


# the change between two steps, and whether it moves the counts of the steps
# after it
CHANGES = {
    "temperature": (lambda g: g.set_env(1, 500.0, 2e4), True),
    "scale_weights": (lambda g: g.scale_weights(1, 4.0), True),
    "weights": (other_weights, True),
    "classes": (more_classes, True),
    "upload": (new_particles, True),
    "append": (appended, True),
    "dilute": (lambda g: g.dilute([0.0, 0.5]), True),
    "particle_loss": (lambda g: g.particle_loss(2, 400.0), True),
    "rebalance": (halved, True),
    "grid": (lambda g: g.set_bin_grid(1, 60, 2e-9, 2e-4), True),
    "exact step": (exact_step, True),
    "precision": (precision, True),
    "kernel": (kernel_type, True),
    "reserve": (bigger_store, False),
}


def run(change, checked):
    g = gpu_boxes(pops(), 5, capacity_factor=3)
    g.set_mode(MODE_PARALLEL, PREC_FP32_RECHECK, 1e-5)
    counts = []

    def step():
        if checked:
            for b in range(N_BOX):
                g.set_next_id(b, g.next_id(b))
        s, c = g.mc_coag(P.KERNEL_BROWN, 60.0)
        counts.append((s.tolist(), c.tolist()))

    for _ in range(2):
        step()
    if change:
        change(g)
    for _ in range(2):
        step()
    end = [{k: np.asarray(v) for k, v in g.download(b).items()} for b in range(N_BOX)]
    end += [{"id": a, "action": b, "other": c} for a, b, c in map(g.removed, range(N_BOX))]
    g.close()
    return counts, end


@pytest.fixture(scope="module")
def unchanged():
    return run(None, False)[0]


@pytest.mark.parametrize("name", sorted(CHANGES))
def test_a_change_between_steps_is_seen(name, unchanged):
    change, moves = CHANGES[name]
    c0, d0 = run(change, False)
    c1, d1 = run(change, True)
    assert c0 == c1
    for x, y in zip(d0, d1):
        assert x.keys() == y.keys()
        for k in x:
            np.testing.assert_array_equal(x[k], y[k], err_msg=k)
    assert (c0[2:] != unchanged[2:]) == moves
