"""Parallel steps that follow one another: a step after another starts from
the keys, terms and tables the last one left, a step after a call that may
have changed a box checks them again, and a box that outgrows its grid sends
the step back to the keys.  All three give the same bits."""
import numpy as np
import pytest

from helpers import gpu_boxes, small
from partmc_amd import MODE_PARALLEL, PREC_FP32_RECHECK, populations as P

pytestmark = pytest.mark.gpu


def state(g, n_box):
    return [{k: np.asarray(v) for k, v in g.download(b).items()} for b in range(n_box)]


def assert_same(a, b):
    for x, y in zip(a, b):
        assert x.keys() == y.keys()
        for k in x:
            np.testing.assert_array_equal(x[k], y[k], err_msg=k)


def run(pops, kernel, dt, n, touch):
    g = gpu_boxes(pops, 5)
    g.set_mode(MODE_PARALLEL, PREC_FP32_RECHECK, 1e-5)
    out = []
    edges = []
    for i in range(n):
        if touch:
            # a call that leaves a box as it is, but not known to be so
            for b in range(len(pops)):
                g.set_next_id(b, g.next_id(b))
        s, c = g.mc_coag(kernel, dt)
        out.append((s.tolist(), c.tolist()))
        edges.append(tuple(g.grid(b)[0][-1] for b in range(len(pops))))
    d = state(g, len(pops))
    g.close()
    return out, edges, d


@pytest.mark.parametrize("kernel,n_part,n_box,dt", [
    (P.KERNEL_ADDITIVE, 700, 1, 400.0), (P.KERNEL_ADDITIVE, 5000, 3, 400.0),
    (P.KERNEL_BROWN, 3000, 2, 600.0)])
def test_chained_steps_equal_checked_steps(kernel, n_part, n_box, dt):
    make = (lambda s: P.config_c1prime(seed=s, n_part=n_part)) if kernel == P.KERNEL_ADDITIVE \
        else (lambda s: small(P.config_c2(seed=s), n_part))
    pops = [make(40 + b) for b in range(n_box)]
    if kernel == P.KERNEL_ADDITIVE:
        for p in pops:
            p.grid = (70, 1e-8, 1e-4)  # outgrown by particles of a third of its last edge
    o0, e0, d0 = run(pops, kernel, dt, 8, False)
    o1, e1, d1 = run(pops, kernel, dt, 8, True)
    assert o0 == o1 and e0 == e1
    assert_same(d0, d1)
    if kernel == P.KERNEL_ADDITIVE:
        # a box outgrew its grid in a step that followed another
        assert any(x != y for x, y in zip(e0[1:], e0[:-1]))


@pytest.mark.parametrize("others", [1, 7])
def test_box_alone_equals_box_among_many_holes(others):
    """The holes of all boxes are sorted together, few of them in one
    workgroup: box 0 ends the same however many the others have."""
    mine = P.config_c1prime(seed=9, n_part=1500)
    rest = [P.config_c1prime(seed=10 + b, n_part=4000) for b in range(others)]
    a, _, d0 = run([mine], P.KERNEL_ADDITIVE, 100.0, 3, False)
    b, _, d1 = run([mine] + rest, P.KERNEL_ADDITIVE, 100.0, 3, False)
    assert [(s[0], c[0]) for s, c in a] == [(s[0], c[0]) for s, c in b]
    assert_same(d0, d1[:1])
    if others == 7:
        assert max(sum(c) for _, c in b) > 2048  # two holes a merge of the flat weighting
