"""Particles to and from a box at the sizes where a workgroup's or a chunk's
share of the transfer ends: every field comes back as it went, absent fields
as their defaults, and components past a particle's count as zero."""
import time

import numpy as np
import pytest
import torch

from partmc_amd import CoagGPU, MAX_COMP, load, populations as P
from helpers import gpu_boxes, small

pytestmark = pytest.mark.gpu

PART = 1 << 20  # bytes of a chunk


def records(n, ns, seed):
    rng = np.random.default_rng(seed)
    nco = rng.integers(1, MAX_COMP + 1, n).astype(np.int32)
    return dict(vol=rng.uniform(1e-24, 1e-20, (n, ns)), id=rng.permutation(n).astype(np.int64) + 1,
                group=np.ones(n, np.int32), klass=np.ones(n, np.int32),
                n_primary=rng.integers(1, 99, n).astype(np.int32), n_comp=nco,
                comp_source=rng.integers(0, 9, (n, MAX_COMP)).astype(np.int32),
                comp_time=rng.uniform(0, 9, (n, MAX_COMP)), least=rng.uniform(0, 1, n),
                greatest=rng.uniform(1, 2, n))


def sizes(record):
    chunk = PART // record
    return [1, 127, 128, 129, chunk - 1, chunk, chunk + 1, 4 * chunk + 1, 5 * chunk]


@pytest.mark.parametrize("ns", [1, 4, 32])
def test_whole_records(ns):
    g = CoagGPU(2, np.linspace(1000.0, 1800.0, ns))
    for n in sizes(8 * ns + 8 + 16 + 4 * 4 + 12 * MAX_COMP):
        want = records(n, ns, n)
        for b in range(2):  # the second box's slots begin where the first's end
            g.upload(b, want["vol"], want["id"], want["group"], want["klass"], want["n_primary"],
                     0, want["n_comp"], want["comp_source"], want["comp_time"], want["least"],
                     want["greatest"])
        kept = np.arange(MAX_COMP) < want["n_comp"][:, None]
        want["comp_source"] = np.where(kept, want["comp_source"], 0)
        want["comp_time"] = np.where(kept, want["comp_time"], 0.0)
        for b in range(2):
            got = g.download(b)
            for k, v in want.items():
                np.testing.assert_array_equal(got[k], v, err_msg=f"{n} {k}")
    g.close()


@pytest.mark.parametrize("ns", [1, 20])
def test_defaults_and_part_of_the_fields(ns):
    g = CoagGPU(1, np.linspace(1000.0, 1800.0, ns))
    for n in sizes(8 * ns + 8 + 8):
        want = records(n, ns, n)
        g.upload(0, want["vol"], want["id"], want["group"], want["klass"])
        ids, vol = g.download_ids_vols(0)
        np.testing.assert_array_equal(ids, want["id"])
        np.testing.assert_array_equal(vol, want["vol"])
    got = g.download(0)
    assert (got["n_primary"] == 1).all() and (got["n_comp"] == 1).all()
    for k in ("comp_source", "comp_time", "least", "greatest"):
        assert not got[k].any()
    g.close()


def test_a_long_removal_log():
    n = 4 * PART // 20 + 1000  # more records than the ring holds
    pop = P.config_c1prime(n_part=n)
    pop.grid = None
    g = gpu_boxes([pop], 3, capacity_factor=1)
    g.dilute([1.0])
    ids, action, other = g.removed(0)
    np.testing.assert_array_equal(ids, np.arange(n, 0, -1))
    assert (action == 1).all() and not other.any()
    g.close()


def test_scaled_weights_and_ids():
    pop = small(P.config_c2(), 300)
    g = gpu_boxes([pop, pop], 3)
    g.scale_weights(1, 0.3)
    assert g.weights(0)[1][0, 0] == pop.weight_magnitude
    assert g.weights(1)[1][0, 0] == pop.weight_magnitude * 0.3
    g.set_next_id(1, 777)
    assert (g.next_id(0), g.next_id(1)) == (301, 777)
    g.close()


def mapped_bytes():
    """Address space of this process that the device's driver maps."""
    total = 0
    with open("/proc/self/maps") as f:
        for line in f:
            if "/dev/dri/" in line:
                lo, hi = line.split()[0].split("-")
                total += int(hi, 16) - int(lo, 16)
    return total


def test_a_handle_pins_its_ring_with_the_first_particles():
    """Handles that move no particles hold no ring: each grows by one when its
    first particle arrives, in slots that are there already."""
    handles = [CoagGPU(1, np.array([1000.0])) for _ in range(4)]
    for g in handles:
        g.reserve([16])
        g.sync()
    before = mapped_bytes()
    for g in handles:
        g.upload(0, np.array([[1e-20]]), [1], [1], [1])
        g.sync()
    grown = mapped_bytes() - before
    for g in handles:
        np.testing.assert_array_equal(g.download(0)["id"], [1])
        g.close()
    assert grown >= len(handles) * 4 * PART


def test_whole_records_go_up_at_the_rate_of_a_copy():
    """Records with their components (240 of 296 bytes each here) from pinned
    arrays of the caller's take less than twice a plain copy of as many bytes:
    the least of seven."""
    n = 200000
    host = dict(vol=torch.rand((n, 1), dtype=torch.float64, pin_memory=True))
    for k, t in (("id", torch.int64), ("group", torch.int32), ("klass", torch.int32),
                 ("n_primary", torch.int32), ("n_comp", torch.int32)):
        host[k] = torch.ones(n, dtype=t, pin_memory=True)
    host["comp_source"] = torch.zeros((n, MAX_COMP), dtype=torch.int32, pin_memory=True)
    host["comp_time"] = torch.zeros((n, MAX_COMP), dtype=torch.float64, pin_memory=True)
    for k in ("least", "greatest"):
        host[k] = torch.zeros(n, dtype=torch.float64, pin_memory=True)
    g = CoagGPU(1, np.array([1000.0]))
    g.reserve([n])
    at = [x.data_ptr() for x in host.values()]

    def upload():
        assert load().pmc_gpu_upload(g._h, 0, n, 0, *at) == 0
        g.sync()

    plain = torch.zeros(sum(x.nbytes for x in host.values()), dtype=torch.uint8, pin_memory=True)
    device = torch.empty_like(plain, device="cuda")

    def copy():
        device.copy_(plain, non_blocking=True)
        torch.cuda.synchronize()

    def least(f):
        times = []
        for _ in range(7):
            t = time.perf_counter()
            f()
            times.append(time.perf_counter() - t)
        return min(times)

    a, b = least(upload), least(copy)
    g.close()
    assert a < 2.0 * b, (a, b)
