"""The time step of large sphere systems (more than one launch can hold) against
the general sweep, which a system that collects contact statistics runs: same
lists, same order of the sums, so the same bits.  Packings with walls and
weight, a last tile that is not full, uniform crust and coupling factor and
not, both precisions, every scheme; a gas with a touch list, just above the
size at which it is kept, with batches that end in a half kick, with a list
too short for its neighbours (searched in their cells) and with as many
particles in contact, later or from the start, as the list is not used for."""
import numpy as np
import pytest

from pacific_amd import MIXED, workloads
from tests.helpers import make_gpu

pytestmark = pytest.mark.gpu


def uneven(wl):
    rng = np.random.default_rng(8)
    n = len(wl["x"])
    wl["crust"] = wl["crust"] * rng.uniform(0.9, 1.0, n)
    wl["density"] = wl["density"] * rng.uniform(0.5, 1.5, n)
    wl["radius"] = wl["radius"] * rng.uniform(0.9995, 1.0, n)
    return wl


def bed():
    return workloads.dense_pack(side=41)


def uneven_bed():
    return uneven(bed())


def weighted_gas():
    wl = uneven(workloads.periodic_gas(70001, sigma=0.6, phi=0.25))
    wl["gravity"] = (0.3, 0.0, -0.2)
    return wl


def gas():
    return uneven(workloads.periodic_gas(500001, sigma=0.6, phi=0.25))


def dense_gas():
    return uneven(workloads.dense_pack(side=80, periodic=True, gravity=(0.0, 0.0, 0.0)))


def run(wl, precision, scheme, cap, general, steps):
    # (the fluid's density makes the coupling factors differ with the particles')
    g = make_gpu(wl, precision=precision, scheme=scheme, fluid_density=100.0, nbr=cap, record=False, stats=general)
    for k in steps:
        g.step(k)
    return g.state(), g.neighbor_stats()[1]


@pytest.mark.parametrize("make,scheme,precision,cap", [
    (bed, 0, 0, 32), (bed, 0, MIXED, 32), (uneven_bed, 0, 0, 32), (uneven_bed, 0, MIXED, 32), (uneven_bed, 0, 0, 3),
    (uneven_bed, 1, 0, 32), (uneven_bed, 2, 0, 32), (uneven_bed, 3, MIXED, 32), (weighted_gas, 0, 0, 32),
    (gas, 0, 0, 32), (gas, 0, MIXED, 32), (gas, 0, 0, 1), (gas, 2, 0, 32), (dense_gas, 0, 0, 32),
])
def test_same_bits_as_general_sweep(gpu, make, scheme, precision, cap):
    wl = make()
    steps = (20, 1, 7) if make in (bed, uneven_bed, dense_gas) else (40, 1, 70)
    if scheme == 1 or (make is gas and scheme == 2):
        # the explicit schemes gain energy in contacts; a particle that moves
        # by the crust's thickness in one step (4.5 m/s) is an error.  By the
        # oracle: first order, packing, 2.9 m/s after 20 steps; second order,
        # a gas of 20,000, 2.6 m/s after 10, 3.5 after 20, the error after 41
        steps = (9, 1, 2)
    a, builds_a = run(wl, precision, scheme, cap, False, steps)
    b, builds_b = run(wl, precision, scheme, cap, True, steps)
    for k in ("x", "v", "w", "wb", "q", "F", "T"):
        assert np.array_equal(a[k], b[k]), k
    assert builds_a == builds_b and np.abs(a["F"]).max() > 0
    if make is gas and scheme == 0:
        assert builds_a >= 3 and np.count_nonzero(a["F"][:, 0]) > 1000
