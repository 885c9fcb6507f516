"""The one-launch step of small sphere systems against the general launches
(list rebuild, contact filter, force sweep), which a system that collects
contact statistics runs: same list, same order of the sums, so the same bits.
Sizes around a workgroup's 64 particles and the rebuild's pieces, gases fast
enough to rebuild the list many times, packings whose workgroups hold more
contacts than lanes, lists too short for their neighbours (searched in their
cells), contact memory, and the size above which the general launches run
anyway."""
import numpy as np
import pytest

from pacific_amd import MIXED, workloads
from tests.helpers import make_gpu

pytestmark = pytest.mark.gpu


def gas(n):
    return workloads.periodic_gas(n, sigma=0.6, phi=0.25)


def bed(n):
    return workloads.settling_box(n, box=(0.02, 0.02, 0.3), spacing=(1.999e-3, 1.999e-3, 1.999e-3), jitter=2e-6)


def memory(n, mur=0.0):
    wl = bed(n)
    wl["models"] = [("memory", 0, 0, 1e4, 0.8, 0.4, 2e3, -1.0, mur, 0.1, 1e-10)]
    return wl


def run(wl, precision, cap, general, steps):
    g = make_gpu(wl, precision=precision, nbr=cap, record=False, stats=general)
    for k in steps:
        g.step(k)
    return g.state(), g.neighbor_stats()[1]


@pytest.mark.parametrize("precision", [0, MIXED])
@pytest.mark.parametrize("make,n,cap", [
    (bed, 1, 32), (bed, 63, 32), (bed, 64, 32), (bed, 65, 32), (bed, 1025, 32), (bed, 1000, 3),
    (gas, 512, 32), (gas, 4097, 32), (gas, 4097, 1), (gas, 65536, 32), (gas, 65537, 32),
    (memory, 300, 32), (memory, 300, 3),
])
def test_same_bits_as_general_launches(gpu, make, n, cap, precision):
    wl = make(n)
    # batches of several steps and single steps, odd and even
    steps = (70, 1, 1, 2, 33) if n < 60000 else (40, 1)
    a, builds_a = run(wl, precision, cap, False, steps)
    b, builds_b = run(wl, precision, cap, True, steps)
    for k in ("x", "v", "w", "wb", "q", "F", "T"):
        assert np.array_equal(a[k], b[k]), k
    assert builds_a == builds_b
    if make is gas:
        assert builds_a >= 3
    if n > 1:
        assert np.abs(a["F"]).max() > 0


@pytest.mark.parametrize("precision", [0, MIXED])
@pytest.mark.parametrize("model", ["kr", "mur"])
def test_rolling_resistance(gpu, precision, model):
    # the rolling moment enters a contact's torque before the sum instead of
    # after it: one rounding (1e-16, mixed 6e-8) of the torque per contact,
    # amplified by contacts that open and close over 40 steps
    if model == "kr":
        wl = bed(500)
        wl["models"] = [(0, 0, 1e4, 0.8, 0.4, 0.02, -1.0)]
    else:
        wl = memory(500, mur=0.02)
    a, _ = run(wl, precision, 32, False, (40,))
    b, _ = run(wl, precision, 32, True, (40,))
    eps = 1e-4 if precision and model == "kr" else 1e-9
    for k in ("x", "v", "w"):
        assert np.max(np.abs(a[k] - b[k])) <= eps * np.max(np.abs(b[k])), k


def test_many_obstacles(gpu):
    # more walls than the one-launch step keeps as bits: the general launches
    wl = bed(300)
    wl["boxes"] = wl["boxes"] + [((1e-4,) * 3, (0.5e-3 + 1e-3 * (i % 19), 0.5e-3 + 1e-3 * (i // 19), 0.25), None, 5e-5, 0)
                                 for i in range(70)]
    a, _ = run(wl, 0, 32, False, (50,))
    b, _ = run(wl, 0, 32, True, (50,))
    assert np.array_equal(a["x"], b["x"]) and np.array_equal(a["F"], b["F"])
