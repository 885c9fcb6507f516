"""The per-step contact search at the particle counts where the number of lanes
that share a particle changes, against the force sweep that searches the cells
itself: the same contacts in the same order, so the same bits.  Packings and
gases, periodic and walled; polyhedra with spheres among them, whose search
writes the narrow phase's work list, and lists too short for most bodies."""
import numpy as np
import pytest

from pacific_amd import MIXED, workloads
from tests.helpers import make_gpu

pytestmark = pytest.mark.gpu


def compare(wl, cap, steps, precision=0):
    a = make_gpu(wl, precision=precision, skin=0.0, nbr=cap, record=False)
    b = make_gpu(wl, precision=precision, nbr=0, record=False)
    for k in steps:
        a.step(k)
        b.step(k)
        sa, sb = a.state(), b.state()
        for f in ("x", "v", "w", "q", "F", "T"):
            assert np.array_equal(sa[f], sb[f]), f
    return sa


@pytest.mark.parametrize("n", [1, 33, 1000, 32768, 32769, 49152, 49153])
@pytest.mark.parametrize("cap", [32, 3])
def test_spheres(gpu, n, cap):
    if n <= 1000:
        wl = workloads.settling_box(n, box=(0.02, 0.02, 0.3), spacing=(1.999e-3,) * 3, jitter=2e-6)
    else:
        wl = workloads.periodic_gas(n, sigma=0.6, phi=0.25)
    s = compare(wl, cap, (20, 3), MIXED if n % 2 else 0)
    assert n == 1 or np.abs(s["F"]).max() > 0


@pytest.mark.parametrize("side", [(2, 2, 2), (32, 32, 32), (33, 33, 31), (40, 40, 40), (41, 40, 40)])
@pytest.mark.parametrize("cap", [32, 4])
def test_work_list(gpu, side, cap):
    wl = workloads.polyhedra_box(side, seed=11, spheres=True, sigma=0.3)
    # touching from the start: the lattice pulled together
    wl["groups"] = [(g[0], 2.2e-3 + (g[1] - 1.9e-3) * (2.9 / 3.8)) + g[2:] for g in wl["groups"]]
    s = compare(wl, cap, (2, 1))
    touching = np.count_nonzero(np.abs(s["T"]).max(1))
    assert side == (2, 2, 2) or touching > 100, touching
