"""The work list of the polyhedra narrow phase (a lane per distance search,
refilled) where its shape can go wrong, against the oracle: vertex counts
that are no multiple of the group a support scans, more shape classes or
vertices than a workgroup keeps in LDS, fewer bodies than lanes, and lists so
short that most bodies are searched in their cells beside it.

Pair sets equal; forces within 1e-12 of the weight plus the contact force (the
narrow phase is the oracle's bit for bit, only the order of a body's force sum
differs: a few dozen roundings of 1e-16)."""
import numpy as np
import pytest

from pacific_amd import shapes, workloads
from tests.helpers import contact_scale, make_gpu, make_oracle, pair_set, rel_force_error

pytestmark = pytest.mark.gpu


def bipyramid(k, r):
    """k-gon of circumradius r with an apex on either side: k + 2 vertices"""
    a = 2 * np.pi * np.arange(k) / k
    v = np.concatenate([np.stack([r * np.cos(a), r * np.sin(a), 0 * a], 1), [[0, 0, r], [0, 0, -r]]])
    f = [[i, (i + 1) % k, k] for i in range(k)] + [[(i + 1) % k, i, k + 1] for i in range(k)]
    return v, f


def packing(counts, side, spheres):
    """bodies of the given vertex counts in touching distance, slightly overlapping, walls beside them"""
    wl = workloads.polyhedra_box((side, side, side), seed=31, spheres=spheres, en=0.5)
    shp = [dict(kind=2, verts=v, faces=f, crust=5e-5) for v, f in (bipyramid(k - 2, 1.2e-3) for k in counts)]
    if spheres:
        shp.append(dict(kind=0, radius=1e-3, crust=5e-5))
        shp.append(dict(kind=1, L=(1.6e-3,) * 3, crust=5e-5))
    wl["shapes"] = shp
    rng = np.random.default_rng(5)
    # two bodies of circumradius 1.2 mm at 1.55 mm: most pairs are searched to
    # the end, some touch, none is deeper than the recovery can handle
    wl["groups"] = [(i % len(shp), 2e-3 + (g[1] - 1.9e-3) * (1.75 / 3.8) + rng.uniform(-2e-5, 2e-5, (1, 3))) + g[2:]
                    for i, g in enumerate(wl["groups"])]
    return wl


@pytest.mark.parametrize("counts,side,spheres,cap", [
    ([5, 6, 7], 5, False, 32),             # no whole group of vertices
    ([5, 8, 9], 5, True, 32),              # with closed forms beside the searches
    ([5, 6, 7, 8, 9, 10, 11, 12, 13], 5, False, 32),   # more classes than LDS keeps
    ([40, 41], 4, False, 32),              # more vertices than LDS keeps
    ([6, 7], 2, False, 32),                # fewer bodies than lanes
    ([5, 6, 9], 5, True, 2),               # lists too short for most bodies
])
def test_work_list_against_oracle(gpu, counts, side, spheres, cap):
    wl = packing(counts, side, spheres)
    o = make_oracle(wl)
    g = make_gpu(wl, nbr=cap)
    for steps in (0, 40):
        o.step(steps)
        g.step(steps)
        so = o.state()
        if steps:
            g.set_basis(o.basis().reshape(-1, 9))
            g.set_state(x=so["x"], v=so["v"], w=so["w"], q=so["q"], recompute=True)
            o.set_state(x=so["x"], v=so["v"], w=so["w"], q=so["q"], recompute=True)
            so = o.state()
        sg = g.state()
        po = pair_set(o.pairs())
        assert pair_set(g.pairs()) == po
        assert len(po) >= (10 if side > 2 else 0)
        scale = contact_scale(so, o.masses()[2])
        assert rel_force_error(sg["F"], so["F"], scale) <= 1e-12
        assert float(np.max(np.linalg.norm(sg["T"] - so["T"], axis=1) / (scale * 1.8e-3))) <= 1e-12
