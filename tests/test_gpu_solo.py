"""The one-launch step of small sphere systems against the general launches
(list rebuild, contact filter, force sweep), which a system that collects
contact statistics runs: same list, same order of the sums, so the same bits.
Sizes around a workgroup's 64 particles and the rebuild's pieces, gases fast
enough to rebuild the list many times, packings whose workgroups hold more
contacts than lanes, lists too short for their neighbours (searched in their
cells), contact memory, and the size above which the general launches run
anyway."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from pacific_amd import GrainsError, MIXED, workloads
from tests.helpers import contact_scale, make_gpu, make_oracle, pair_set, rel_force_error

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
    # more walls than the one-launch step keeps as bits: the general launches.
    # The six that are touched come last, behind 70 that are not
    wl = bed(300)
    wl["boxes"] = [((1e-4,) * 3, (0.5e-3 + 1e-3 * (i % 19), 0.5e-3 + 1e-3 * (i // 19), 0.25), None, 5e-5, 0)
                   for i in range(70)] + wl["boxes"]
    g, o = make_gpu(wl), make_oracle(wl)
    touched = set()
    for k in (0, 1, 49):
        g.step(k)
        o.step(k)
        po = pair_set(o.pairs())
        assert pair_set(g.pairs()) == po
        touched |= {-b - 1 for _, b in po if b < 0}
        scale = contact_scale(o.state(), o.masses()[2])
        if k < 2:
            assert rel_force_error(g.state()["F"], o.state()["F"], scale) <= 1e-12
    assert len(touched) >= 4 and min(touched) >= 70
    a, _ = run(wl, 0, 32, False, (50,))
    b, _ = run(wl, 0, 32, True, (50,))
    assert np.array_equal(a["x"], b["x"]) and np.array_equal(a["F"], b["F"])


# laws of the material pairs (particles 0 and 1, walls 2); some with memory,
# the others without: only the former have an entry in a particle's memory
LAWS = {
    "walls without": {(0, 0): 1, (0, 1): 1, (1, 1): 1, (0, 2): 0, (1, 2): 0},
    "walls with": {(0, 0): 0, (0, 1): 0, (1, 1): 0, (0, 2): 1, (1, 2): 1},
    "mixture": {(0, 0): 1, (0, 1): 0, (1, 1): 1, (0, 2): 1, (1, 2): 0},
}


def with_laws(wl, laws):
    wl["models"] = [("memory", a, b, 1e4, 0.8, 0.4, 2e3, -1.0, 0.0, 0.1, 1e-10) if m else
                    (a, b, 1e4, 0.8, 0.4, 0.0, -1.0) for (a, b), m in LAWS[laws].items()]
    wl["boxes"] = [(L, c, B, crust, 2) for L, c, B, crust, _ in wl["boxes"]]
    return wl


@pytest.mark.parametrize("precision", [0, MIXED])
@pytest.mark.parametrize("laws", sorted(LAWS))
def test_memory_beside_plain_laws(gpu, laws, precision):
    # contacts that open and close: against the general launches, bit for bit,
    # and in FP64 the oracle (each side of a pair evaluates its own contact
    # point: rounding, amplified over the steps as in the one-law packings)
    wl = with_laws(workloads.dense_pack(side=6, sigma=0.2, squeeze=-1e-5), laws)
    wl["material"] = (np.arange(216) % 2).astype(np.int32)
    a = make_gpu(wl, precision=precision, record=True)
    b = make_gpu(wl, precision=precision, record=True, stats=True)
    o = make_oracle(wl)
    npairs = set()
    for k in (1, 60, 139):
        a.step(k)
        b.step(k)
        o.step(k)
        sa, sb, so = a.state(), b.state(), o.state()
        for f in ("x", "v", "w", "F", "T"):
            assert np.array_equal(sa[f], sb[f]), f
        if precision == 0:
            assert pair_set(a.pairs()) == pair_set(o.pairs())
            scale = contact_scale(so, o.masses()[2])
            # positions that differ by dx change a contact's force by kn dx: six
            # neighbours, both ends, against a scale as small as the weight
            dx = np.abs(sa["x"] - so["x"]).max()
            assert dx <= 1e-13
            assert rel_force_error(sa["F"], so["F"], scale) <= 1e-9 + 12 * 1e4 * dx / scale.min()
        npairs.add(len(a.pairs()))
    assert len(npairs) > 1 and max(npairs) > 100


def test_many_plain_contacts_few_with_memory(gpu):
    # a sphere on the floor (memory) with 40 small ones around it (none): more
    # contacts than a particle keeps entries, but one entry
    i = np.arange(40) + 0.5
    th, ph = np.arccos(1 - 1.6 * i / 40), np.pi * (1 + 5 ** 0.5) * i
    R, r = 4e-3, 0.4e-3
    d = np.stack([np.cos(ph) * np.sin(th), np.sin(ph) * np.sin(th), np.cos(th)], 1)
    c = np.array([0.01, 0.01, R - 1e-6])
    wl = with_laws(workloads.settling_box(41), "mixture")
    wl["x"] = np.concatenate([[c], c + d * (R + r - 1e-6)])
    wl["radius"] = np.concatenate([[R], np.full(40, r)])
    wl["material"] = np.array([0] + [1] * 40, np.int32)
    a, b, o = make_gpu(wl, nbr=64), make_gpu(wl, nbr=64, stats=True), make_oracle(wl)
    assert len(a.pairs()) == 81 and pair_set(a.pairs()) == pair_set(o.pairs())
    for s in (a, b, o):
        s.step(30)
    for f in ("x", "v", "w", "F", "T"):
        assert np.array_equal(a.state()[f], b.state()[f]), f
    assert np.abs(a.state()["x"] - o.state()["x"]).max() <= 1e-12


@pytest.mark.parametrize("laws", [None, "mixture"])
@pytest.mark.parametrize("precision", [0, MIXED])
def test_nothing_searched_after_an_error(gpu, precision, laws):
    # one sphere too fast (more than the crust's thickness in a step): the
    # batch goes on without contacts, at a force that is the weight alone, over
    # graph replays and single steps, and reports the first error
    wl = workloads.dense_pack(side=6)
    if laws:
        with_laws(wl, laws)
    wl["v"][17] = (6.0, 0.0, 0.0)
    g = make_gpu(wl, precision=precision, record=False)
    assert np.abs(g.state()["F"] - g.masses()[2]).max() > 1e-3
    L = g._check.__globals__["lib"]()
    for k in (200, 1, 2):
        with pytest.raises(GrainsError, match="MotionError") as e:
            g.step(k)
        assert e.value.ids[0] == 18
        F = np.empty((216, 3))
        p = F.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
        L.grains_gpu_get_state(g.h, None, None, None, None, None, p, None)
        assert np.array_equal(F, g.masses()[2])


@pytest.mark.parametrize("scheme", [0, 2])
def test_general_evaluation_between_one_launch_steps(gpu, scheme):
    # force sums come from the general sweep, over the list as the steps left
    # it: current after a LeapFrog step, to be checked after an explicit one;
    # against a system that builds its list there (sums in another order)
    wl = gas(4097)
    g = make_gpu(wl, scheme=scheme, record=False)
    for k in (9, 1, 2, 9, 70):
        if scheme and k > 9:
            continue  # the explicit scheme gains energy in contacts
        g.step(k)
        a = g.force_sums()
        assert np.array_equal(a, g.force_sums())
        s = g.state()
        h = make_gpu(wl, scheme=scheme, record=False)
        h.set_state(**{f: s[f] for f in ("x", "v", "w", "q")})
        b = h.force_sums()
        assert b.max() > 0 and np.max(np.abs(a - b)) <= 1e-12 * b.max()


@pytest.mark.parametrize("precision", [0, MIXED])
@pytest.mark.parametrize("with_memory", [False, True])
def test_list_too_short_for_some(gpu, precision, with_memory):
    # large spheres among small ones: more neighbours than a list of 16 holds
    wl = memory(2000) if with_memory else bed(2000)
    big = np.arange(50, 2000, 333)
    near = np.linalg.norm(wl["x"][:, None] - wl["x"][big][None], axis=2) < 3.9e-3
    keep = ~near.any(1)
    keep[big] = True
    for k in ("radius", "density", "crust", "material", "x", "v", "w"):
        wl[k] = np.asarray(wl[k])[keep]
    wl["radius"] = np.where(np.isin(np.flatnonzero(keep), big), 2.9995e-3, 1e-3)
    wl["x"] = wl["x"] + np.array([2e-3, 2e-3, 2e-3])
    wl["max"] = (0.03, 0.03, 0.3)
    wl["boxes"] = []
    a, builds_a = run(wl, precision, 16, False, (40, 1, 2))
    b, builds_b = run(wl, precision, 16, True, (40, 1, 2))
    assert builds_a == builds_b
    for f in ("x", "v", "w", "F", "T"):
        assert np.array_equal(a[f], b[f]), f


@pytest.mark.parametrize("precision", [0, MIXED])
def test_rebuilds_often_and_seldom(gpu, precision):
    # near the size limit a system whose list goes stale often steps by the
    # general launches, as its velocities and then its rebuilds say: slow, made
    # fast from outside, slow again, over graph replays and single steps
    wl = gas(40001)
    slow = dict(wl, v=wl["v"] * 0.05)
    a, b = make_gpu(slow, precision=precision, record=False), make_gpu(slow, precision=precision, record=False, stats=True)
    for v in (None, wl["v"], slow["v"]):
        for k in (70, 1, 2, 70):
            if v is not None and k == 70:
                for s in (a, b):
                    s.set_state(v=v)
            a.step(k)
            b.step(k)
        sa, sb = a.state(), b.state()
        for f in ("x", "v", "w", "F", "T"):
            assert np.array_equal(sa[f], sb[f]), f
        assert a.neighbor_stats() == b.neighbor_stats()
    assert a.neighbor_stats()[1] > 20


@pytest.mark.parametrize("precision", [0, MIXED])
@pytest.mark.parametrize("scheme", [0, 1, 2, 3])
def test_list_builds_are_counted_as_by_general_launches(gpu, scheme, precision):
    # steps, states set and evaluations in between; a list of 8 entries takes
    # the general launches, which rebuild right after the drift (after an
    # explicit step also where a state set next builds it again: left out)
    wl = gas(700)
    a = make_gpu(wl, scheme=scheme, precision=precision, record=False)
    b = make_gpu(wl, scheme=scheme, precision=precision, record=False, nbr=8)
    rng = np.random.default_rng(scheme)
    for k in range(24):
        op, m = int(rng.integers(0, 5)), int(rng.choice([1, 2, 5]))
        for g in (a, b):
            g.step(m)
            if op == 1:
                g.compute_forces()
            if op == 2:
                g.force_sums()
            if op == 3 and scheme == 0:
                s = g.state()
                g.set_state(x=s["x"], v=0.9 * s["v"], recompute=bool(k % 2))
        assert a.neighbor_stats() == b.neighbor_stats(), k
        if k % 3 == 0:
            sa, sb = a.state(), b.state()
            for f in ("x", "v", "w", "F", "T"):
                assert np.array_equal(sa[f], sb[f]), (k, f)
    assert a.neighbor_stats()[1] > 5


def test_systems_stepping_at_once(gpu):
    # one-launch steps with rebuilds of several systems on their own streams,
    # from four threads: the same bits as one after the other
    sizes = (700, 4097, 8000, 20000)

    def work(n):
        g = make_gpu(gas(n), precision=MIXED if n == 8000 else 0, record=False)
        for k in (1, 70, 2, 70):
            g.step(k)
        return g.state(), g.neighbor_stats()

    alone = [work(n) for n in sizes]
    with ThreadPoolExecutor(4) as pool:
        together = list(pool.map(work, sizes))
    for (a, na), (b, nb) in zip(alone, together):
        assert na == nb and na[1] >= 3
        for f in ("x", "v", "w", "F", "T"):
            assert np.array_equal(a[f], b[f]), f
