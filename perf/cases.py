"""Time-step workloads of the DEM library, each one pass of what a program does with it: build a system once,
then advance it and read its state.

    bed       spheres at rest on each other in a walled box (a settled packing that a run continues from)
    gas       a periodic granular gas of unequal spheres (homogeneous cooling), the headline workload
    coupled   one exchange with a fluid solver: import the fluid's forces, ten sub-steps, read the bodies back
    memory    a bed with the tangential-spring contact model
    poly      cubes, tetrahedra and icosahedra in a hopper, or in a closed box when few
    batch     an ensemble of independent walled beds of uneven sizes, advanced together
    adjoint   a differentiable rollout: spheres landing on an inclined plane, forward and backward

Every pass goes through the public binding and returns the whole state (or the rollout's gradients).  Runs go on
from pass to pass, as a simulation does.  Particles are stored in lattice order or, as after random insertion, in
random order.
"""
import math

import numpy as np
import torch

R = 1e-3
RHO = 2500.0
CRUST = 5e-5
KN = 1e4


# ---------------------------------------------------------------------------------------------------------------
# the cases

def listed():
    return [
        # the smallest call: what a fluid solver makes each of its time steps (latency and launches)
        dict(name="coupled_500", kind="coupled", n=500, steps=10, precision="fp64", order="lattice"),
        # the 1,000-sphere box of the validation runs, once it has settled
        dict(name="bed_1000", kind="bed", n=1000, steps=100, precision="fp64", order="lattice"),
        # contact memory (tangential springs), a mid-sized laboratory sample in insertion order
        dict(name="memory_5003", kind="memory", n=5003, steps=50, precision="fp64", order="random"),
        # a mid-sized gas, mixed precision, as for parameter studies
        dict(name="gas_27000_mixed", kind="gas", n=27000, steps=300, precision="mixed", order="lattice"),
        # a bed an experiment would have, mixed precision, odd size
        dict(name="bed_48611_mixed", kind="bed", n=48611, steps=50, precision="mixed", order="lattice"),
        # a large bed whose particles were inserted at random places: neighbours are far apart in memory
        dict(name="bed_200000_random", kind="bed", n=200000, steps=100, precision="fp64", order="random"),
        # the headline: a million spheres, both precisions
        dict(name="gas_1000000", kind="gas", n=1000000, steps=500, precision="fp64", order="lattice"),
        dict(name="gas_1000000_mixed", kind="gas", n=1000000, steps=500, precision="mixed", order="lattice"),
        # non-spherical bodies: a few hundred (parity-run size) and the hopper of the silo benchmark
        dict(name="poly_343", kind="poly", n=343, steps=50, precision="fp64", order="lattice"),
        dict(name="poly_200000_mixed", kind="poly", n=200000, steps=50, precision="mixed", order="lattice"),
        # an ensemble: parameter sweep over 512 boxes of 200 to 5,000 spheres
        dict(name="batch_512", kind="batch", n=512, steps=100, precision="fp64", order="lattice"),
        # calibration by gradients: forward, recomputation from checkpoints and reverse sweep
        dict(name="adjoint_20000", kind="adjoint", n=20000, steps=100, precision="fp64", order="lattice"),
    ]


RANGES = {"coupled": (100, 5000), "bed": (200, 200000), "memory": (300, 20000), "gas": (1000, 1000000),
          "poly": (60, 200000), "batch": (8, 512), "adjoint": (300, 20000)}


def draw(rng):
    kind = rng.choice(["coupled", "bed", "bed", "memory", "gas", "gas", "poly", "poly", "batch", "adjoint"])
    lo, hi = RANGES[kind]
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    steps = {"coupled": 10, "bed": rng.randint(30, 100), "memory": rng.randint(20, 50), "gas": rng.randint(60, 300),
             "poly": rng.randint(20, 50), "batch": rng.randint(30, 100), "adjoint": rng.randint(40, 100)}[kind]
    mixed = kind in ("bed", "gas", "poly", "batch") and rng.random() < 0.5
    return dict(kind=kind, n=min(max(n, lo), hi), steps=min(steps, 50) if mixed and kind in ("bed", "batch") else steps,
                precision="mixed" if mixed else "fp64",
                order=rng.choice(["lattice", "random"]) if kind in ("bed", "memory") else "lattice")


def tolerance(case):
    # Measured: the cell search's order of the contact sums against the Verlet list's after two passes, and either
    # against the 64-bit restatement below; four times the largest.  Contacts that open and close amplify rounding:
    # beds in 64 bits reach 6e-9 (6e-7 in one body); with forces in 32 bits beds and solids reach 2.4e-6 (2.2e-4),
    # a gas, whose bodies fly on between collisions, 1e-4 (5e-2).
    if case["precision"] == "fp64":
        return {"rel": 2.5e-8, "max": 2.5e-6}
    return {"rel": 4e-4, "max": 0.2} if case["kind"] == "gas" else {"rel": 1e-5, "max": 1e-3}


# ---------------------------------------------------------------------------------------------------------------
# inputs, from the case and the seed alone

def _rng(seed):
    return np.random.default_rng(0x5EED + 7919 * int(seed))


def _walls(lo, hi, thick=5e-4, over=5e-4):
    """six thin boxes (edge lengths, centre) around [lo, hi]"""
    lo, hi = np.asarray(lo, float), np.asarray(hi, float)
    out = []
    for a in (2, 0, 1):
        for side in (0, 1):
            L = hi - lo + 2 * over
            L[a] = thick
            c = (lo + hi) / 2
            c[a] = lo[a] - thick / 2 if side == 0 else hi[a] + thick / 2
            out.append((tuple(L), tuple(c), None))
    return out


def _bed(n, rng, order, en=0.9, mu=0.5):
    """Equal spheres on a cubic lattice 1 um closer than touching, jittered by more than that, so that about seven
    in ten neighbours touch; walls on every side; slow motion."""
    nx = max(1, math.ceil((n / 2.0) ** (1.0 / 3.0)))
    nz = math.ceil(n / (nx * nx))
    pitch = 2 * R - 1e-6
    i = np.arange(n)
    x = np.stack([(i % nx + 0.5) * pitch, (i // nx % nx + 0.5) * pitch, (i // (nx * nx) + 0.5) * pitch], 1)
    x += rng.uniform(-1e-6, 1e-6, x.shape)
    if order == "random":
        x = x[rng.permutation(n)]
    hi = np.array([nx * pitch, nx * pitch, nz * pitch])
    return dict(origin=(-2e-3,) * 3, max=tuple(hi + 2e-3), periodic=(0, 0, 0), gravity=(0.0, 0.0, -9.81), dt=1e-5,
                radius=np.full(n, R), x=x, v=rng.normal(0, 0.01, (n, 3)), w=rng.normal(0, 10.0, (n, 3)),
                walls=_walls(np.zeros(3), hi), kn=KN, en=en, mu=mu)


def _gas(n, rng):
    """Radii U[0.8, 1.2] mm, solid fraction 0.3, Gaussian velocities of 0.1 m/s, no gravity, triply periodic."""
    radius = rng.uniform(0.8e-3, 1.2e-3, n)
    m = math.floor(n ** (1.0 / 3.0) + 1e-9)
    mz = math.ceil(n / (m * m))
    # sites far enough apart also where the last layer is not full
    a = max((float(np.sum(4.0 / 3.0 * np.pi * radius ** 3)) / 0.3 / (m * m * mz)) ** (1.0 / 3.0), 2.41e-3)
    i = np.arange(n)
    x = np.stack([(i % m + 0.5) * a, (i // m % m + 0.5) * a, (i // (m * m) + 0.5) * a], 1)
    x += rng.uniform(-1, 1, x.shape) * 0.125 * (a - 2.4e-3)
    v = rng.normal(0.0, 0.1, (n, 3))
    return dict(origin=(0.0,) * 3, max=(m * a, m * a, mz * a), periodic=(1, 1, 1), gravity=(0.0, 0.0, 0.0), dt=1e-5, radius=radius,
                x=x, v=v - v.mean(0), w=np.zeros((n, 3)), walls=[], kn=KN, en=0.8, mu=0.3)


def _incline(n, rng):
    """Two layers of spheres thrown at 0.2 m/s onto a plate tilted by 25 degrees."""
    radius = rng.uniform(0.9e-3, 1.1e-3, n)
    per = math.ceil(n / 2)
    side = math.ceil(math.sqrt(per))
    c, s = math.cos(math.radians(25)), math.sin(math.radians(25))
    B = np.array([[c, 0, s], [0, 1, 0], [-s, 0, c]])
    i = np.arange(n)
    lay, rem = i // per, i % per
    u = (rem % side - (side - 1) / 2) * 2.3e-3
    t = (rem // side - (side - 1) / 2) * 2.3e-3
    h = 1e-3 + 2e-5 + radius + lay * 2.3e-3
    x = u[:, None] * B[:, 0] + t[:, None] * B[:, 1] + h[:, None] * B[:, 2]
    plate = side * 2.3e-3 + 10e-3
    lo, hi = x.min(0) - 10e-3, x.max(0) + 10e-3
    lo[2] = min(lo[2], -0.5 * plate * s - 10e-3)
    return dict(origin=tuple(lo), max=tuple(hi), periodic=(0, 0, 0), gravity=(0.0, 0.0, -9.81), dt=1e-5,
                radius=radius, x=x, v=-0.2 * B[:, 2] + rng.normal(0, 0.02, (n, 3)), w=np.zeros((n, 3)),
                walls=[((plate, plate, 2e-3), (0.0, 0.0, 0.0), B)], kn=KN, en=0.8, mu=0.4)


def _solids():
    """cube of 2 mm edge; regular tetrahedron and icosahedron of circumradius 1.2 mm: (vertices, triangles, edges)"""
    p = (1 + math.sqrt(5)) / 2
    cube = np.array([[a, b, c] for a in (-1, 1) for b in (-1, 1) for c in (-1, 1)], float) * 1e-3
    tet = np.array([[1, 1, 1], [1, -1, -1], [-1, 1, -1], [-1, -1, 1]], float) * (1.2e-3 / math.sqrt(3))
    ico = np.array([q for a in (-1, 1) for b in (-p, p) for q in ((a, b, 0), (0, a, b), (b, 0, a))], float)
    ico *= 1.2e-3 / math.sqrt(1 + p * p)
    out = []
    for verts, faces in ((cube, 4), (tet, 3), (ico, 3)):
        # faces of the hull: the vertices furthest along a normal
        found = {}
        for i in range(len(verts)):
            for j in range(len(verts)):
                for k in range(j):
                    nrm = np.cross(verts[j] - verts[i], verts[k] - verts[i])
                    if np.linalg.norm(nrm) < 1e-12:
                        continue
                    h = verts @ nrm
                    if h.max() - h[i] < 1e-9 * abs(h).max():
                        on = [q for q in range(len(verts)) if h.max() - h[q] < 1e-9 * abs(h).max()]
                        found[tuple(on)] = nrm / np.linalg.norm(nrm)
        ring, edges, tris = [], set(), []
        for on, nrm in sorted(found.items()):
            c = verts[list(on)].mean(0)
            e1 = verts[on[0]] - c
            ang = [math.atan2(np.dot(np.cross(e1, verts[q] - c), nrm), np.dot(e1, verts[q] - c)) for q in on]
            loop = [q for _, q in sorted(zip(ang, on))]
            ring.append(loop)
            edges |= {tuple(sorted((loop[t - 1], loop[t]))) for t in range(len(loop))}
            tris += [(loop[0], loop[t], loop[t + 1]) for t in range(1, len(loop) - 1)]
        assert all(len(f) == faces for f in ring)
        out.append((verts, ring, np.array(tris), np.array(sorted(edges))))
    return out


def _rotations(q):
    """rotation matrices of unit quaternions (x, y, z, w)"""
    x, y, z, w = q.T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)], 1).reshape(-1, 3, 3)


def _poly(n, rng):
    """Equal thirds of the three solids in rows along x, no two neighbours of one kind: the cubes nearly square to the
    rows, the others turned anyhow, every neighbour in a row moved up until their extents along x meet, give or take
    a few um, so that some touch from the start and most pairs have to be looked at; all in motion.  Few in a closed
    box, many in a hopper with a 12 mm slot and a collecting floor."""
    pitch, t = 2.45e-3, 2e-3
    hopper = n >= 20000
    m = 40 if hopper else max(3, math.ceil(n ** (1.0 / 3.0) - 1e-9))
    i = np.arange(n)
    ijk = np.stack([i % m, i // m % m, i // (m * m)], 1)
    kind = ijk.sum(1) % 3
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1)[:, None]
    q[kind == 0] = q[kind == 0] * 0.001 + np.array([0, 0, 0, 1.0])
    q /= np.linalg.norm(q, axis=1)[:, None]
    # of q and -q the one whose largest component is positive
    q *= np.sign(q[i, abs(q).argmax(1)])[:, None]
    B = _rotations(q)
    right, left = np.zeros(n), np.zeros(n)
    for k, solid in enumerate(_solids()):
        e = (B[kind == k, 0] @ solid[0].T)
        right[kind == k], left[kind == k] = e.max(1), -e.min(1)
    gap = rng.uniform(-4e-6, 2e-6, n)
    step = np.zeros(n)
    step[1:] = np.where(ijk[1:, 0] > 0, right[:-1] + left[1:] + gap[1:], 0.0)
    run = np.cumsum(step)
    row = ijk[:, 1] + m * ijk[:, 2]
    at = run - run[row * m]  # the first of each row at 0
    ends = np.minimum((row + 1) * m, n) - 1
    length = at.max()
    nz = int(ijk[-1, 2]) + 1
    side = 1.25e-3
    lo, hi = np.zeros(3), np.array([length + 3.6e-3, (m - 1) * pitch + 2 * side, (nz - 1) * pitch + 2 * side])
    x = np.stack([at + (hi[0] - at[ends]) / 2, ijk[:, 1] * pitch + side, ijk[:, 2] * pitch + side], 1)
    by = np.argsort(kind, kind="stable")  # ids by shape, as a program adds them
    walls = []
    if hopper:
        half = (hi[0] - 12e-3) / 2
        walls = [((half, hi[1] + 2 * t, t), (half / 2, hi[1] / 2, -t / 2), None),
                 ((half, hi[1] + 2 * t, t), (hi[0] - half / 2, hi[1] / 2, -t / 2), None)]
        lo[2] = -30e-3
    walls += _walls(lo, hi, t, t)
    return dict(origin=tuple(lo - 4e-3), max=tuple(hi + 4e-3), periodic=(0, 0, 0), gravity=(0.0, 0.0, -9.81), dt=5e-6,
                kind=kind[by], x=x[by], v=rng.normal(0, 0.05, (n, 3)), w=rng.normal(0, 50.0, (n, 3)),
                basis=B[by], q=q[by], walls=walls, kn=KN, en=0.6, mu=0.5)


def _members(nsys, rng):
    # the sizes are the case's, whatever the seed
    u = np.random.default_rng(nsys).uniform(math.log(200), math.log(5000), nsys)
    sizes = np.rint(np.exp(u)).astype(int)
    return [_bed(int(n), rng, "lattice", en=float(rng.uniform(0.5, 0.95)), mu=float(rng.uniform(0.1, 0.8)))
            for n in sizes]


def _inputs(case, seed):
    rng, n, kind = _rng(seed), case["n"], case["kind"]
    if kind == "batch":
        return _members(n, rng)
    if kind == "gas":
        return _gas(n, rng)
    if kind == "adjoint":
        d = _incline(n, rng)
        d["cot"] = [rng.normal(0, 1.0, (n, 3)) for _ in range(3)]
        return d
    if kind == "poly":
        return _poly(n, rng)
    d = _bed(n, rng, case["order"])
    if kind == "memory":
        d["memory"] = dict(kt=2e3, mur=0.02, etarpf=0.1, epst=1e-10)
    if kind == "coupled":
        d["fluid"] = 1000.0
        weight = RHO * 4.0 / 3.0 * math.pi * R ** 3 * 9.81
        d["hydro"] = rng.normal(0, 1.0, (n, 6)) * weight * np.array([1, 1, 1, R, R, R])
    return d


# ---------------------------------------------------------------------------------------------------------------
# the framework's side

def _system(d, precision, skin=None):
    from pacific_amd import FP64, GrainsGPU, MIXED
    g = GrainsGPU(d["origin"], d["max"], d["periodic"], 1.0, d["gravity"], d.get("fluid", 0.0), d["dt"], 0,
                  MIXED if precision == "mixed" else FP64)
    if "memory" in d:
        g.memory_contact_model(0, 0, d["kn"], d["en"], d["mu"], **d["memory"])
    else:
        g.contact_model(0, 0, d["kn"], d["en"], d["mu"])
    if "kind" in d:
        (_, _, _, _), (tv, tf, _, _), (iv, jf, _, _) = _solids()
        ids = [g.add_shape(1, L=(2e-3,) * 3, crust=CRUST), g.add_shape(2, verts=tv, faces=tf, crust=CRUST),
               g.add_shape(2, verts=iv, faces=jf, crust=CRUST)]
        for k in range(3):
            s = d["kind"] == k
            g.add_particles(ids[k], RHO, 0, d["x"][s], d["v"][s], d["w"][s], d["basis"][s].reshape(-1, 9))
    else:
        g.add_spheres(d["radius"], RHO, CRUST, 0, d["x"], d["v"], d["w"])
    for L, c, B in d["walls"]:
        g.add_box(L, c, None if B is None else np.asarray(B).ravel(), CRUST, 0)
    if skin is not None:
        g.neighbor_list(32, skin)
    return g


def prepare(case, seed):
    d = _inputs(case, seed)
    state = {"case": case}
    if case["kind"] == "batch":
        from pacific_amd import FP64, GrainsBatch, MIXED
        state["batch"] = GrainsBatch([_system(m, case["precision"]) for m in d],
                                     MIXED if case["precision"] == "mixed" else FP64)
        return state
    # the reverse sweep replays the per-step search: no Verlet skin
    g = state["system"] = _system(d, case["precision"], 0.0 if case["kind"] == "adjoint" else None)
    g.init()
    if case["kind"] == "coupled":
        state["hydro"] = d["hydro"]
    if case["kind"] == "adjoint":
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        state["in"] = [torch.tensor(d[k], device=dev) for k in ("x", "v", "w")]
        state["theta"] = torch.tensor([d["kn"], d["en"], d["mu"]], dtype=torch.float64, device=dev)
        state["cot"] = [torch.tensor(c, device=dev) for c in d["cot"]]
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        b = state["batch"]
        b.step(case["steps"])
        parts = [b.state(i) for i in range(b.nsys)]
        return {k: np.concatenate([p[k] for p in parts]) for k in ("x", "v", "w", "q", "F", "T")}
    g = state["system"]
    if case["kind"] == "adjoint":
        from pacific_amd.adjoint import rollout
        leaf = [t.detach().clone().requires_grad_(True) for t in state["in"] + [state["theta"]]]
        out = rollout(g, leaf[0], leaf[1], leaf[2], leaf[3], case["steps"], 50)
        grads = torch.autograd.grad(out, leaf, state["cot"])
        return {"out": [t.detach() for t in out], "grads": list(grads)}
    if case["kind"] == "coupled":
        g.set_hydro_ft(state["hydro"])
    g.step(case["steps"])
    return g.state()


def work(case):
    n, steps = case["n"], case["steps"]
    if case["kind"] == "batch":
        n = n * 1491  # mean of exp(U[ln 200, ln 5000])
    touching = {"gas": 0.01}.get(case["kind"], 2.0)  # contacts per body, each seen once
    if case["kind"] == "poly":
        # position, velocity, spin and quaternion read and written, shape and mass; a pair: 16 B and about six
        # iterations of the distance search
        b, f = n * (2 * 104 + 16) + 2 * n * 16, n * 400 + 2 * n * 6 * 400
    else:
        b, f = n * (2 * 104 + 16) + touching * n * 16, n * 300 + touching * n * 250
    if case["kind"] == "memory":
        b += touching * n * 2 * 80  # the springs of every contact, read and written
    if case["kind"] == "adjoint":
        # forward, recomputation of each segment and the reverse sweep with its own state of 72 B
        b, f = 3 * b + n * 144, 4 * f
    # the state handed back: 22 numbers per body
    return {"bytes": float(steps * b + 22 * 8 * n), "flops": float(steps * f)}


# ---------------------------------------------------------------------------------------------------------------
# the same time steps in plain torch, 64 bits

def exact(case, seed):
    if case["kind"] == "poly" and case["n"] > 3000:
        return None  # the brute-force polytope distances of every pair and step: minutes
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    if dev.type == "cpu" and case["n"] * case["steps"] > 2000000:
        return None
    d = _inputs(case, seed)
    if case["kind"] == "adjoint":
        sim = _Sim([d], dev)
        leaf = [t.detach().clone().requires_grad_(True) for t in (sim.x, sim.v, sim.w)]
        theta = torch.tensor([d["kn"], d["en"], d["mu"]], dtype=torch.float64, device=dev, requires_grad=True)
        sim.x, sim.v, sim.w = leaf
        sim.kn, sim.en, sim.mu = theta[0].expand(1), theta[1].expand(1), theta[2].expand(1)
        sim.start()
        sim.steps(case["steps"])
        out = [sim.x, sim.v, sim.w]
        grads = torch.autograd.grad(out, leaf + [theta], [torch.tensor(c, device=dev) for c in d["cot"]])
        return {"out": [t.detach() for t in out], "grads": list(grads)}
    sim = _Sim(d if case["kind"] == "batch" else [d], dev)
    with torch.no_grad():
        sim.start()
        if case["kind"] == "coupled":
            ft = torch.tensor(d["hydro"], device=dev)
            sim.hydro = (ft[:, :3], ft[:, 3:])
        sim.steps(case["steps"])
    out = sim.state()
    if case["kind"] == "batch":
        out.pop("wb")
    return {k: v.cpu().numpy() for k, v in out.items()}


def _cross(a, b):
    return torch.linalg.cross(a, b)


def _dot(a, b):
    return (a * b).sum(-1, keepdim=True)


def _norm(a):
    return _dot(a, a).sqrt()


def _qmul(a, b):
    v = _cross(a[:, :3], b[:, :3]) + a[:, 3:] * b[:, :3] + b[:, 3:] * a[:, :3]
    return torch.cat([v, a[:, 3:] * b[:, 3:] - _dot(a[:, :3], b[:, :3])], 1)


def _qconj(q):
    return torch.cat([-q[:, :3], q[:, 3:]], 1)


def _turn(q, u):
    """u rotated by the unit quaternion q"""
    return _qmul(_qmul(q, torch.cat([u, torch.zeros_like(u[:, :1])], 1)), _qconj(q))[:, :3]


class _Sim:
    """Kick-drift-kick steps of one or more systems, plain tensors; pairs from a list with a margin, searched again
    every `every` steps."""
    MARGIN = 3e-4
    CHUNK = 20000  # polytope pairs evaluated at a time

    def __init__(self, systems, dev):
        cat = lambda k: torch.tensor(np.concatenate([s[k] for s in systems]), device=dev)  # noqa: E731
        d = systems[0]
        self.dev, self.d, self.dt = dev, d, d["dt"]
        self.x, self.v, self.w = cat("x"), cat("v"), cat("w")
        n = len(self.x)
        self.grp = torch.tensor(np.repeat(np.arange(len(systems)), [len(s["x"]) for s in systems]), device=dev)
        self.q = torch.zeros(n, 4, dtype=torch.float64, device=dev)
        self.q[:, 3] = 1
        per = lambda k: torch.tensor([s[k] for s in systems], dtype=torch.float64, device=dev)  # noqa: E731
        self.kn, self.en, self.mu = per("kn"), per("en"), per("mu")
        self.g = torch.tensor(d["gravity"], dtype=torch.float64, device=dev)
        self.lo = torch.tensor(d["origin"], dtype=torch.float64, device=dev)
        self.L = torch.tensor(d["max"], dtype=torch.float64, device=dev) - self.lo
        self.periodic = bool(d["periodic"][0])
        self.poly = "kind" in d
        if self.poly:
            self._solid_tables()
        else:
            r = self.r = cat("radius")
            self.mass = RHO * 4.0 * math.pi * r ** 3 / 3.0
            self.inertia = RHO * 8.0 * math.pi * r ** 5 / 15.0
            # the inner face of every wall as a plane (point, normal into the domain), per system
            rows = []
            for s in systems:
                mid = np.mean(s["x"], axis=0)
                row = []
                for Lw, c, B in s["walls"]:
                    B = np.eye(3) if B is None else B
                    a = int(np.argmin(Lw))
                    nrm = np.asarray(B)[:, a] * (1.0 if np.dot(mid - c, np.asarray(B)[:, a]) > 0 else -1.0)
                    row.append(np.concatenate([np.asarray(c) + nrm * Lw[a] / 2, nrm]))
                rows.append(np.reshape(row, (-1, 6)))
            self.planes = torch.tensor(np.stack(rows), device=dev)
        buoy = 1 - d.get("fluid", 0.0) / RHO
        self.weight = (self.mass * buoy)[:, None] * self.g
        self.m_eff, self.i_eff = (self.mass * buoy)[:, None], (self.inertia * buoy)[:, None]
        self.hydro = None
        self.springs = {}
        # steps over which nobody crosses half the margin, with room for acceleration
        self.every = max(1, int(0.5 * self.MARGIN / (1.5 * float(self.v.norm(dim=1).max()) * self.dt + 1e-9)))

    # --- pairs closer than the contact distance plus the margin, i < j
    def search(self):
        with torch.no_grad():
            reach = 2 * float(self.r.max()) + self.MARGIN
            x = self.x.detach() - self.lo
            nc = torch.clamp((self.L / reach).floor().long(), min=1)
            if not self.periodic:  # systems of a batch differ in size: one grid wide enough for all
                nc = torch.clamp((x.amax(0) / reach).floor().long() + 1, min=1)
            size = self.L / nc if self.periodic else torch.full((3,), reach, dtype=torch.float64, device=self.dev)
            c = torch.minimum((x / size).floor().long().clamp(min=0), nc - 1)
            key = lambda cc: ((self.grp * nc[1] + cc[:, 1]) * nc[2] + cc[:, 2]) * nc[0] + cc[:, 0]  # noqa: E731
            skey, order = key(c).sort()
            me = torch.arange(len(x), device=self.dev)
            got = []
            for o in range(27):
                cc = c + torch.tensor([o % 3 - 1, o // 3 % 3 - 1, o // 9 - 1], device=self.dev)
                ok = torch.ones_like(me, dtype=torch.bool)
                if self.periodic:
                    cc = cc % nc
                else:
                    ok = ((cc >= 0) & (cc < nc)).all(1)
                k = torch.where(ok, key(cc), torch.full_like(me, -1))
                b, e = torch.searchsorted(skey, k), torch.searchsorted(skey, k, right=True)
                for t in range(int((e - b).max())):
                    has = (b + t < e) & ok
                    i, j = me[has], order[(b + t)[has]]
                    keep = i < j
                    i, j = i[keep], j[keep]
                    near = _norm(self._apart(i, j))[:, 0] < self.r[i] + self.r[j] + self.MARGIN
                    got.append(torch.stack([i[near], j[near]]))
            ij = torch.cat(got, 1)
            # with fewer than three cells on a periodic axis a pair is met more than once
            code = torch.unique(ij[0] * len(x) + ij[1])
            self.i, self.j = code // len(x), code % len(x)

    def _apart(self, i, j):
        a = self.x[j] - self.x[i]
        if self.periodic:
            a = a - self.L * (a.detach() / self.L).round()
        return a

    # --- contact law: force on body 0 of a contact at lever l0 with overlap vector ov
    def law(self, ov, tv, m0, m1, grp, spring=None):
        kn, en, mu = self.kn[grp][:, None], self.en[grp][:, None], self.mu[grp][:, None]
        ln = en.log()
        beta = ln / (math.pi ** 2 + ln * ln).sqrt()
        nrm = ov / _norm(ov)
        vn = nrm * _dot(tv, nrm)
        vt = tv - vn
        ms = (1.0 / (1.0 / m0 + 1.0 / m1))[:, None]
        gn = -2.0 * beta * (ms * kn).sqrt()
        fn = kn * ov - gn * vn
        nfn = _norm(fn)
        gt = -2.0 * beta * (kn / ms).sqrt() * ms
        ft = -gt * vt
        if spring is None:
            vt2 = _dot(vt, vt)
            nvt = torch.where(vt2 > 1e-20, vt2, torch.ones_like(vt2)).sqrt()
            slip = mu * nfn < gt * nvt * (vt2 > 1e-20)
            return fn + torch.where(slip, -mu * nfn * vt / nvt, ft), None
        return self._spring_law(nrm, vt, fn, nfn, gn, gt, ft, mu, kn, spring)

    def _spring_law(self, nrm, vt, fn, nfn, gn, gt, ft, mu, kn, spring):
        """tangential and rolling springs: kd, previous normal, rolling torque of each contact, updated in place"""
        p = self.d["memory"]
        old, kd, pn, sr, wrel, req = spring
        # rotation taking the previous normal to this one
        re = _norm(pn) * _norm(nrm) + _dot(pn, nrm)
        qv = _cross(pn, nrm)
        s = 1.0 / (_dot(qv, qv) + re * re).sqrt()
        rot = torch.cat([qv * s, re * s], 1)
        kd = torch.where(old, _turn(rot, kd), torch.zeros_like(kd)) + self.dt * p["kt"] * vt
        sr = torch.where(old, _turn(rot, sr), torch.zeros_like(sr))
        nvt, a = _norm(vt), kd + gt * vt
        na = _norm(a)
        stuck = ((_norm(kd) > p["epst"]) | (_norm(gt * vt) > p["epst"])) & (na > p["epst"])
        t = torch.where(nvt > 1e-3, -vt / nvt, torch.where(stuck, -a / na, torch.zeros_like(a)))
        size = _norm(-kd + ft)
        slip = size > mu * nfn
        tang = torch.where(slip, mu * nfn * t, size * t)
        kd = torch.where(slip, (-mu * nfn * t + ft) / p["kt"], kd)
        kr = 3.0 * kn * p["mur"] ** 2 * req ** 2
        sr = sr - kr * self.dt * wrel
        most, nsr = p["mur"] * req * nfn, _norm(sr)
        sr = torch.where(nsr > most, sr * most / nsr, sr)
        roll = sr - p["etarpf"] * 3.0 * gn * p["mur"] ** 2 * req ** 2 * wrel
        return fn + tang, (kd, nrm, sr, roll)

    def _with_springs(self, key, touch, wrel, req):
        if "memory" not in self.d:
            return None
        n = len(self.i) if key == "pairs" else len(self.x)
        if key not in self.springs:
            z = lambda: torch.zeros(n, 3, dtype=torch.float64, device=self.dev)  # noqa: E731
            self.springs[key] = [torch.zeros(n, 1, dtype=torch.bool, device=self.dev), z(), z(), z()]
        old, kd, pn, sr = self.springs[key]
        return (old[touch], kd[touch], pn[touch], sr[touch], wrel, req)

    def _keep_springs(self, key, touch, got):
        if got is None:
            return
        s = self.springs[key]
        s[0] = torch.zeros_like(s[0])
        s[0][touch] = True
        for k in range(3):
            s[k + 1] = torch.zeros_like(s[k + 1]).index_put((touch,), got[k])

    # --- forces and torques at the present state
    def forces(self):
        F, T = self.weight.clone(), torch.zeros_like(self.weight)
        contacts = self._poly_contacts() if self.poly else self._sphere_contacts()
        for key, touch, i, j, l0, l1, ov in contacts:
            wi = self.w[i]
            wj = self.w[j] if j is not None else torch.zeros_like(wi)
            tv = self.v[i] + _cross(wi, l0)
            if j is not None:
                tv = tv - self.v[j] - _cross(wj, l1)
            m1 = self.mass[j] if j is not None else torch.full_like(self.mass[i], 1e20)
            spring = None
            if not self.poly and "memory" in self.d:
                r1 = self.r[j] if j is not None else self.wall_req[key][i]
                spring = self._with_springs(key, touch, wi - wj, (1 / (1 / self.r[i] + 1 / r1))[:, None])
            f, got = self.law(ov, tv, self.mass[i], m1, self.grp[i], spring)
            self._keep_springs(key, touch, got)
            roll = got[3] if got is not None else 0.0
            F = F.index_add(0, i, f)
            T = T.index_add(0, i, _cross(l0, f) + roll)
            if j is not None:
                F = F.index_add(0, j, -f)
                T = T.index_add(0, j, _cross(l1, -f) - roll)
        if self.hydro is not None:
            F, T = F + self.hydro[0], T + self.hydro[1]
        self.F, self.T = F, T

    def _sphere_contacts(self):
        out = []
        ab = self._apart(self.i, self.j)
        d = ab.norm(dim=1) - (self.r[self.i] + self.r[self.j])
        touch = (d < 0).nonzero()[:, 0]
        i, j, ab, d = self.i[touch], self.j[touch], ab[touch], d[touch][:, None]
        u = ab / _norm(ab)
        out.append(("pairs", touch, i, j, (self.r[i][:, None] + 0.5 * d) * u, -(self.r[j][:, None] + 0.5 * d) * u,
                    d * u))
        self.wall_req = {}
        for k in range(self.planes.shape[1]):
            pl = self.planes[self.grp, k]
            nrm = pl[:, 3:]
            d = _dot(self.x - pl[:, :3], nrm)[:, 0] - self.r
            i = (d < 0).nonzero()[:, 0]
            if "memory" in self.d:
                Lw = self.d["walls"][k][0]
                self.wall_req["wall%d" % k] = torch.full_like(self.r, (0.75 / math.pi * Lw[0] * Lw[1] * Lw[2])
                                                              ** (1 / 3))
            u, dd = -nrm[i], d[i][:, None]
            out.append(("wall%d" % k, i, i, None, (self.r[i][:, None] + 0.5 * dd) * u, None, dd * u))
        return out

    # --- polytopes
    def _solid_tables(self):
        d, dev = self.d, self.dev
        t = lambda a: torch.tensor(np.asarray(a), device=dev)  # noqa: E731
        solids = _solids()
        pad = lambda a, m: np.concatenate([a, np.repeat(a[:1], m - len(a), 0)])  # noqa: E731
        shapes = [(s[0], s[2], s[3], abs(s[0]).max(0)) for s in solids]
        for Lw, _, _ in d["walls"]:
            shapes.append((solids[0][0] / 1e-3 * np.asarray(Lw) / 2, solids[0][2], solids[0][3], np.asarray(Lw) / 2))
        # vertices pulled in by the crust, axis by axis
        self.verts = t(np.stack([pad(s[0] * ((s[3] - CRUST) / s[3]), 12) for s in shapes]))
        self.tris, self.edges = t(np.stack([pad(s[1], 20) for s in shapes])), t(np.stack([pad(s[2], 30) for s in shapes]))
        self.ext = t(np.stack([s[3] for s in shapes]))
        self.kind = t(d["kind"]).long()
        circ = t([math.sqrt(3) * 1e-3, 1.2e-3, 1.2e-3])
        edge = [2e-3, 1.2e-3 / math.sqrt(3 / 8), 1.2e-3 / math.sin(2 * math.pi / 5)]
        phi = (1 + math.sqrt(5)) / 2
        vol = [edge[0] ** 3, edge[1] ** 3 / (6 * math.sqrt(2)), 5 * (3 + math.sqrt(5)) / 12 * edge[2] ** 3]
        per = [edge[0] ** 2 / 6, edge[1] ** 2 / 20, phi ** 2 * edge[2] ** 2 / 10]  # inertia over mass
        self.r = circ[self.kind]
        self.mass = RHO * t(vol)[self.kind]
        self.inertia = self.mass * t(per)[self.kind]
        self.q = t(d["q"])
        self.wall_c = t(np.stack([c for _, c, _ in d["walls"]]))

    def _world(self, who):
        """points of bodies (i >= 0) or walls (-1 - k) in the frame of the world, relative to the first's centre"""
        body = who.clamp(min=0)
        wall = (-1 - who).clamp(min=0)
        isw = (who < 0)[:, None]
        shape = torch.where(who < 0, 3 + wall, self.kind[body])
        cen = torch.where(isw, self.wall_c[wall], self.x[body])
        v = self.verts[shape]
        q = self.q[body][:, None].expand(-1, 12, -1).reshape(-1, 4)
        turned = _turn(q, v.reshape(-1, 3)).reshape(v.shape)
        return torch.where(isw[:, :, None], v, turned) + cen[:, None], shape

    def _poly_contacts(self):
        near = _norm(self._apart(self.i, self.j))[:, 0] < self.r[self.i] + self.r[self.j]
        a, b = [self.i[near]], [self.j[near]]
        for k in range(len(self.wall_c)):
            hit = ((self.x - self.wall_c[k]).abs() <= self.ext[3 + k] + self.r[:, None]).all(1).nonzero()[:, 0]
            a.append(hit)
            b.append(torch.full_like(hit, -1 - k))
        a, b = torch.cat(a), torch.cat(b)
        got = [self._closest(a[s:s + self.CHUNK], b[s:s + self.CHUNK]) for s in range(0, len(a), self.CHUNK)]
        pa, pb = torch.cat([g[0] for g in got]), torch.cat([g[1] for g in got])
        ba = pa - pb
        dist = _norm(ba)
        ov = ba / dist * (2 * CRUST - dist)
        touch = dist[:, 0] < 2 * CRUST
        out = []
        for walls in (False, True):
            s = (touch & ((b < 0) == walls)).nonzero()[:, 0]
            P = (pa[s] + pb[s]) / 2
            i = a[s]
            j = None if walls else b[s]
            out.append(("poly", s, i, j, P - self.x[i], None if walls else P - self.x[b[s]], ov[s]))
        return out

    def _closest(self, a, b):
        """closest points of two disjoint polytopes: vertices against triangles, edges against edges"""
        va, sa = self._world(a)
        vb, sb = self._world(b)
        m = torch.arange(len(a), device=self.dev)[:, None]
        cand = []
        for first, (p, pv, ps) in ((True, (va, vb, sb)), (False, (vb, va, sa))):
            tri = pv[m[:, :, None], self.tris[ps]]
            pt = p[:, :, None].expand(-1, -1, 20, -1).reshape(-1, 3)
            on = _on_triangle(pt, *[tri[:, None, :, c].expand(-1, 12, -1, -1).reshape(-1, 3) for c in range(3)])
            pt, on = pt.reshape(len(a), -1, 3), on.reshape(len(a), -1, 3)
            cand.append((pt, on) if first else (on, pt))
        ea, eb = va[m[:, :, None], self.edges[sa]], vb[m[:, :, None], self.edges[sb]]
        ea, eb = ea[:, :, None].expand(-1, -1, 30, -1, -1), eb[:, None].expand(-1, 30, -1, -1, -1)
        s, t = _on_segments(ea.reshape(-1, 2, 3), eb.reshape(-1, 2, 3))
        cand.append((s.reshape(len(a), -1, 3), t.reshape(len(a), -1, 3)))
        pa, pb = torch.cat([c[0] for c in cand], 1), torch.cat([c[1] for c in cand], 1)
        k = (pa - pb).square().sum(2).argmin(1)
        return pa[m[:, 0], k], pb[m[:, 0], k]

    # --- time
    def start(self):
        # the evaluation that primes the integrator is also the first that the springs see
        self.since = 0
        self.search()
        self.forces()

    def kick(self):
        h = 0.5 * self.dt
        self.v = self.v + self.F / self.m_eff * h
        self.w = self.w + self.T / self.i_eff * h

    def steps(self, count):
        for _ in range(count):
            self.kick()
            x = self.x + self.v * self.dt
            if self.periodic:
                low, high = (x < self.lo).double(), (x >= self.lo + self.L).double()
                x = x + self.L * (low - high)
            self.x = x
            with torch.no_grad():
                nw = _norm(self.w)
                half = 0.5 * nw * self.dt
                turn = torch.cat([torch.where(nw > 1e-10, half.sin() / nw.clamp(min=1e-30), 0 * nw) * self.w,
                                  half.cos()], 1)
                self.q = _qmul(turn, self.q)
            self.since += 1
            if self.since >= self.every and "memory" not in self.d:
                self.search()
                self.since = 0
            self.forces()
            self.kick()

    def state(self):
        return {"x": self.x, "v": self.v, "w": self.w, "wb": _turn(_qconj(self.q), self.w), "F": self.F, "T": self.T,
                "q": self.q}


def _on_triangle(p, a, b, c):
    """the point of triangle a b c closest to p"""
    ab, ac, ap = b - a, c - a, p - a
    d1, d2 = _dot(ab, ap), _dot(ac, ap)
    d3, d4 = _dot(ab, p - b), _dot(ac, p - b)
    d5, d6 = _dot(ab, p - c), _dot(ac, p - c)
    va, vb, vc = d3 * d6 - d5 * d4, d5 * d2 - d1 * d6, d1 * d4 - d3 * d2
    den = va + vb + vc
    den = torch.where(den == 0, torch.ones_like(den), den)
    out = a + ab * (vb / den) + ac * (vc / den)
    unit = lambda n, m: (n / torch.where(m == 0, torch.ones_like(m), m)).clamp(0, 1)  # noqa: E731
    out = torch.where((va <= 0) & (d4 - d3 >= 0) & (d5 - d6 >= 0), b + (c - b) * unit(d4 - d3, (d4 - d3) + (d5 - d6)),
                      out)
    out = torch.where((vb <= 0) & (d2 >= 0) & (d6 <= 0), a + ac * unit(d2, d2 - d6), out)
    out = torch.where((vc <= 0) & (d1 >= 0) & (d3 <= 0), a + ab * unit(d1, d1 - d3), out)
    out = torch.where((d6 >= 0) & (d5 <= d6), c, out)
    out = torch.where((d3 >= 0) & (d4 <= d3), b, out)
    return torch.where((d1 <= 0) & (d2 <= 0), a, out)


def _on_segments(e, f):
    """the closest points of two segments"""
    p, u, q, v = e[:, 0], e[:, 1] - e[:, 0], f[:, 0], f[:, 1] - f[:, 0]
    r = p - q
    a, c, b = _dot(u, u), _dot(v, v), _dot(u, v)
    d, g = _dot(u, r), _dot(v, r)
    den = a * c - b * b
    s = torch.where(den > 1e-12 * a * c, (b * g - d * c) / torch.where(den == 0, torch.ones_like(den), den),
                    torch.zeros_like(den)).clamp(0, 1)
    t = (b * s + g) / c
    s = torch.where(t < 0, (-d / a).clamp(0, 1), torch.where(t > 1, ((b - d) / a).clamp(0, 1), s))
    return p + u * s, q + v * t.clamp(0, 1)
