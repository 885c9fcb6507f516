"""State transfers (rows by id through one block) at the sizes where their
path changes: nothing, one particle, the edges of a copy kernel's block, a
block that just fits the single pinned slice (2 MB: 11,915 particles with all
22 numbers) and one that does not, and one cut into many chunks with a ragged
end; and with every combination of arrays left out.  Values come back bit for
bit, wb as q and w say."""
import ctypes
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from pacific_amd import GrainsGPU

pytestmark = pytest.mark.gpu


def sparse(n, seed=1):
    """n small spheres too far apart to touch, in shuffled places"""
    m = max(2, int(np.ceil(n ** (1 / 3))))
    i = np.random.default_rng(seed).permutation(m ** 3)[:n]
    x = (np.stack([i % m, i // m % m, i // (m * m)], 1) + 0.5) * 4e-3
    g = GrainsGPU((0, 0, 0), (m * 4e-3,) * 3, (0, 0, 0), 1.0, (0, 0, 0))
    g.contact_model(0, 0, 1e4, 0.8, 0.3)
    g.add_spheres(1e-3, 2500.0, 5e-5, 0, x)
    g.init()
    return g, x


@pytest.mark.parametrize("n", [1, 63, 257, 11915, 11916, 100003])
def test_round_trip(gpu, n):
    g, x = sparse(n)
    s = g.state()
    assert np.array_equal(s["x"], x)
    rng = np.random.default_rng(n)
    q = rng.normal(size=(n, 4))
    q /= np.linalg.norm(q, axis=1)[:, None]
    new = dict(x=x + rng.uniform(-1e-4, 1e-4, (n, 3)), v=rng.normal(size=(n, 3)), w=rng.normal(size=(n, 3)), q=q)
    g.set_state(**new)
    s = g.state()
    for k in new:
        assert np.array_equal(s[k], new[k]), k
    # w turned into the body frame: a dozen roundings
    t = 2.0 * np.cross(q[:, :3], new["w"])
    wb = new["w"] - q[:, 3:] * t + np.cross(q[:, :3], t)
    assert np.max(np.abs(s["wb"] - wb)) <= 20 * 2.2e-16 * np.max(np.linalg.norm(new["w"], axis=1))
    ft = rng.normal(size=(n, 6)) * 1e-6
    g.set_hydro_ft(ft)
    g.compute_forces()
    s = g.state()
    assert np.array_equal(s["F"], ft[:, :3]) and np.array_equal(s["T"], ft[:, 3:])


@pytest.mark.parametrize("given", range(16))
def test_arrays_left_out(gpu, given):
    n = 12001
    g, x = sparse(n)
    rng = np.random.default_rng(given)
    q = rng.normal(size=(n, 4))
    new = dict(x=x + 1e-5, v=rng.normal(size=(n, 3)), w=rng.normal(size=(n, 3)),
               q=q / np.linalg.norm(q, axis=1)[:, None])
    old = g.state()
    g.set_state(**{k: a for b, (k, a) in enumerate(new.items()) if given >> b & 1})
    s = g.state()
    for b, (k, a) in enumerate(new.items()):
        assert np.array_equal(s[k], a if given >> b & 1 else old[k]), k
    # the same arrays fetched alone
    L = g._check.__globals__["lib"]()
    dp = ctypes.POINTER(ctypes.c_double)
    out = [np.zeros_like(new[k]) if given >> b & 1 else None for b, k in enumerate(("x", "v", "w", "q"))]
    p = [None if o is None else o.ctypes.data_as(dp) for o in out]
    g._check(L.grains_gpu_get_state(g.h, p[0], p[1], p[2], None, p[3], None, None))
    for o, k in zip(out, ("x", "v", "w", "q")):
        assert o is None or np.array_equal(o, s[k])


@pytest.mark.parametrize("n", [0, 3])
def test_basis_rows(gpu, n):
    from pacific_amd import shapes
    v, f = shapes.tetrahedron(1.2e-3)
    g = GrainsGPU((0, 0, 0), (0.1, 0.1, 0.1), (0, 0, 0), 1.0, (0, 0, 0))
    g.contact_model(0, 0, 1e4, 0.8, 0.3)
    k = g.add_shape(2, verts=v, faces=f)
    B = shapes.random_rotations(max(n, 1), 3).reshape(-1, 9)[:n]
    if n:
        g.add_particles(k, 2500.0, 0, (np.arange(3 * n).reshape(n, 3) + 1) * 1e-2, basis=B)
    g.init()
    assert np.array_equal(g.basis().reshape(n, 9), B)
    g.set_basis(B[::-1])
    assert np.array_equal(g.basis().reshape(n, 9), B[::-1])


def test_systems_of_several_threads(gpu):
    # the buffers are shared: transfers of one chunk and of many, set and
    # fetched from threads at once, the first of them growing the buffers
    sizes = (40, 5000, 30000, 120000)

    def work(n):
        g, x = sparse(n)
        rng = np.random.default_rng(n)
        for _ in range(10):
            v, w = rng.normal(size=(n, 3)), rng.normal(size=(n, 3))
            g.set_state(v=v, w=w)
            s = g.state()
            if not (np.array_equal(s["v"], v) and np.array_equal(s["w"], w) and np.array_equal(s["x"], x)):
                return n
        return 0

    with ThreadPoolExecutor(4) as pool:
        assert list(pool.map(work, sizes)) == [0] * 4


# hipMalloc and hipHostMalloc as the library finds them: they have no room for
# requests of `room` bytes or more once told so
SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
int refused = 0;
static size_t room[2] = {(size_t)-1, (size_t)-1};
void leave(size_t device, size_t host) { room[0] = device; room[1] = host; }
int hipMalloc(void** p, size_t n) {
  if (n >= room[0]) { ++refused; *p = 0; return 2; }
  return ((int (*)(void**, size_t))dlsym(RTLD_NEXT, "hipMalloc"))(p, n);
}
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  if (n >= room[1]) { ++refused; *p = 0; return 2; }
  return ((int (*)(void**, size_t, unsigned))dlsym(RTLD_NEXT, "hipHostMalloc"))(p, n, flags);
}
"""

NO_ROOM = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
shim.leave.argtypes = [ctypes.c_size_t] * 2
import numpy as np
from tests.test_gpu_rows import sparse
n, every = int(sys.argv[2]), 2 ** 64 - 1
if sys.argv[3] == "host":
    shim.leave(every, 0)
g, x = sparse(n)
h, _ = sparse(n)
rng = np.random.default_rng(n)
q = rng.normal(size=(n, 4))
new = dict(x=x + 1e-5, v=rng.normal(size=(n, 3)), w=rng.normal(size=(n, 3)), q=q / np.linalg.norm(q, axis=1)[:, None])
shim.leave(0 if sys.argv[3] == "device" else every, 0 if sys.argv[3] == "host" else every)
g.set_state(**new)
g.set_state(v=new["v"][::-1])
a = g.state()
assert ctypes.c_int.in_dll(shim, "refused").value >= 3
shim.leave(every, every)
h.set_state(**new)
h.set_state(v=new["v"][::-1])
for s in (h.state(), g.state()):
    for k in a:
        assert np.array_equal(a[k], s[k]), k
print("same")
"""


@pytest.mark.parametrize("n,where", [(257, "device"), (257, "host"), (100003, "device"), (100003, "host")])
def test_no_room_for_buffers(gpu, tmp_path, n, where):
    # transfers need no memory: on a full card, or host, they take longer
    (tmp_path / "shim.c").write_text(SHIM)
    so = str(tmp_path / "shim.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", so, str(tmp_path / "shim.c"), "-Wl,--no-as-needed,-rpath,/opt/rocm/lib",
                    "-L/opt/rocm/lib", "-lamdhip64", "-ldl"], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", NO_ROOM, so, str(n), where], cwd=root, stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, text=True, timeout=100)
    assert out.returncode == 0 and out.stdout.endswith("same\n"), out.stdout[-2000:]
