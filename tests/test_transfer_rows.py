"""Offsets of the state transfers' rows (dem_io.hpp) for particle counts whose
rows need more than 32 bits to number, on the host alone and without memory
for them: x, v, w, wb, q, F and T of 230 million particles are 5.06e9
numbers."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pacific_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "dem_io.hpp"
int main(int argc, char** argv) {
  const int widths[7] = {3, 3, 3, 3, 4, 3, 3};
  double host, comp[4];
  double* const comps[4] = {comp, comp + 1, comp + 2, comp + 3};
  dem::RowIO io(std::atoi(argv[1]));
  for (int w : widths) io.add(&host, comps, w);
  if (argc == 2) {
    const dem::RowMap m = io.map(0, io.segs().size());
    for (int c = 0; c < m.nc; ++c) std::printf("%zu %d\n", (size_t)m.base[c], m.stride[c]);
  } else {
    for (size_t k = 0; k < io.segs().size(); k = io.part(k))
      std::printf("%zu %zu\n", io.part(k) - k, (size_t)io.map(k, io.part(k)).base[0]);
  }
}
"""


@pytest.fixture(scope="module")
def offsets(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("rows")
    (d / "rows.cpp").write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", CSRC, "-o",
                    str(d / "rows"), str(d / "rows.cpp")], check=True)

    def run(*args):
        out = subprocess.run([str(d / "rows")] + [str(a) for a in args], check=True, stdout=subprocess.PIPE, text=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


@pytest.mark.parametrize("n", [1, 1000, 226050910, 226050911, 230000000, 2147483647])
def test_offsets(offsets, n):
    want, at = [], 0
    for w in (3, 3, 3, 3, 4, 3, 3):
        want += [(at + c, w) for c in range(w)]
        at += w * n
    assert offsets(n) == want


@pytest.mark.parametrize("n,arrays", [(1, [7]), (1143901, [7]), (1143902, [6, 1]), (3000000, [2, 2, 2, 1]),
                                      (10000000, [1] * 7), (230000000, [1] * 7)])
def test_parts(offsets, n, arrays):
    # whole arrays up to 192 MB, the rows of each part from 0
    assert offsets(n, "parts") == [(k, 0) for k in arrays]
