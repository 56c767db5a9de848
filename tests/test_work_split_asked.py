"""The step's work split (fivonagi_amd/csrc/fv_tables.cpp) of instances that ask
for rows per wave (fivonagi_params.rows_per_wave) beside some that do not, or for
other numbers: each is cut at its own height."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "fivonagi_amd/csrc/fv_tables.h"
// args: skew rotate, then triples: nx ny rows_per_wave; prints the tallest
// item of each instance
int main(int argc, char** argv) {
  std::vector<fivonagi_params> ps;
  for (int a = 3; a + 2 < argc; a += 3) {
    fivonagi_params p;
    std::memset(&p, 0, sizeof(p));
    p.nx = std::atoi(argv[a]);
    p.ny = std::atoi(argv[a + 1]);
    p.rows_per_wave = std::atoi(argv[a + 2]);
    ps.push_back(p);
  }
  fvh::WorkList wl;
  fvh::build_work(ps, std::vector<int>(ps.size(), 0),
                  std::vector<std::vector<uint32_t>>(ps.size()), 256, 16,
                  fvh::auto_rows(ps, 4096), std::atof(argv[1]), std::atoi(argv[2]) != 0, wl);
  std::vector<int> tall(ps.size(), 0);
  for (const auto& w : wl.items) tall[w.inst] = std::max(tall[w.inst], w.y1 - w.y0);
  for (int t : tall) std::printf("%d ", t);
  return 0;
}
"""


@pytest.fixture(scope="module")
def tallest(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("asked")
    (d / "check.cpp").write_text(CHECK)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", ROOT, "-o", str(d / "check"),
                    str(d / "check.cpp"),
                    os.path.join(ROOT, "fivonagi_amd", "csrc", "fv_tables.cpp")], check=True)

    def run(skew, rotate, grids):
        args = [str(v) for v in (skew, rotate, *(x for g in grids for x in g))]
        r = subprocess.run([str(d / "check"), *args], capture_output=True, text=True, timeout=20)
        return [int(t) for t in r.stdout.split()]
    return run


# (3/2 of the mean height at the tallest level, and the three rows the march rounds to)
@pytest.mark.parametrize("skew,rotate", [(-1, 0), (0, 0), (0, 1), (0.5, 1)])
@pytest.mark.parametrize("grids", [
    [(64, 64, 16), (2048, 1024, 0)],
    [(2048, 1024, 0), (8, 8, 8), (300, 300, 40)],
    [(1024, 1024, 12), (1024, 1024, 48)],
    [(4096, 1024, 1), (512, 512, 0)],
])
def test_each_instance_is_cut_at_its_own_height(tallest, skew, rotate, grids):
    free = tallest(skew, rotate, [(nx, ny, 0) for nx, ny, _ in grids])
    for (nx, ny, rows), tall, auto in zip(grids, tallest(skew, rotate, grids), free):
        assert tall <= (1.5 * max(rows, 5) + 3 if rows else 1.1 * auto + 3), (rows, tall, auto)
        assert rows == 0 or tall >= min(ny, rows) // 2
