"""The step's work split (fivonagi_amd/csrc/fv_tables.cpp) of launches with more
strips than the device holds waves: build_work returns, and its workgroups
hold every row of every strip once, in the fewest rounds of resident groups
that whole strips, one to a wave, take."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include "fivonagi_amd/csrc/fv_tables.h"
// args: per_cu skew rotate, then triples: instances nx ny
int main(int argc, char** argv) {
  const int per_cu = std::atoi(argv[1]);
  const float skew = std::atof(argv[2]);
  const bool rotate = std::atoi(argv[3]) != 0;
  std::vector<fivonagi_params> ps;
  for (int a = 4; a + 2 < argc; a += 3) {
    fivonagi_params p;
    std::memset(&p, 0, sizeof(p));
    p.nx = std::atoi(argv[a + 1]);
    p.ny = std::atoi(argv[a + 2]);
    ps.insert(ps.end(), std::atoi(argv[a]), p);
  }
  fvh::WorkList wl;
  fvh::build_work(ps, std::vector<int>(ps.size(), 0),
                  std::vector<std::vector<uint32_t>>(ps.size()), 256, per_cu,
                  fvh::auto_rows(ps, 256L * per_cu), skew, rotate, wl, per_cu == 8 ? 48 : 24);
  std::map<std::pair<int, int>, std::vector<char>> cover;
  long strips = 0, bad = 0;
  for (const auto& p : ps) strips += (p.nx + fv::kStripCols - 1) / fv::kStripCols;
  for (const auto& w : wl.items) {
    auto& c = cover[{w.inst, w.x0}];
    c.resize(ps[w.inst].ny, 0);
    for (int j = w.y0; j < w.y1; ++j) bad += c[j]++ != 0;
  }
  for (const auto& c : cover)
    for (char n : c.second) bad += n != 1;
  const long groups = (long)wl.group_first.size() - 1, room = 64L * per_cu;
  const long rounds = ((strips + 3) / 4 + room - 1) / room;
  std::printf("%ld %ld %ld %d\n", bad, strips - (long)cover.size(), groups,
              groups <= rounds * room);
  return 0;
}
"""


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("many")
    (d / "check.cpp").write_text(CHECK)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", ROOT, "-o", str(d / "check"),
                    str(d / "check.cpp"),
                    os.path.join(ROOT, "fivonagi_amd", "csrc", "fv_tables.cpp")], check=True)
    return str(d / "check")


# per_cu: 16 resident step waves per CU in FP32, 8 in FP64 (256 CUs: 4096 and 2048 waves)
@pytest.mark.parametrize("per_cu,skew,rotate,grids", [
    (16, -1, 0, [(4096, 32, 32)]),                       # as many strips as waves
    (16, -1, 0, [(4097, 32, 32)]),
    (16, -1, 0, [(5000, 16, 16)]),
    (16, -1, 0, [(600, 400, 16)]),
    (16, -1, 0, [(1, 240000, 8)]),
    (16, -1, 0, [(9000, 48, 21)]),                       # three rounds
    (16, -1, 0, [(1, 58, 8192), (4200, 16, 16)]),        # one strip far above the rest
    (16, 0.5, 1, [(600, 400, 400)]),
    (16, 0.95, 1, [(4300, 58, 100), (3, 700, 9)]),
    (8, -1, 0, [(2049, 48, 48)]),
    (8, -1, 0, [(1, 118785, 8)]),
])
def test_more_strips_than_resident_waves(check, per_cu, skew, rotate, grids):
    args = [str(v) for v in (per_cu, skew, rotate, *(x for g in grids for x in g))]
    r = subprocess.run([check, *args], capture_output=True, text=True, timeout=20)
    bad, missing, groups, few = r.stdout.split()
    assert (bad, missing, few) == ("0", "0", "1"), r.stdout


@pytest.mark.gpu
def test_more_instances_than_resident_waves():
    """4100 instances of a strip each: every one steps as it does alone."""
    import numpy as np

    import fivonagi_amd as fa
    from fivonagi_amd import workloads as wl
    probs = [wl.gauss_pulse(20 + k % 7, 18 + k % 5, sigma_cells=2.0 + 0.3 * (k % 11))
             for k in range(4100)]
    print("[many] 4100 instances, 9 steps", flush=True)
    with fa.Context(probs) as ctx:
        ctx.step(9)
        got = {k: ctx.collect(k) for k in (0, 1, 2047, 4095, 4096, 4099)}
    for k, (q, s) in got.items():
        with fa.Context(probs[k]) as one:
            one.step(9)
            q1, s1 = one.collect(0)
        assert np.array_equal(q, q1) and s == s1, k
