"""What the step kernel reads of the work split (fvh::launch_items of
fivonagi_amd/csrc/fv_tables.cpp): every row of every strip in exactly one place,
every local index of an instance once, both cuts."""
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
// args: 0, 1 (a place's item drawn a second time in place of another's) or 2
// (one row taken from an item)
int main(int argc, char** argv) {
  const int plant = std::atoi(argv[1]);
  const int sizes[][2] = {{8, 8}, {58, 9}, {59, 17}, {64, 21}, {400, 400}, {1021, 777},
                          {4096, 1024}, {70, 4000}, {2048, 333}, {8192, 4096}};
  long bad = 0, cuts = 0;
  for (const auto& a : sizes)
    for (const auto& b : sizes)
      for (int per_cu : {8, 16})
        for (int kind = 0; kind < 4; ++kind)      // automatic, both cuts, asked rows
          for (int rows : {0, 7}) {
            if ((long)a[0] * a[1] + (long)b[0] * b[1] > 20000000L && kind == 3) continue;
            std::vector<fivonagi_params> ps(2);
            std::memset(ps.data(), 0, sizeof(fivonagi_params) * 2);
            ps[0].nx = a[0]; ps[0].ny = a[1]; ps[1].nx = b[0]; ps[1].ny = b[1];
            ps[0].rows_per_wave = rows;
            if (kind != 3) ps[1].rows_per_wave = rows;
            const float skew = kind == 0 || kind == 3 ? -1.0f : 0.7f;
            fvh::WorkList wl;
            fvh::build_work(ps, {0, 0}, {{}, {}}, 256, per_cu, fvh::auto_rows(ps, 256L * per_cu),
                            skew, kind == 2, wl, per_cu == 8 ? 48 : 24);
            auto v = fvh::launch_items(wl, 256);
            size_t first = v.size(), last = 0;
            for (size_t i = 0; i < v.size(); ++i)
              if (v[i].y1 > v[i].y0) { first = std::min(first, i); last = i; }
            if (plant == 1) v[last] = v[first];
            if (plant == 2) --v[last].y1;
            std::vector<int> cover[2], local[2];
            for (int k = 0; k < 2; ++k) {
              const int strips = (ps[k].nx + fv::kStripCols - 1) / fv::kStripCols;
              cover[k].assign((size_t)strips * ps[k].ny, 0);
              local[k].assign(wl.n_items[k], 0);
            }
            long wrong = 0;
            for (const auto& w : v) {
              if (w.y1 <= w.y0) continue;
              const auto& p = ps[w.inst];
              if (w.x0 % fv::kStripCols || w.y0 < 0 || w.y1 > p.ny || w.local < 0 ||
                  w.local >= wl.n_items[w.inst]) { ++wrong; continue; }
              ++local[w.inst][w.local];
              for (int j = w.y0; j < w.y1; ++j)
                ++cover[w.inst][(size_t)(w.x0 / fv::kStripCols) * p.ny + j];
            }
            for (int k = 0; k < 2; ++k) {
              for (int n : cover[k]) wrong += n != 1;
              for (int n : local[k]) wrong += n != 1;
            }
            bad += plant ? wrong == 0 : wrong != 0;
            ++cuts;
          }
  std::printf("%ld of %ld\n", bad, cuts);
  return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("plant", [0, 1, 2])
def test_every_row_in_one_place(tmp_path, plant):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECK)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", ROOT, "-o", str(exe), str(src),
                    os.path.join(ROOT, "fivonagi_amd", "csrc", "fv_tables.cpp")], check=True)
    r = subprocess.run([str(exe), str(plant)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("0 of "), r.stdout + r.stderr
