"""The step's work split (fivonagi_amd/csrc/fv_tables.cpp, cut "running on").

On the CPU: what the step kernel assumes of the list -- workgroups of at most
four places, each chain of waves in one strip with no gap, heights below a
seam of 2 mod 3 and at least 5.  On the GPU: both cuts give the same bits, at
heights from one row to a full group and where a group holds the end of one
strip and the start of the next."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include <cstdio>
#include <cstring>
#include "fivonagi_amd/csrc/fv_tables.h"
int main() {
  int bad = 0;
  const int sizes[][2] = {{8, 8}, {58, 9}, {59, 17}, {64, 21}, {400, 400}, {1021, 777},
                          {4096, 1024}, {70, 4000}, {2048, 333}};
  for (const auto& a : sizes)
    for (const auto& b : sizes)
      for (int per_cu : {8, 16})
        for (float skew : {-1.0f, 0.0f, 0.7f})
          for (int rows : {0, 1, 7}) {
            std::vector<fivonagi_params> ps(2);
            std::memset(ps.data(), 0, sizeof(fivonagi_params) * 2);
            ps[0].nx = a[0]; ps[0].ny = a[1]; ps[1].nx = b[0]; ps[1].ny = b[1];
            ps[0].rows_per_wave = ps[1].rows_per_wave = rows;
            fvh::WorkList wl;
            fvh::build_work(ps, {0, 0}, {{}, {}}, 256, per_cu,
                            fvh::auto_rows(ps, 256L * per_cu), skew, true, wl);
            for (size_t g = 0; g + 1 < wl.group_first.size(); ++g) {
              const int f = wl.group_first[g], n = wl.group_first[g + 1] - f;
              if (n < 1 || n > fv::kGroupWaves) ++bad;
              for (int i = 0; i < n; ++i) {
                const fv::WorkItem& w = wl.items[f + i];
                if ((w.role & fv::kRoleIndex) != i) ++bad;
                if (!(w.role & fv::kRoleAbove)) continue;
                const int H = w.y1 - w.y0;
                if (H < 5 || H % 3 != 2 || i + 1 >= n) { ++bad; continue; }
                const fv::WorkItem& u = wl.items[f + i + 1];
                if (u.inst != w.inst || u.x0 != w.x0 || u.y0 != w.y1 ||
                    u.mrow != w.mrow + H) ++bad;
              }
            }
            // the launch's places hold each item once
            const auto v = fvh::launch_items(wl, 256);
            size_t used = 0;
            for (const auto& w : v) used += w.y1 > w.y0;
            if (v.size() != (wl.group_first.size() - 1) * fv::kGroupWaves ||
                used != wl.items.size()) ++bad;
          }
  std::printf("%d\n", bad);
  return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_groups_are_what_the_kernel_assumes(tmp_path):
    src = tmp_path / "check.cpp"
    src.write_text(CHECK)
    exe = tmp_path / "check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", ROOT, "-o", str(exe), str(src),
                    os.path.join(ROOT, "fivonagi_amd", "csrc", "fv_tables.cpp")], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "0", r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("fp64", [False, True])
@pytest.mark.parametrize("nx,ny,rows", [(64, 8, 0), (59, 17, 0), (130, 21, 0), (200, 100, 0),
                                        (117, 75, 7), (300, 64, 1), (59, 400, 23)])
def test_cuts_give_the_same_bits(nx, ny, rows, fp64):
    import fivonagi_amd as fa
    from fivonagi_amd import workloads as wl
    rng = np.random.default_rng(nx * ny)
    q0 = 1e-3 * rng.standard_normal((3, ny, nx))
    out = []
    for prob in (wl.gauss_pulse(nx, ny, sigma_cells=6.0, rows_per_wave=rows),
                 wl.edge_drive(nx, ny, halfwidth_cells=ny / 4.0, rows_per_wave=rows)):
        prob.q0 = q0.astype(np.float32)
        prob.q0_f64 = q0.copy()
        for skew, rotate in ((0.0, False), (0.0, True), (0.7, True), (-1.0, False)):
            print(f"[cut] {nx}x{ny} rows {rows} fp64 {fp64} bc {prob.bc} skew {skew} {rotate}",
                  flush=True)
            with fa.Context(prob, fp64=fp64) as ctx:
                ctx.set_skew(skew, rotate)
                ctx.step(7)
                out.append((ctx.collect(0), ctx.info(0)["last_cfl"]))
        (qa, sa), ca = out[-4]
        for (q, s), c in out[-3:]:
            assert np.array_equal(q, qa) and s == sa and c == ca
