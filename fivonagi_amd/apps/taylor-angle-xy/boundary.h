// apps/taylor-angle-xy/boundary.h -- the Taylor shock's ghost cells
// (apps/taylor-angle-xy/boundary.h:38-55 of the reference): every ghost cell
// holds the closed form
//   rho' = rhoa tanh(c (x cos(theta) + y sin(theta) - T)),
//   (rho u, rho v) = rho' (cos(theta), sin(theta)),
// taken at (i + MDX, j + MDY) (the window's offset).  The values depend on
// the cell and T only, so they are made ahead of the step that reads them: into
// the state buffer's ghost ring (InstDesc::ring), by the attempt before, for
// the T and offset that follow if it is accepted; where a buffer has no ring,
// into the grid before the step, as the reference's boundary kernel.
#ifndef FIVONAGI_APPS_TAYLOR_ANGLE_XY_BOUNDARY_H
#define FIVONAGI_APPS_TAYLOR_ANGLE_XY_BOUNDARY_H

#include "../common/boundary.h"

namespace fvbc {

struct Taylor {
  static constexpr int kId = fv::kBcTaylor;
  static constexpr bool kRowData = false;
  static constexpr bool kPrepass = true;
  static constexpr bool kExtOnly = false;
  // bB: ring offset of the lane's column on row 0 of its column run (ghost
  // columns; 0 elsewhere)
  __device__ static void lane(int ic, int nx, LaneMap& m, uint32_t size) {
    m.ic = ic;
    m.left = false;
    m.bA = size * (uint32_t)ic;
    const int cc = ic <= 1 ? ic : ic - (nx - 4);       // 0, 1, 2, 3
    const bool ghost = m.ring != 0 && (ic <= 1 || ic >= nx - 2);
    m.bB = ghost ? m.ring + size * (uint32_t)(4 * nx + cc * (m.ny - 4) - 2) : 0u;
  }
  __device__ static uint32_t offset(int rc, int ny, const LaneMap& m, uint32_t row_bytes,
                                    uint32_t size) {
    if (m.ring == 0) return (uint32_t)rc * row_bytes + m.bA;
    const bool grow = rc <= 1 || rc >= ny - 2;
    const uint32_t row =
        grow ? m.ring + (uint32_t)(rc <= 1 ? rc : rc - (ny - 4)) * row_bytes
             : (uint32_t)rc * row_bytes;
    return (!grow && m.bB != 0) ? m.bB + (uint32_t)rc * size : row + m.bA;
  }
  template <typename R>
  __device__ static void load_row(const Tables&, int, RowData<R>&) {}
  template <typename R>
  __device__ static void patch(const PatchCtx<R>&, int, Cell<R>&, const RowData<R>&) {}
  // the closed form at cell (i, j) of the unmoved frame (i + MDX, j + MDY)
  template <typename R>
  __device__ static void prepass(const fv::InstDesc& D, double T, int i, int j, Cell<R>& q) {
    const double arg = D.tay_c * ((double)i * D.dx * D.tay_cos +
                                  ((double)(j - D.tay_jc) * D.dy + D.tay_yoff) * D.tay_sin - T);
    const double r = D.tay_rhoa * tanh(arg);
    q.q1 = (R)r;
    q.q2 = (R)(r * D.tay_cos);
    q.q3 = (R)(r * D.tay_sin);
  }
};

}  // namespace fvbc

#endif  // FIVONAGI_APPS_TAYLOR_ANGLE_XY_BOUNDARY_H
