// fv_adjoint_march.hip -- the reverse step of the discrete adjoint as one
// march kernel (gfx950).
//
// The reference has no adjoint.  The step it differentiates (reference:
// common/main.cu:310-635, apps/na/fv.h, apps/na/source.h, common/boundary.h)
// is the one csrc/fv_step.hip runs:
//   q_b = B(q_n), q_y = Y(q_b), q_xy = X(q_y), q_{n+1} = S(q_xy)
// with J = sum_n dt_n sum_box rho'_{n+1}^2 (dt frozen).  One launch of
// adj_reverse_kernel takes lam_{n+1} (the adjoint of q_{n+1}) to
//   lam_n = B^T Y^T X^T S^T (lam_{n+1} + dJ_n/dq_{n+1})
// and adds step n's share to the drive gradient and to J.
//
// Each wave marches up a strip of 56 output columns (4-column halo on each
// side), like the step kernel: per row it recomputes the forward values of
// q_n with the step kernel's own functions (the app's boundary patch, the
// solver.h Riemann solve, limiter and fluxes, and the control block the
// forward step ran with: its dt/dx, dt/dy and drive phase as the step used
// them), so every branch it differentiates is the one the forward step took,
// and applies the transposes in the same pass:
//   row m = r - 2:  q_y(m), the x sweep of m, S^T and X^T of m -> lam_y(m)
//   interface m:    the y limiter's transpose (lam_y of m and m-1)
//   interface m-1:  the Riemann transpose (its wave adjoint is complete once
//                   the limiters of m-2, m-1 and m are done) -> lam_b(m-2)
//   row m-2:        B^T -> lam_n(m-2)
// x neighbours come from DPP lane shifts, y neighbours from register windows.
// A wave runs one or more work items (row ranges of a strip) in turn; the
// host groups them into waves of about equal cost.
//
// Bound by VALU issue: two waves per SIMD (255 registers each) keep it busy 86%
// of the step (counters, 2048x1024: 32.5 M issue quad-cycles, 61.4 us), and memory
// moves 1.85 TB/s, 39% of what a copy reaches.  So the row is kept short: the limiter's transpose
// takes factors formed with the forward values, neighbours' waves enter the
// multiply-adds by DPP, rules of single rows and columns stand in branches,
// and four rows per round leave no window moves: 872 -> about 680 VALU
// instructions per row, a reverse step of 2048x1024 75 -> 63 us, of eight
// 512x512 instances 81 -> 69 us (3 rows per round: 18 more moves a row).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../apps/apps.h"
#include "../apps/na/adjoint.h"
#include "../apps/na/source.h"
#include "fv_adjoint.h"
#include "fv_lanes.h"
#include "fv_types.h"

// no contraction but the written-out fma_: the copies of the unrolled row
// must round alike
#pragma clang fp contract(off)

namespace fv {
namespace adjm {

constexpr int kLanes = 64;
constexpr int kHalo = 4;                       // x halo of the reverse march, each side
constexpr int kCols = kLanes - 2 * kHalo;      // 56 output columns per strip
static_assert(kCols == 56, "the host cuts the reverse march's strips at 56 columns (fv_tables.cpp)");

typedef __attribute__((address_space(1))) float gfloat;
typedef __attribute__((address_space(1))) const float cgfloat;
typedef __attribute__((address_space(1))) char gchar;
typedef __attribute__((address_space(1))) const char cgchar;
typedef __attribute__((address_space(4))) const float kfloat;   // read-only: scalar loads

__device__ __forceinline__ float* state_at(const AdjDesc& D, StateSlot s, size_t cells3) {
  return s >= 0 ? D.kept + (size_t)s * cells3 : D.seg + (size_t)~s * cells3;
}

__device__ __forceinline__ void add_f64(double* p, double v) {
  __builtin_amdgcn_global_atomic_fadd_f64((__attribute__((address_space(1))) double*)p, v);
}

// loads and stores at a 32-bit byte offset from a uniform base
__device__ __forceinline__ float ldg(cgfloat* base, uint32_t off) {
  return *(cgfloat*)((cgchar*)base + off);
}
__device__ __forceinline__ void stg(gfloat* base, uint32_t off, float v) {
  *(gfloat*)((gchar*)base + off) = v;
}

struct Vec3 {
  float a, b, c;       // rho', rho u, rho v
};
__device__ __forceinline__ Vec3 v3(float a, float b, float c) { return Vec3{a, b, c}; }
__device__ __forceinline__ Vec3 operator+(const Vec3& x, const Vec3& y) {
  return Vec3{x.a + y.a, x.b + y.b, x.c + y.c};
}
__device__ __forceinline__ Vec3 sel(bool p, const Vec3& x) {
  return Vec3{p ? x.a : 0.0f, p ? x.b : 0.0f, p ? x.c : 0.0f};
}
using fv::shl1;
using fv::shr1;
__device__ __forceinline__ Vec3 shr1(const Vec3& x) { return Vec3{shr1(x.a), shr1(x.b), shr1(x.c)}; }
__device__ __forceinline__ Vec3 shl1(const Vec3& x) { return Vec3{shl1(x.a), shl1(x.b), shl1(x.c)}; }

struct Row {           // one cell of q_b as the y sweep sees it
  float q1, q2, q3;    // rho', rho u, rho v
  float un, ut;        // v = q3/rho (y normal), u = q2/rho (tangential)
};

struct XRow {          // one cell of q_xy (the recomputed-state check)
  float q1, q2, q3, u, v;
};

struct Vec2 {          // momentum parts
  float b, c;
};

// ga += kp[p] times family p of the waves of the interface to the left (kR
// false) or right: the lane move is the operand of the multiply-add (which
// the compiler forms only where a moved value has a single use).  The s_nop
// covers the two wait states between a write of W and its read across lanes;
// g[6], which the Riemann transpose passes on to a lane move as it is, is written
// first, so that it has its two as well.
#define FV_FMAC7(dir)                                                                  \
  asm("s_nop 1\n\t"                                                                    \
      "v_fmac_f32_dpp %6, %13, %16 " dir " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %0, %7, %14 " dir " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"  \
      "v_fmac_f32_dpp %1, %8, %14 " dir " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"  \
      "v_fmac_f32_dpp %2, %9, %14 " dir " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"  \
      "v_fmac_f32_dpp %3, %10, %15 " dir " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %4, %11, %15 " dir " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t" \
      "v_fmac_f32_dpp %5, %12, %15 " dir " row_mask:0xf bank_mask:0xf bound_ctrl:1"     \
      : "+&v"(ga.g[0]), "+&v"(ga.g[1]), "+&v"(ga.g[2]), "+&v"(ga.g[3]), "+&v"(ga.g[4]),     \
        "+&v"(ga.g[5]), "+&v"(ga.g[6])                                                   \
      : "v"(W.a1), "v"(W.w21), "v"(W.w31), "v"(W.a2), "v"(W.w22), "v"(W.w32), "v"(W.a3), \
        "v"(kp[0]), "v"(kp[1]), "v"(kp[2]))
template <bool kR>
__device__ __forceinline__ void add_scaled_lane(fvad::WaveAdj& ga, const float kp[3],
                                                const fvna::Waves& W) {
  if (kR)
    FV_FMAC7("wave_shl:1");
  else
    FV_FMAC7("wave_shr:1");
}
#undef FV_FMAC7

// Keeps the block it stands in a branch: a uniform condition that seldom
// holds is then skipped, not turned into a select per register.
__device__ __forceinline__ void stay_branch() { asm volatile(""); }

// The reverse step of one work item of an instance whose ghost cells follow
// the boundary policy BC.  kCheck: also recompute q_{n+1} on the item's
// cells and count those that differ from the stored one (D.mismatch).
template <class BC, bool kCheck>
__device__ __forceinline__ void reverse_item(const AdjDesc& D, const AdjItem& it, int item,
                                             int k, StateSlot from, StateSlot to, int par) {
  const int nx = D.nx, ny = D.ny;
  const uint32_t n = (uint32_t)nx * (uint32_t)ny;
  const Ctl* __restrict__ C = D.ctl_log + k;
  const double dt = C->dt;
  const float dtx = C->dtx, dty = C->dty, ddx2 = C->ddx2, ddy2 = C->ddy2;
  const float sin_t = (float)C->drive_s, cos_t = (float)C->drive_c;
  const float hbeta = D.hbeta;
  const float* qs = state_at(D, from, 3 * (size_t)n);
  const float* qn = state_at(D, to, 3 * (size_t)n);            // q_{n+1}
  cgfloat* __restrict__ in1 = (cgfloat*)qs;
  cgfloat* __restrict__ in2 = (cgfloat*)(qs + n);
  cgfloat* __restrict__ in3 = (cgfloat*)(qs + 2 * (size_t)n);
  cgfloat* __restrict__ nq1 = (cgfloat*)qn;
  cgfloat* __restrict__ nq2 = (cgfloat*)(qn + n);
  cgfloat* __restrict__ nq3 = (cgfloat*)(qn + 2 * (size_t)n);
  cgfloat* __restrict__ g1p = (cgfloat*)D.lam[par];
  cgfloat* __restrict__ g2p = (cgfloat*)(D.lam[par] + n);
  cgfloat* __restrict__ g3p = (cgfloat*)(D.lam[par] + 2 * (size_t)n);
  gfloat* __restrict__ o1 = (gfloat*)D.lam[par ^ 1];
  gfloat* __restrict__ o2 = (gfloat*)(D.lam[par ^ 1] + n);
  gfloat* __restrict__ o3 = (gfloat*)(D.lam[par ^ 1] + 2 * (size_t)n);

  const int lane = threadIdx.x;
  const int i = it.x0 - kHalo + lane;
  const bool col_in = i >= 0 && i < nx;
  const int ic = min(max(i, 0), nx - 1);
  const bool col_int = i >= 2 && i <= nx - 3;
  const bool out_lane = i >= it.xo0 && i < it.xo1;
  // dt/d on the lanes of interior columns, 0 on ghost columns
  const float dty_c = col_int ? dty : 0.0f, dtx_c = col_int ? dtx : 0.0f;
  const bool box_col = i >= D.bx0 && i < D.bx0 + D.bnx;
  const uint32_t row_bytes = 4u * (uint32_t)nx;
  const uint32_t cb = 4u * (uint32_t)ic;
  const float two_dt = (float)(2.0 * dt);
  const int y0 = it.y0, y1 = it.y1;

  // the boundary policy's source columns and patch, as the step kernel
  fvbc::LaneMap lm;
  BC::lane(ic, nx, lm, 4u);
  fvbc::Tables tb{D.edge_c, D.edge_s, nullptr};
  fvbc::PatchCtx<float> pc;
  pc.sin_t = sin_t;
  pc.cos_t = cos_t;
  pc.T = C->T;
  pc.hk = 0.0f;
  pc.mdx = 0;
  pc.x0 = it.x0 - 1;     // the column of lane 3 (the step kernel's first output lane)
  pc.nx = nx;
  pc.ny = ny;
  pc.ic = ic;
  pc.left = lm.left;
  pc.any_left = __builtin_amdgcn_ballot_w64(lm.left) != 0;
  auto load_raw = [&](int r, float& a, float& b, float& c, fvbc::RowData<float>& h) {
    const int rc = min(max(r, 0), ny - 1);
    const uint32_t o = BC::offset(rc, ny, lm, row_bytes, 4u);
    a = ldg(in1, o);
    b = ldg(in2, o);
    c = ldg(in3, o);
    if (BC::kRowData) BC::template load_row<float>(tb, rc, h);
  };
  auto patch = [&](Row& q, const fvbc::RowData<float>& h, int r) {
    fvbc::Cell<float> c{q.q1, q.q2, q.q3};
    BC::patch(pc, min(max(r, 0), ny - 1), c, h);
    q.q1 = c.q1;
    q.q2 = c.q2;
    q.q3 = c.q3;
    const float ir = fvna::rcp(1.0f + q.q1);
    q.un = q.q3 * ir;
    q.ut = q.q2 * ir;
  };
  // g(l) = lam_{n+1}(l) + dJ_n/dq_{n+1}(l), where the box term is
  // 2 dt rho'_{n+1}; row l is requested one step before it is used
  // (load_g), then completed (finish_g), which also adds J_n's share of the
  // item's own rows
  double jacc = 0.0;
  const bool in_box_col = col_in && box_col;
  const int box0 = max(D.by0, 0), box1 = min(D.by0 + D.bny, ny);
  auto box_row = [&](int l) { return l >= box0 && l < box1; };
  // rows off the grid read a copy of the nearest row: what follows gives
  // weight 0 to all but the interior rows and columns of g, which also
  // covers the lanes off the grid
  auto load_g = [&](int l, Vec3& g, float& rn) {
    const uint32_t o = (uint32_t)min(max(l, 0), ny - 1) * row_bytes + cb;
    g.a = ldg(g1p, o);
    g.b = ldg(g2p, o);
    g.c = ldg(g3p, o);
    if (box_row(l)) {
      stay_branch();
      rn = ldg(nq1, o);
    }
  };
  auto finish_g = [&](int l, Vec3& g, Vec2& G, float rn) {
    if (box_row(l)) {
      stay_branch();
      g.a = in_box_col ? fvna::fma_(two_dt, rn, g.a) : g.a;
      if (l >= y0 && l < y1 && in_box_col && out_lane) jacc = fma((double)rn, (double)rn, jacc);
    }
    const bool in = col_int && l >= 2 && l <= ny - 3;
    G.b = in ? g.b : 0.0f;
    G.c = in ? g.c : 0.0f;
  };
  const bool strip_l = it.xo0 <= 2 && 2 < it.xo1;             // holds column 2
  const bool strip_r = it.xo0 <= nx - 3 && nx - 3 < it.xo1;   // holds column nx-3

  // ---- windows (every one zeroed: the first rows of the march only warm
  // them up, and nothing they hold reaches an emitted row) ----
  Row b1{}, b2{}, b3{}, b4{};               // q_b rows r-1 .. r-4
  fvna::Iface f1{}, f2{}, f3{};             // y interfaces r-1, r-2, r-3
  fvad::LimT lim2{};                        // limiter of interface r-2
  float dl1[3] = {0.f, 0.f, 0.f};           // W(r-1) . W(r-2) per family
  float Pp[3] = {0.f, 0.f, 0.f};            // P of interface r-2
  fvad::WaveAdj acc3, acc2;                 // wave adjoints of interfaces r-3, r-2
  fvad::zero(acc3);
  fvad::zero(acc2);
  Vec3 ly1{}, ly2{};                        // lam_y rows r-3, r-4
  float gR1 = 0.f, gRn = 0.f, gRt = 0.f, gRun = 0.f, gRut = 0.f;   // what the transpose of
                                            // interface r-4 gives cell r-4
  Vec3 g0{}, gu{}, gnx{};                   // g rows m, m+1 and the prefetched row
  Vec2 Gd{}, G0{}, Gu{};                    // g's momenta on the interior cells of rows m-1, m, m+1
  float rnx = 0.0f;                         // rho' of q_{n+1} on the prefetched row (box rows)
  Vec3 held{};                              // lam_b(0) + lam_b(1), later lam_n(ny-3) waiting for
                                            // lam_b(ny-2) + lam_b(ny-1)
  XRow xc1{}, xc2{};                        // check: q_xy rows m-1, m-2
  uint32_t bad = 0;

  const int r0 = y0 - 3, r_end = y1 + 3;
  float n1, n2, n3;
  fvbc::RowData<float> nh{0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  load_raw(r0 - 1, n1, n2, n3, nh);
  b1.q1 = n1; b1.q2 = n2; b1.q3 = n3;
  patch(b1, nh, r0 - 1);
  load_raw(r0, n1, n2, n3, nh);
  load_g(r0 - 1, gnx, rnx);

  // q_b of row r, g of row r-1, the y interface r (rows r-1 | r; normal = q3,
  // tangential = q2) and the y limiter at interface r-1
  auto forward = [&](int r, Row& bn, fvna::Iface& fn, float* dln, float* P1, float* M,
                     fvad::LimT& lim1) {
    bn.q1 = n1; bn.q2 = n2; bn.q3 = n3;
    patch(bn, nh, r);
    load_raw(r + 1, n1, n2, n3, nh);     // row index clamped (past r_end: unused)
    g0 = gu; gu = gnx;
    Gd = G0; G0 = Gu;
    finish_g(r - 1, gu, Gu, rnx);
    load_g(r, gnx, rnx);
    fvna::riemann(fvna::jump(b1.q1, b1.q3, b1.q2, b1.un, b1.ut, bn.q1, bn.q3, bn.q2, bn.un,
                             bn.ut),
                  hbeta, fn);
    dln[0] = fvna::dot1(fn.w, f1.w);
    dln[1] = fvna::dot2(fn.w, f1.w);
    dln[2] = fn.w.a3 * f1.w.a3;
    fvad::limiter_rec<false>(f1, dl1[0], dln[0], dl1[1], dln[1], dl1[2], dln[2], dty, P1, M, lim1);
  };
  auto rotate = [&](const Row& bn, const fvna::Iface& fn, const float* dln, const float* P1,
                    const fvad::LimT& lim1) {
    b4 = b3; b3 = b2; b2 = b1; b1 = bn;
    f3 = f2; f2 = f1; f1 = fn;
    lim2 = lim1;
    dl1[0] = dln[0]; dl1[1] = dln[1]; dl1[2] = dln[2];
    Pp[0] = P1[0]; Pp[1] = P1[1]; Pp[2] = P1[2];
  };

  // The rows before y0 only warm up the windows of the forward recompute (the
  // y interfaces and limiters the first emitted rows need); everything from
  // q_y on is skipped there, and its windows stay at zero (no emitted row
  // reads them).
#pragma unroll 1
  for (int r = r0; r < y0; ++r) {
    Row bn;
    fvna::Iface fn;
    fvad::LimT lim1;
    float dln[3], P1[3], M[3];
    forward(r, bn, fn, dln, P1, M, lim1);
    rotate(bn, fn, dln, P1, lim1);
  }
  auto row = [&](int r) {
    Row bn;
    fvna::Iface fn;
    fvad::LimT lim1;
    float dln[3], P1[3], M[3];
    forward(r, bn, fn, dln, P1, M, lim1);

    // ---- q_y on row m = r-2 (components: density, normal=q3, tangential=q2) ----
    const int m = r - 2;
    const bool row_int = m >= 2 && m <= ny - 3;
    const float dtyu = row_int ? dty_c : 0.0f, dtxu = row_int ? dtx_c : 0.0f;
    const float y1q = fvna::sub_prod(b2.q1, dtyu, Pp[0] + M[0]);
    const float y3q = fvna::sub_prod(b2.q3, dtyu, Pp[1] + M[1]);
    const float y2q = fvna::sub_prod(b2.q2, dtyu, Pp[2] + M[2]);

    // ---- x sweep on row m: normal = q2, tangential = q3 ----
    const float ir = fvna::rcp(1.0f + y1q);
    const float un = y2q * ir, ut = y3q * ir;
    fvna::Iface fx;
    fvna::SolveT<float> vx;
    const fvna::Jump jx = fvna::jump(shr1(y1q), shr1(y2q), shr1(y3q), shr1(un), shr1(ut), y1q,
                                     y2q, y3q, un, ut);
    fvna::riemann(jx, hbeta, fx, vx);
    float dlx1, dlx2, dlx3;
    dots_left<true>(fx.w, dlx1, dlx2, dlx3);
    const float drx1 = shl1(dlx1), drx2 = shl1(dlx2), drx3 = shl1(dlx3);
    float PX[3], MX[3];
    fvad::LimT limx;
    fvad::limiter_rec<true>(fx, dlx1, drx1, dlx2, drx2, dlx3, drx3, dtx, PX, MX, limx);
    const float mr0 = shl1(MX[0]), mr1 = shl1(MX[1]), mr2 = shl1(MX[2]);
    XRow xc;
    xc.q1 = fvna::sub_prod(y1q, dtxu, mr0 + PX[0]);
    xc.q2 = fvna::sub_prod(y2q, dtxu, mr1 + PX[1]);
    xc.q3 = fvna::sub_prod(y3q, dtxu, mr2 + PX[2]);
    const float ir2 = fvna::rcp(1.0f + xc.q1);
    xc.u = xc.q2 * ir2;
    xc.v = xc.q3 * ir2;

    if (kCheck) {
      // the source of row m-1 from q_xy rows m-2, m-1, m, against q_{n+1}
      const int s = m - 1;
      const float uwe = shr1(xc1.u) + shl1(xc1.u);
      const float vwe = shr1(xc1.v) + shl1(xc1.v);
      const float i2 = fvna::source_increment(ddx2, ddy2, xc1.u, uwe, xc2.u, xc.u);
      const float i3 = fvna::source_increment(ddx2, ddy2, xc1.v, vwe, xc2.v, xc.v);
      const bool s_int = col_int && s >= 2 && s <= ny - 3;
      const float r2 = s_int ? fvna::apply_source(xc1.q2, i2) : xc1.q2;
      const float r3 = s_int ? fvna::apply_source(xc1.q3, i3) : xc1.q3;
      // a Taylor state's ghost ring is rewritten in place by the next step's
      // prepass (its closed form at the next T): only the cells the step
      // computes are compared there
      const bool cmp = BC::kId != kBcTaylor || s_int;
      if (s >= y0 && s < y1 && out_lane && cmp) {
        const uint32_t o = (uint32_t)s * row_bytes + cb;
        const bool same = __float_as_uint(ldg(nq1, o)) == __float_as_uint(xc1.q1) &&
                          __float_as_uint(ldg(nq2, o)) == __float_as_uint(r2) &&
                          __float_as_uint(ldg(nq3, o)) == __float_as_uint(r3);
        bad += same ? 0u : 1u;
      }
      xc2 = xc1;
      xc1 = xc;
    }

    // ---- S^T on row m: the source adds ddx2 (u_W - 2u + u_E) +
    // ddy2 (u_S - 2u + u_N) to rho u, the same with v to rho v, on interior cells ----
    const float sU = fvna::fma_(ddx2, fvna::fma_(-2.0f, G0.b, shr1(G0.b) + shl1(G0.b)),
                                ddy2 * fvna::fma_(-2.0f, G0.b, Gd.b + Gu.b));
    const float sV = fvna::fma_(ddx2, fvna::fma_(-2.0f, G0.c, shr1(G0.c) + shl1(G0.c)),
                                ddy2 * fvna::fma_(-2.0f, G0.c, Gd.c + Gu.c));
    Vec3 lxy;
    lxy.a = fvna::fma_(-fvna::fma_(sU, xc.u, sV * xc.v), ir2, g0.a);
    lxy.b = fvna::fma_(sU, ir2, g0.b);
    lxy.c = fvna::fma_(sV, ir2, g0.c);

    // ---- X^T on row m ----
    // q_xy(k) = q_y(k) - dtxu(k) (PX(k) + MX(k+1)).  The adjoints gPX, gMX are
    // 0 but for the interfaces 2 .. nx-2 (dtxu is 0 on ghost columns), so the
    // waves' adjoints are 0 off the interfaces 1 .. nx-1 of the grid, and so is
    // what their Riemann transposes give; the same holds for y.
    Vec3 lyc;                                 // lam_y of row m
    {
      const float gPX[3] = {-dtxu * lxy.a, -dtxu * lxy.b, -dtxu * lxy.c};
      const float gMX[3] = {shr1(gPX[0]), shr1(gPX[1]), shr1(gPX[2])};
      fvad::WaveAdj gx;
      fvad::zero(gx);
      float gdx[3];
      fvad::limiter_bw(fx, limx, gPX, gMX, gx, gdx);
      // family p of interface k dotted with k-1 (L_p > 0) or with k+1
      const float Ls[3] = {fx.L1, fx.L2, fx.L3};
      float kl[3], kr[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const float gdl = Ls[p] > 0.0f ? gdx[p] : 0.0f;
        const float gdr = gdx[p] - gdl;
        kl[p] = gdl + shr1(gdr);      // times W(k-1): own left dot, and k-1's right dot
        kr[p] = gdr + shl1(gdl);      // times W(k+1): own right dot, and k+1's left dot
      }
      add_scaled_lane<false>(gx, kl, fx.w);
      add_scaled_lane<true>(gx, kr, fx.w);
      const fvad::SumAdj sx =
          fvad::riemann_bw(jx.s1, jx.s2, jx.s3, jx.drho, jx.dn, hbeta, fx, vx, gx);
      // cell k: interface k's R part and interface k+1's L part (lane k+1)
      const float ar1 = (sx.s1 + sx.dr) + shl1(sx.s1 - sx.dr);
      const float an = sx.dn - shl1(sx.dn);
      const float at = sx.dt - shl1(sx.dt);
      const float aun = sx.s2 + shl1(sx.s2);
      const float aut = sx.s3 + shl1(sx.s3);
      lyc.a = fvna::fma_(-fvna::fma_(aun, un, aut * ut), ir, lxy.a + ar1);
      lyc.b = lxy.b + fvna::fma_(aun, ir, an);
      lyc.c = lxy.c + fvna::fma_(aut, ir, at);
    }

    // ---- Y^T: limiter of interface m (P -> cell m, M -> cell m-1) ----
    fvad::WaveAdj acc1;                       // wave adjoint of interface r-1
    fvad::zero(acc1);
    {
      // y component order (rho', normal = rho v, tangential = rho u)
      const float dtyu1 = (m - 1 >= 2 && m - 1 <= ny - 3) ? dty_c : 0.0f;
      const float gPy[3] = {-dtyu * lyc.a, -dtyu * lyc.c, -dtyu * lyc.b};
      const float gMy[3] = {-dtyu1 * ly1.a, -dtyu1 * ly1.c, -dtyu1 * ly1.b};
      float gdy[3];
      fvad::limiter_bw(f2, lim2, gPy, gMy, acc2, gdy);
      const float Ls[3] = {f2.L1, f2.L2, f2.L3};
      float kdn[3], kup[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        kdn[p] = Ls[p] > 0.0f ? gdy[p] : 0.0f;   // dotted with interface m-1
        kup[p] = gdy[p] - kdn[p];                // ... with m+1
      }
      fvad::add_scaled(acc2, kdn, f3.w);
      fvad::add_scaled(acc2, kup, f1.w);
      fvad::add_scaled(acc3, kdn, f2.w);
      fvad::add_scaled(acc1, kup, f2.w);
    }
    // ---- Riemann transpose of interface m-1 = r-3 (rows r-4 | r-3) ----
    const float ys1 = fvna::add_nc(b4.q1, b3.q1), ys2 = fvna::add_nc(b4.un, b3.un);
    const float ys3 = fvna::add_nc(b4.ut, b3.ut);
    const fvad::SumAdj sy =
        fvad::riemann_bw(ys1, ys2, ys3, b3.q1 - b4.q1, b3.q3 - b4.q3, hbeta, f3,
                         fvad::solve_again(ys1, ys2, ys3, f3), acc3);
    // ---- lam_b of row r-4: lam_y, interface r-4's R part, interface r-3's L part ----
    Vec3 lb;
    {
      const float br1 = gR1 + (sy.s1 - sy.dr);
      const float bn_ = gRn - sy.dn;
      const float bt = gRt - sy.dt;
      const float bun = gRun + sy.s2;
      const float but = gRut + sy.s3;
      const float ir4 = fvna::rcp(1.0f + b4.q1);
      lb.a = fvna::fma_(-fvna::fma_(bun, b4.un, but * b4.ut), ir4, ly2.a + br1);
      lb.c = ly2.c + fvna::fma_(bun, ir4, bn_);     // normal = rho v
      lb.b = ly2.b + fvna::fma_(but, ir4, bt);      // tangential = rho u
    }
    gR1 = sy.s1 + sy.dr;
    gRn = sy.dn;
    gRt = sy.dt;
    gRun = sy.s2;
    gRut = sy.s3;

    // ---- B^T and the drive gradient of row j = r-4 (< y1) ----
    const int j = r - 4;
    if (j >= y0) {
      stay_branch();
      const bool interior = col_int && j >= 2 && j <= ny - 3;
      Vec3 a = sel(interior, lb);
      uint32_t o = (uint32_t)j * row_bytes + cb;
      bool defer = false;
      if (BC::kId != kBcTaylor) {
        // zero-gradient copies (apps/common/boundary.h): left columns <- 2
        // (zero-gradient app only; the edge drive sets them), right columns
        // <- nx-3 on rows 2..ny-3, rows 0, 1 <- 2 and ny-2, ny-1 <- ny-3 off
        // the left columns
        if (BC::kId == kBcZeroGrad && strip_l) {
          stay_branch();
          const Vec3 w1 = shr1(lb), w2 = shr1(w1);
          if (i == 2) a = a + w1 + w2;
        }
        if (strip_r && j >= 2 && j <= ny - 3) {
          stay_branch();
          const Vec3 e1 = shl1(lb), e2 = shl1(e1);
          if (i == nx - 3) a = a + e1 + e2;
        }
        if (j <= 2 || j >= ny - 3) {
          stay_branch();
          if (j == 0) held = lb;
          if (j == 1) held = held + lb;
          if (j == 2) a = a + sel(i >= 2, held);
          if (j == ny - 3) {
            held = a;
            defer = true;
          }
          if (j >= ny - 2) held = held + sel(i >= 2, lb);
          if (j == ny - 1 && out_lane) {
            const uint32_t ot = (uint32_t)(ny - 3) * row_bytes + cb;
            stg(o1, ot, held.a);
            stg(o2, ot, held.b);
            stg(o3, ot, held.c);
          }
        }
      }
      if (out_lane && !defer) {
        stg(o1, o, a.a);
        stg(o2, o, a.b);
        stg(o3, o, a.c);
      }
      if (BC::kId == kBcEdgeDrive && it.xo0 == 0) {
        stay_branch();
        // left columns hold p = ampc sin(theta) + amps cos(theta), rho u = p (p + 1)
        const float ec = ((kfloat*)D.edge_c)[j], es = ((kfloat*)D.edge_s)[j];
        fvbc::Cell<float> dc;
        fvbc::drive(ec, es, sin_t, cos_t, dc);
        const float p = dc.q1;
        const float tp = (i == 0 || i == 1) ? fvna::fma_(lb.b, fvna::fma_(2.0f, p, 1.0f), lb.a) : 0.0f;
        // columns 0 and 1 are lanes kHalo and kHalo + 1 of the first strip
        const int tb0 = __builtin_amdgcn_readlane(__float_as_int(tp), kHalo);
        const int tb1 = __builtin_amdgcn_readlane(__float_as_int(tp), kHalo + 1);
        const double g = (double)__int_as_float(tb0) + (double)__int_as_float(tb1);
        // one adder per row and launch (the sum's order is the steps'): the
        // atomic is sent off without waiting for the old value
        if (lane == 0) {
          add_f64(D.grad_ec + j, g * (double)sin_t);
          add_f64(D.grad_es + j, g * (double)cos_t);
        }
      }
    }

    rotate(bn, fn, dln, P1, lim1);
    acc3 = acc2; acc2 = acc1;
    ly2 = ly1; ly1 = lyc;
  };
  // Four rows per round: the windows are four rows deep, so all but a few of
  // the 94 register moves a row would take to shift them vanish (the compiler
  // cannot unroll a loop with cross-lane moves by itself).
  for (int r = y0; r <= r_end; ++r) {
    row(r);
    if (kCheck) continue;
    if (++r > r_end) break;
    row(r);
    if (++r > r_end) break;
    row(r);
    if (++r > r_end) break;
    row(r);
  }

  // J of this step over the item's box cells, one double per item
  double v = jacc;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if (lane == 0 && v != 0.0) D.jpart[item] += dt * v;
  if (kCheck) {
    if (__builtin_amdgcn_ballot_w64(bad != 0) != 0) {
      uint32_t s = bad;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
      if (lane == 0) atomicAdd(D.mismatch, s);
    }
  }
}

}  // namespace adjm

using namespace adjm;

// One reverse step of every instance: step index k of the run (its logged
// control block), the places of q_n and q_{n+1}, adjoint ping-pong index par
// (lam[par] -> lam[par^1]).  Wave w runs the items
// wave_first[w] .. wave_first[w+1] in turn (the end of one strip and the
// start of the next, when the host balances the waves' rows).
template <bool kCheck>
__global__ __launch_bounds__(64, 2) void adj_reverse_kernel(const AdjDesc* __restrict__ ds,
                                                         const AdjItem* __restrict__ items,
                                                         const int32_t* __restrict__ wave_first,
                                                         int n_waves, int k, StateSlot from,
                                                         StateSlot to, int par) {
  // XCD-aware order, as the step kernel: consecutive waves of a strip on one XCD
  int w;
  {
    const int b = blockIdx.x;
    const int q = n_waves >> 3, rem = n_waves & 7, x = b & 7, kk = b >> 3;
    w = x * q + min(x, rem) + kk;
  }
  const int i0 = wave_first[w], i1 = wave_first[w + 1];
  for (int item = i0; item < i1; ++item) {
    const AdjItem it = items[item];
    const AdjDesc& D = ds[it.inst];
    switch (__builtin_amdgcn_readfirstlane(D.bc)) {
      case kBcZeroGrad:
        reverse_item<fvbc::ZeroGradient, kCheck>(D, it, item, k, from, to, par);
        break;
      case kBcEdgeDrive:
        reverse_item<fvbc::EdgeDrive, kCheck>(D, it, item, k, from, to, par);
        break;
      case kBcTaylor:
        reverse_item<fvbc::Taylor, kCheck>(D, it, item, k, from, to, par);
        break;
      default:
        break;
    }
  }
}

// The call's buffers before the forward run: state 0 kept, everything that is
// accumulated or checked cleared, in one launch (seven copies and fills per
// instance took 0.3 ms for 8).  blockIdx.y strides over the instances.
__global__ __launch_bounds__(256) void adj_begin_kernel(const AdjDesc* __restrict__ ds,
                                                        int n_inst, int n_items, int nsteps,
                                                        uint32_t* __restrict__ sync,
                                                        int sync_words) {
  const size_t t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t step = (size_t)gridDim.x * blockDim.x;
  for (int k = blockIdx.y; k < n_inst; k += gridDim.y) {
    const AdjDesc& D = ds[k];
    const size_t n = (size_t)D.nx * (size_t)D.ny;
    for (int f = 0; f < 3; ++f)
      for (size_t e = t0; e < n; e += step) {
        D.kept[f * n + e] = D.start[f][e];
        D.lam[0][f * n + e] = 0.0f;
      }
    for (size_t e = t0; e < (size_t)D.ny; e += step) D.grad_ec[e] = D.grad_es[e] = 0.0;
    for (size_t e = t0; e < (size_t)nsteps; e += step) D.ctl_log[e].dt = 0.0;
  }
  if (blockIdx.y == 0) {
    const AdjDesc& D = ds[0];
    for (size_t e = t0; e < (size_t)n_items; e += step) D.jpart[e] = 0.0;
    for (size_t e = t0; e < (size_t)sync_words; e += step) sync[e] = 0u;
    if (t0 < 2) D.mismatch[t0] = 0u;
  }
}

// A segment's tables, one thread per (local step, instance): the step kernel's
// control blocks from the log -- the logged block as the attempt's own, which
// an idle fold keeps as it is -- and the state each step reads.  Formed here,
// a segment needs no upload and no wait for the one before it.
__global__ __launch_bounds__(64) void adj_segment_kernel(const AdjDesc* __restrict__ ds, int n_inst,
                                                         int s0, int len, int keep_all,
                                                         StateSlot first,
                                                         InstDesc* __restrict__ rdesc,
                                                         Ctl* __restrict__ rctl) {
  const int e = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (e >= len * n_inst) return;
  const int s = e / n_inst;
  const AdjDesc& D = ds[e - s * n_inst];
  Ctl t = D.ctl_log[s0 + s];
  t.cur = 0;
  t.err = 0;
  t.target_acc = INT64_MAX;
  t.T_stop = __builtin_inf();
  rctl[2 * e] = t;
  rctl[2 * e + 1] = t;
  const size_t n = (size_t)D.nx * (size_t)D.ny;
  float* q = state_at(D, s == 0 ? first : keep_all ? first + s : ~(StateSlot)(s - 1), 3 * n);
  for (int f = 0; f < 3; ++f) rdesc[e].q[0][f] = q + f * n;
}

// After a forward run that kept its state in the history alone: the last state
// into the buffer the settled control block names.
__global__ __launch_bounds__(256) void adj_back_kernel(const InstDesc* __restrict__ insts,
                                                       int n_inst, int phase) {
  for (int k = blockIdx.y; k < n_inst; k += gridDim.y) {
    const InstDesc& D = insts[k];
    const Ctl& P = D.ctl[(phase + 1) & 1];
    const int64_t t = P.n_acc - D.log_base;
    if (!D.hist_state || t < 1) continue;
    const size_t n = (size_t)D.nx * (size_t)D.ny;
    const float* s = D.hist + (size_t)t * 3 * n;
    for (int f = 0; f < 3; ++f) {
      float* q = D.q[P.cur][f];
      for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
           e += (size_t)gridDim.x * blockDim.x)
        q[e] = s[f * n + e];
    }
  }
}

// After the forward run: steps the log does not hold (none, by then).
__global__ __launch_bounds__(256) void adj_log_kernel(const AdjDesc* __restrict__ ds, int n_inst,
                                                      int nsteps) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int k = blockIdx.y; k < n_inst; k += gridDim.y)
    if (e < (size_t)nsteps && !(ds[k].ctl_log[e].dt > 0.0)) atomicAdd(ds[k].mismatch + 1, 1u);
}

// dJ/dq0 into the grids the context keeps, unless a check failed.
__global__ __launch_bounds__(256) void adj_end_kernel(const AdjDesc* __restrict__ ds, int n_inst,
                                                      int par) {
  if (ds[0].mismatch[0] != 0u || ds[0].mismatch[1] != 0u) return;
  for (int k = blockIdx.y; k < n_inst; k += gridDim.y) {
    const AdjDesc& D = ds[k];
    const size_t n3 = 3 * (size_t)D.nx * (size_t)D.ny;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n3;
         e += (size_t)gridDim.x * blockDim.x)
      D.lam_out[e] = D.lam[par][e];
  }
}

}  // namespace fv

// ---------------------------------------------------------------- launches --

extern "C" hipError_t fv_adj_reverse(const fv::AdjDesc* ds, const fv::AdjItem* items,
                                     const int32_t* wave_first, int n_waves, int k,
                                     fv::StateSlot from, fv::StateSlot to, int par, int check,
                                     hipStream_t s) {
  if (n_waves <= 0) return hipSuccess;
  if (check)
    hipLaunchKernelGGL(fv::adj_reverse_kernel<true>, dim3(n_waves), dim3(64), 0, s, ds, items,
                       wave_first, n_waves, k, from, to, par);
  else
    hipLaunchKernelGGL(fv::adj_reverse_kernel<false>, dim3(n_waves), dim3(64), 0, s, ds, items,
                       wave_first, n_waves, k, from, to, par);
  return hipGetLastError();
}

// Grid of the copying kernels: 4 cells per thread, up to a few blocks per CU.
static dim3 adj_grid(size_t max_cells, int n_inst) {
  const size_t b = (max_cells + 1023) / 1024;
  return dim3((unsigned)(b > 2048 ? 2048 : b), (unsigned)(n_inst > 65535 ? 65535 : n_inst));
}

extern "C" hipError_t fv_adj_begin(const fv::AdjDesc* ds, int n_inst, size_t max_cells,
                                   int n_items, int nsteps, fv::SyncSlots* sync, int n_sync,
                                   hipStream_t s) {
  hipLaunchKernelGGL(fv::adj_begin_kernel, adj_grid(max_cells, n_inst), dim3(256), 0, s, ds,
                     n_inst, n_items, nsteps, (uint32_t*)sync,
                     (int)(sizeof(fv::SyncSlots) / 4) * n_sync);
  return hipGetLastError();
}

extern "C" hipError_t fv_adj_segment(const fv::AdjDesc* ds, int n_inst, int s0, int len,
                                     int keep_all, fv::StateSlot first, fv::InstDesc* rdesc,
                                     fv::Ctl* rctl, hipStream_t s) {
  hipLaunchKernelGGL(fv::adj_segment_kernel, dim3((len * n_inst + 63) / 64), dim3(64), 0, s, ds,
                     n_inst, s0, len, keep_all, first, rdesc, rctl);
  return hipGetLastError();
}

extern "C" hipError_t fv_adj_back(const fv::InstDesc* insts, int n_inst, size_t max_cells,
                                  int phase, hipStream_t s) {
  hipLaunchKernelGGL(fv::adj_back_kernel, adj_grid(max_cells, n_inst), dim3(256), 0, s, insts,
                     n_inst, phase);
  return hipGetLastError();
}

extern "C" hipError_t fv_adj_log(const fv::AdjDesc* ds, int n_inst, int nsteps, hipStream_t s) {
  hipLaunchKernelGGL(fv::adj_log_kernel, dim3((nsteps + 255) / 256, adj_grid(1, n_inst).y), dim3(256),
                     0, s, ds, n_inst, nsteps);
  return hipGetLastError();
}

extern "C" hipError_t fv_adj_end(const fv::AdjDesc* ds, int n_inst, size_t max_cells, int par,
                                 hipStream_t s) {
  hipLaunchKernelGGL(fv::adj_end_kernel, adj_grid(max_cells, n_inst), dim3(256), 0, s, ds, n_inst, par);
  return hipGetLastError();
}

// Resident reverse waves per CU.
extern "C" hipError_t fv_adj_occupancy(int* waves_per_cu) {
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(waves_per_cu, fv::adj_reverse_kernel<false>,
                                                      64, 0);
}
