// apps/na/adjoint.h -- reverse-mode pieces of the "na" plug-in (device code),
// used by the adjoint march kernel (csrc/fv_adjoint_march.hip).
//
// The forward values the reverse pass branches on (waves, speeds, the
// limiter's ratios, P and M) come from the functions of apps/na/solver.h that
// the step kernel calls, with the same operands, so the upwind side, the sign
// of each speed and the limiter case of every interface are those of the
// executed forward step.  What the transposes need beyond those values is
// formed next to them here.
//
// Forward (solver.h riemann; L = cell k-1, R = cell k, components
// (rho', normal momentum n, tangential momentum t), un = n/rho, ut = t/rho):
//   s1 = r1L + r1R, s2 = unL + unR, s3 = utL + utR, S1 = s1 + 2
//   drho = r1R - r1L, dn = nR - nL, dtg = tR - tL
//   tmp1 = s2/S1, tmp3 = tmp1 (tmp1 - s2) + hbeta s1 + 1, sq = sqrt(tmp3)
//   L1,2 = tmp1 +- sq, L3 = tmp1, d_p = L_p S1 - s3, A_p = s3 (L_p - s2)/d_p
//   a1 = (dn - drho L2)/(2 sq), a2 = drho - a1, a3 = dtg - (a1 A1 + a2 A2)
//   W1 = a1 (1, L1, A1), W2 = a2 (1, L2, A2), W3 = (0, 0, a3)
// Limiter (solver.h limited_flux), per family p:
//   r_p = W_p . W_p(upwind) / |W_p|^2, h_p = clamp(min((1 + r_p)/4, r_p), 0, 1)
//   c_p = |L_p| (1 - |L_p| dt/d) h_p, al_p = max(L_p, 0) - c_p, be_p = L_p - al_p
//   P = sum_p al_p W_p, M = sum_p be_p W_p
// Every multiply-add is written out and contraction is off in these bodies:
// the kernel holds several copies of its row, and they must round alike.
// The derivatives are those of that branch path with dt frozen; a limiter
// ratio at a clamp (h = 0 or 1) or of a zero wave has derivative 0.
#ifndef FIVONAGI_APPS_NA_ADJOINT_H
#define FIVONAGI_APPS_NA_ADJOINT_H

#include <hip/hip_runtime.h>

#include "solver.h"

namespace fvad {

using fvna::Iface;
using fvna::Waves;

// What the limiter's transpose needs of one interface, per wave family, formed
// with the forward values rather than from them a second time: with g2 the
// adjoint of al - be,
//   adjoint of the dot product with the upwind neighbour  g2 kd
//   adjoint of the speed, beside be's                     g2 ks
//   twice the adjoint of |W|^2                            g2 kn
// kd and kn are 0 where h is clamped or the wave is zero, so no infinity or
// NaN of the forward enters a product.
struct LimT {
  float al[3], kd[3], ks[3], kn[3];
};

// The limited fluxes of interface f as the step kernel forms them (same
// call), and the transpose's quantities.  dl_p = W_p . W_p(k-1),
// dr_p = W_p . W_p(k+1).
template <bool kL3Product>
__device__ __forceinline__ void limiter_rec(const Iface& f, float dl1, float dr1, float dl2,
                                            float dr2, float dl3, float dr3, float dtd,
                                            float P[3], float M[3], LimT& t) {
#pragma clang fp contract(off)
  const float up1 = fvna::upwind(f.L1, dl1, dr1), up2 = fvna::upwind(f.L2, dl2, dr2);
  const float up3 = fvna::upwind(f.L3, dl3, dr3);
  fvna::LimitT<float> v;
  float n1, n2;
  fvna::norms(f.w, n1, n2);
  fvna::limited_flux<kL3Product>(f, n1, n2, up1, up2, up3, dtd, P, M, v);
  const float L[3] = {f.L1, f.L2, f.L3};
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    // al = max(L, 0) - c, be = L - al, c = g h, g = s om, om = 1 - s dt/d,
    // s = |L|, h = min(t, r) where it is not clamped, r = dot / |W|^2
    t.al[p] = v.al[p];
    const bool live = v.mn[p] > 0.0f && v.mn[p] < 1.0f;
    const float qd = v.r[p] < v.t[p] ? v.rn[p] : 0.25f * v.rn[p];   // dh/ddot
    t.kd[p] = live ? -v.g[p] * qd : 0.0f;
    t.kn[p] = -2.0f * t.kd[p] * (live ? v.r[p] : 0.0f);
    const float e = v.h[p] * fvna::fma_(2.0f, v.om[p], -1.0f);      // dc/ds
    t.ks[p] = L[p] > 0.0f ? 1.0f - e : (L[p] < 0.0f ? e : 0.0f);
  }
}

// Adjoint of one interface's waves (a1, w21, w31, a2, w22, w32, a3) and
// speeds (L1, L2, L3).
struct WaveAdj {
  float g[7];
  float gs[3];
};

// An empty accumulator.  -0 is the exact identity of IEEE addition
// (-0 + x = x for every x, +0 included; fma(a, b, -0) = a b), so the first
// term added to it needs no instruction of its own; +0 is not (+0 + -0 = +0).
__device__ __forceinline__ void zero(WaveAdj& a) {
#pragma unroll
  for (int c = 0; c < 7; ++c) a.g[c] = -0.0f;
  a.gs[0] = a.gs[1] = a.gs[2] = -0.0f;
}

// Transpose of limiter_rec: from the adjoints gP, gM of the interface's P
// and M (component order of the sweep), accumulate the adjoint of its own
// waves and speeds into ga and return the adjoint of each family's dot
// product with its upwind neighbour (gd).  With be = L - al only
// D = gP - gM meets al: sum_p (al_p gP + be_p gM) . W_p =
// sum_p (al_p D + L_p gM) . W_p.
__device__ __forceinline__ void limiter_bw(const Iface& f, const LimT& t, const float gP[3],
                                           const float gM[3], WaveAdj& ga, float gd[3]) {
#pragma clang fp contract(off)
  const Waves& w = f.w;
  const float D[3] = {gP[0] - gM[0], gP[1] - gM[1], gP[2] - gM[2]};
  const float g2[3] = {fvna::fma_(D[0], w.a1, fvna::fma_(D[1], w.w21, D[2] * w.w31)),
                       fvna::fma_(D[0], w.a2, fvna::fma_(D[1], w.w22, D[2] * w.w32)),
                       D[2] * w.a3};
  ga.gs[0] = fvna::fma_(gM[0], w.a1, fvna::fma_(gM[1], w.w21, fvna::fma_(gM[2], w.w31, ga.gs[0])));
  ga.gs[1] = fvna::fma_(gM[0], w.a2, fvna::fma_(gM[1], w.w22, fvna::fma_(gM[2], w.w32, ga.gs[1])));
  ga.gs[2] = fvna::fma_(gM[2], w.a3, ga.gs[2]);
  float gn[3];
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    ga.gs[p] = fvna::fma_(g2[p], t.ks[p], ga.gs[p]);
    gd[p] = g2[p] * t.kd[p];
    gn[p] = g2[p] * t.kn[p];
  }
  auto add = [&](int c, float al, float L, float gn2, int k, float wk) {
    ga.g[c] = fvna::fma_(al, D[k], fvna::fma_(L, gM[k], fvna::fma_(gn2, wk, ga.g[c])));
  };
  add(0, t.al[0], f.L1, gn[0], 0, w.a1);
  add(1, t.al[0], f.L1, gn[0], 1, w.w21);
  add(2, t.al[0], f.L1, gn[0], 2, w.w31);
  add(3, t.al[1], f.L2, gn[1], 0, w.a2);
  add(4, t.al[1], f.L2, gn[1], 1, w.w22);
  add(5, t.al[1], f.L2, gn[1], 2, w.w32);
  add(6, t.al[2], f.L3, gn[2], 2, w.a3);
}

// ga += the dot-product adjoints of the families of a neighbouring
// interface's limiter (or of this one's) times the other interface's waves:
// kp[p] multiplies family p of W.
__device__ __forceinline__ void add_scaled(WaveAdj& ga, const float kp[3], const Waves& W) {
  ga.g[0] = fvna::fma_(kp[0], W.a1, ga.g[0]);
  ga.g[1] = fvna::fma_(kp[0], W.w21, ga.g[1]);
  ga.g[2] = fvna::fma_(kp[0], W.w31, ga.g[2]);
  ga.g[3] = fvna::fma_(kp[1], W.a2, ga.g[3]);
  ga.g[4] = fvna::fma_(kp[1], W.w22, ga.g[4]);
  ga.g[5] = fvna::fma_(kp[1], W.w32, ga.g[5]);
  ga.g[6] = fvna::fma_(kp[2], W.a3, ga.g[6]);
}

// Adjoint of the sums and differences one Riemann solve starts from:
// cell R receives (s1 + dr, dn, dt, s2, s3) and cell L (s1 - dr, -dn, -dt,
// s2, s3) as the adjoint of its (rho', n, t, un, ut).
struct SumAdj {
  float s1, s2, s3, dr, dn, dt;
};

// The values riemann_bw needs of an interface whose solve is rows back (only
// its waves and speeds are kept): formed again, with the square root from
// L1 - L2 = 2 sq.
__device__ __forceinline__ fvna::SolveT<float> solve_again(float s1, float s2, float s3,
                                                           const Iface& f) {
#pragma clang fp contract(off)
  fvna::SolveT<float> v;
  const float S1 = s1 + 2.0f;
  v.rS = fvna::rcp(S1);
  v.rs = 2.0f * fvna::rcp(f.L1 - f.L2);
  v.d1 = fvna::fma_(f.L1, S1, -s3);
  v.d2 = fvna::fma_(f.L2, S1, -s3);
  v.rdd = fvna::rcp(v.d1 * v.d2);
  const float srd = s3 * v.rdd;
  v.A1 = (f.L1 - s2) * (v.d2 * srd);
  v.A2 = (f.L2 - s2) * (v.d1 * srd);
  return v;
}

// Transpose of solver.h riemann at one interface, from the adjoint of its
// waves and speeds (ga).  s1..dn as the forward forms them; f, v its result.
__device__ __forceinline__ SumAdj riemann_bw(float s1, float s2, float s3, float drho, float dn,
                                             float hbeta, const Iface& f,
                                             const fvna::SolveT<float>& v, const WaveAdj& ga) {
#pragma clang fp contract(off)
  const float L1 = f.L1, L2 = f.L2, tmp1 = f.L3;
  const float a1 = f.w.a1, a2 = f.w.a2;
  const float S1 = s1 + 2.0f;
  const float rS = v.rS, hrs = 0.5f * v.rs;             // hrs = 1 / (2 sq)
  const float id1 = v.d2 * v.rdd, id2 = v.d1 * v.rdd;   // 1/d1, 1/d2
  const float A1 = v.A1, A2 = v.A2;
  SumAdj o;
  // a3 = dtg - (a1 A1 + a2 A2), w21 = a1 L1, w31 = a1 A1, w22 = a2 L2, w32 = a2 A2
  const float ga3 = ga.g[6];
  const float gw31 = ga.g[2] - ga3, gw32 = ga.g[5] - ga3;
  o.dt = ga3;
  float ga1 = fvna::fma_(ga.g[1], L1, fvna::fma_(gw31, A1, ga.g[0]));
  const float ga2 = fvna::fma_(ga.g[4], L2, fvna::fma_(gw32, A2, ga.g[3]));
  float gL1 = fvna::fma_(ga.g[1], a1, ga.gs[0]);
  float gL2 = fvna::fma_(ga.g[4], a2, ga.gs[1]);
  const float gA1 = gw31 * a1, gA2 = gw32 * a2;
  // a2 = drho - a1
  float gdr = ga2;
  ga1 -= ga2;
  // a1 = (dn - drho L2) hrs, hrs = 1 / (2 sq)
  const float t1 = ga1 * hrs;
  o.dn = t1;
  gdr = fvna::fma_(-t1, L2, gdr);
  gL2 = fvna::fma_(-t1, drho, gL2);
  // A_p = s3 (L_p - s2) / d_p, d_p = L_p S1 - s3
  const float e1 = gA1 * id1, e2 = gA2 * id2;
  gL1 = fvna::fma_(e1, fvna::fma_(-A1, S1, s3), gL1);
  gL2 = fvna::fma_(e2, fvna::fma_(-A2, S1, s3), gL2);
  float gs2 = -(e1 + e2) * s3;
  o.s3 = fvna::fma_(e1, (L1 - s2) + A1, e2 * ((L2 - s2) + A2));
  float gS1 = -fvna::fma_(e1 * A1, L1, e2 * A2 * L2);
  // L1,2 = tmp1 +- sq, L3 = tmp1; sq = sqrt(tmp3)
  float gt1 = gL1 + gL2 + ga.gs[2];
  const float gsq = fvna::fma_(-2.0f * t1, a1, gL1 - gL2);
  const float gt3 = gsq * hrs;
  // tmp3 = tmp1 (tmp1 - s2) + hbeta s1 + 1
  gt1 = fvna::fma_(gt3, fvna::fma_(2.0f, tmp1, -s2), gt1);
  gs2 = fvna::fma_(-gt3, tmp1, gs2);
  // tmp1 = s2 / S1, S1 = s1 + 2
  const float gtS = gt1 * rS;
  gs2 += gtS;
  gS1 = fvna::fma_(-gtS, tmp1, gS1);
  const float gs1 = fvna::fma_(gt3, hbeta, gS1);
  o.s1 = gs1;
  o.s2 = gs2;
  o.dr = gdr;
  return o;
}

}  // namespace fvad

#endif  // FIVONAGI_APPS_NA_ADJOINT_H
