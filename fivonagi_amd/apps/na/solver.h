// apps/na/solver.h -- the "na" (nonlinear acoustics) plug-in as device code:
// Roe-type Riemann solver, MC limiter and correction flux, delta-diffusion
// source.  These are the per-interface / per-cell bodies that the fused step
// kernel (csrc/fv_step.hip) calls; they are not kernels themselves.
//
// Reference bodies restated here:
//   Riemann solve ........ apps/na/fv.h:88-180 (x) and :276-368 (y)
//   MC limiter ........... apps/na/fv.h:579-662 (philim.f)
//   correction flux ...... apps/na/fv.h:666-711
//   first/second order ... apps/na/fv.h:427-434, :979-986
//   source ............... apps/na/source.h:84-104
//
// Arithmetic form (all algebraically identical to the reference):
//   * rho = 1 + rho' is never differenced: drho = rho'_R - rho'_L and
//     Z1 - 1 = (rho'_R + rho'_L)/2 are taken from rho' directly, so FP32 does
//     not lose the ~7 bits the reference loses to the "+1" (fv.h:62-63).
//   * a3 = dt - (a1*A1 + a2*A2), which is fv.h:119-125 after substituting a1, a2.
//   * 1/x through v_rcp_f32 / v_rsq_f32 (1 ulp); L1 - L2 = 2*sqrt(tmp3).
//   * the fluctuations and the correction flux are folded per wave family
//     (see limited_flux).
//   * the two sweep updates (step + writeLimiters) are fused into one:
//     q - dtd*((apdq - fadd)(k) + (amdq + fadd)(k+1)).
//   * every multiply-add is written out (fma_) and contraction is off in these
//     bodies: which products fuse is part of the result, and it must not
//     depend on how a kernel that inlines them is laid out.
#ifndef FIVONAGI_APPS_NA_SOLVER_H
#define FIVONAGI_APPS_NA_SOLVER_H

#include <hip/hip_runtime.h>

namespace fvna {

// The bodies below are templates on the real type R: float is the
// production path (FP32 with the v_rcp/v_rsq/v_med3 forms), double the FP64
// path (PRECISION=2 of the reference).  In double, 1/x and 1/sqrt(x) are the
// hardware estimates (2^-24 relative at worst) refined by one step of third
// order, whose remainder is below 2^-68: three and five instructions where two
// Newton steps take four and eight (376 -> 358 VALU per row; 2048x1024 38.1 ->
// 36.8 us) at the same error, over 3 x 2^20 arguments from e^-200 to 4: 1/x at
// most 0.5 ulp, 1/sqrt(x) at most 0.995 (Newton: 0.5, 0.998).
// Their arguments here are O(1) away from
// zero (2 Z1, (L1 S1 - s3)(L2 S1 - s3), 1 + rho', the discriminant) except
// the limiter's |W|^2, where 0 gives NaN as the IEEE form's 0 * inf does.
__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double rcp(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);          // e = 1 - x y; 1/x = y (1 + e + e^2 + ..)
  return fma(y, fma(e, e, e), y);
}
__device__ __forceinline__ double rsq(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double r = fma(-x * y, y, 1.0);      // r = 1 - x y^2; y (1 + r/2 + 3 r^2/8 + ..)
  return fma(y * r, fma(0.375, r, 0.5), y);
}
__device__ __forceinline__ float fma_(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double fma_(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float min_(float a, float b) { return fminf(a, b); }

// a + b never contracted with a product feeding it, so that when a is the
// neighbouring lane's value its cross-lane move can fold into this add
template <typename R>
__device__ __forceinline__ R add_nc(R a, R b) {
#pragma clang fp contract(off)
  return a + b;
}

// q - d * flux in one rounding: a sweep's update of a cell
template <typename R>
__device__ __forceinline__ R sub_prod(R q, R d, R flux) {
  return fma_(-d, flux, q);
}

// max(a, b) of finite values as one v_med3_f32 (median of a, b, FLT_MAX;
// with +inf the intrinsic is folded back into a maxnum).
// fmaxf must quiet signalling NaNs in IEEE mode, so on values the compiler
// cannot prove canonical (registers carried around the march loop) it adds a
// canonicalising v_max per operand; the med3 intrinsic is taken as is.
__device__ __forceinline__ float fmax2(float a, float b) {
  return __builtin_amdgcn_fmed3f(a, b, 3.4028234663852886e38f);
}
__device__ __forceinline__ double fmax2(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
// (the FP64 form is the bare instruction for the same reason)
// clamp to [0, 1]; a NaN gives 0
__device__ __forceinline__ float clamp01(float x) { return __builtin_amdgcn_fmed3f(x, 0.0f, 1.0f); }

// Waves of one interface in (density, normal, tangential) component order.
// W1 = a1*(1, L1, A1), W2 = a2*(1, L2, A2), W3 = (0, 0, a3).
template <typename R>
struct WavesT {
  R a1, w21, w31;       // wave 1: W11, W21, W31
  R a2, w22, w32;       // wave 2: W12, W22, W32
  R a3;                 // wave 3: W33 (W13 = W23 = 0)
};

template <typename R>
struct IfaceT {
  WavesT<R> w;
  R L1, L2, L3;         // speeds s1, s2, s3
  R s2, rS;             // L3 = s2 * rS (limited_flux's kL3Product)
  bool bad;             // tmp3 < 0: imaginary eigenvalue (simError = 2)
};
typedef WavesT<float> Waves;
typedef IfaceT<float> Iface;

// Sums and differences of the two cells L, R of an interface, all that its
// Riemann solve needs of them.  r1 = rho', n = normal momentum, t = tangential
// momentum, un/ut = n/rho, t/rho of the same cell (precomputed once per cell).
// Every L operand enters only sums and differences with its R partner, so
// when L is the neighbouring lane's value the cross-lane move folds into
// the add/subtract (DPP operand).
template <typename R>
struct JumpT {
  R s1, s2, s3;         // 2 (Z1 - 1), 2 Z2, 2 Z3   fv.h:91-93
  R drho, dn, dtg;
};
typedef JumpT<float> Jump;
template <typename R>
__device__ __forceinline__ JumpT<R> jump(R r1L, R nL, R tL, R unL, R utL, R r1R, R nR, R tR,
                                         R unR, R utR) {
#pragma clang fp contract(off)
  return JumpT<R>{r1L + r1R, unL + unR, utL + utR, r1R - r1L, nR - nL, tR - tL};
}

// Intermediate values of a Riemann solve that its transpose needs again.
template <typename R>
struct SolveT {
  R rS, rs;             // 1 / (2 Z1), 1 / sqrt(tmp3)
  R d1, d2, rdd;        // L_p S1 - s3, 1 / (d1 d2)
  R A1, A2;
};

// Riemann solve at an interface.  hbeta = BETA - 1.  The fluctuations
// amdq/apdq (fv.h:141-180) are not formed here: limited_flux() folds them with
// the correction flux.
template <typename R>
__device__ __forceinline__ void riemann(const JumpT<R>& j, R hbeta, IfaceT<R>& f, SolveT<R>& v) {
#pragma clang fp contract(off)
  const R s1 = j.s1, s2 = j.s2, s3 = j.s3, drho = j.drho, dn = j.dn, dtg = j.dtg;
  const R S1 = s1 + R(2);                           // 2 Z1
  const R rS = rcp(S1);
  const R tmp1 = s2 * rS;                           // Z2/Z1        fv.h:96
  // tmp1^2 - 2 Z2 tmp1 + 1 + 2 (BETA-1)(Z1-1)                      fv.h:97-101
  const R tmp3 = fma_(tmp1, fma_(s2, rS, -s2), fma_(hbeta, s1, R(1)));
  f.bad = !(tmp3 >= R(0));                          // fv.h:102
  const R rs = rsq(tmp3);
  const R L1 = fma_(tmp3, rs, tmp1), L2 = fma_(-tmp3, rs, tmp1);   // tmp1 +- sqrt, fv.h:105-107
  f.L1 = L1; f.L2 = L2; f.L3 = tmp1;
  f.s2 = s2; f.rS = rS;
  // fv.h:110-113: A_p = (L_p Z3 - 2 Z2 Z3)/(L_p Z1 - Z3) = s3 (L_p - s2)/(L_p S1 - s3),
  // with one reciprocal for both denominators (each is ~ +-2)
  const R d1 = fma_(L1, S1, -s3), d2 = fma_(L2, S1, -s3);
  const R rdd = rcp(d1 * d2);
  const R srd = s3 * rdd;
  const R A1 = (L1 - s2) * (d2 * srd);
  const R A2 = (L2 - s2) * (d1 * srd);
  const R hrs = R(0.5) * rs, dnl = fma_(-drho, L2, dn);
  const R a1 = dnl * hrs;                                       // fv.h:116-117
  const R a2 = fma_(-dnl, hrs, drho);                           // fv.h:118
  f.w.a1 = a1; f.w.w21 = a1 * L1; f.w.w31 = a1 * A1;
  f.w.a2 = a2; f.w.w22 = a2 * L2; f.w.w32 = a2 * A2;
  f.w.a3 = dtg - fma_(a1, A1, f.w.w32);                         // fv.h:119-125
  v = SolveT<R>{rS, rs, d1, d2, rdd, A1, A2};
}
template <typename R>
__device__ __forceinline__ void riemann(const JumpT<R>& j, R hbeta, IfaceT<R>& f) {
  SolveT<R> v;
  riemann(j, hbeta, f, v);
}

// W_p(a) . W_p(b); b is the operand that may come from a neighbouring lane
// (mul, then multiply-accumulates with b as the plain multiplicand)
template <typename R>
__device__ __forceinline__ R dot1(const WavesT<R>& a, const WavesT<R>& b) {
#pragma clang fp contract(off)
  return fma_(b.a1, a.a1, fma_(b.w21, a.w21, b.w31 * a.w31));
}
template <typename R>
__device__ __forceinline__ R dot2(const WavesT<R>& a, const WavesT<R>& b) {
#pragma clang fp contract(off)
  return fma_(b.a2, a.a2, fma_(b.w22, a.w22, b.w32 * a.w32));
}

// The limiter of a ratio r: t = (1+r)/4, mn = min(t, r), h = clamp(mn).  FP64
// (h alone): 1/4 as a scalar operand of the multiply-add -- the compiler's form
// adds into a register pair set to 1/4 first -- and the clamp as the minimum's
// output modifier, without a canonicalising v_max before it.
__device__ __forceinline__ void limit_half(float r, float& t, float& mn, float& h) {
  t = fma_(0.25f, r, 0.25f);
  mn = min_(t, r);
  h = clamp01(mn);
}
__device__ __forceinline__ void limit_half(double r, double& t, double& mn, double& h) {
  asm("v_fma_f64 %0, %2, %3, %3\n\tv_min_f64 %1, %0, %2 clamp"
      : "=&v"(t), "=v"(h) : "v"(r), "s"(0.25));
  mn = h;
}

// |W_1|^2, |W_2|^2
template <typename R>
__device__ __forceinline__ void norms(const WavesT<R>& w, R& n1, R& n2) {
#pragma clang fp contract(off)
  n1 = fma_(w.a1, w.a1, fma_(w.w21, w.w21, w.w31 * w.w31));
  n2 = fma_(w.a2, w.a2, fma_(w.w22, w.w22, w.w32 * w.w32));
}

// The dot product with the upwind neighbour by the sign of the speed s:
// dotl = W . W(k-1), dotr = W . W(k+1).
template <typename R>
__device__ __forceinline__ R upwind(R s, R dotl, R dotr) {
  return s > R(0) ? dotl : dotr;
}

// Fluctuations (fv.h:141-180) and correction flux fadd (fv.h:666-711) of one
// interface, folded into what the two adjacent cells need:
//   P = apdq - fadd = sum_p (max(s_p,0) - c_p) W_p   (cell on the + side)
//   M = amdq + fadd = sum_p (min(s_p,0) + c_p) W_p   (cell on the - side)
// with c_p = g_p phi_p / 2 and g_p = |s_p| (1 - |s_p| dt/d).  A wave with s_p = 0 enters
// neither fluctuation, as in the reference.
// n1, n2: norms(); up_p = W_p . W_p of the upwind neighbour (upwind()).
// kL3Product: be_3 = L3 - al_3 from the product L3 = s2 rS with one rounding
// (the x sweep, which has both factors at hand; the y sweep keeps L3 alone
// in its window).
//
// MC limiter phi(r) = max(0, min((1+r)/2, 2, 2r)) (fv.h:587-605), taken
// halved: h = phi/2 = clamp(min((1+r)/4, r), 0, 1), where the clamp is the VOP3
// output modifier of the min.  The reference sets phi = 1 where wnorm2 == 0;
// such a wave is the zero vector, so its correction phi*W is 0 for any
// finite phi.  Here wnorm2 == 0 gives r = NaN (0 * inf), which the clamp
// turns into 0 (finite), and the select is skipped.
template <typename R>
struct LimitT {         // per wave family
  R rn[3], r[3];        // 1/|W|^2, W . W(upwind) / |W|^2
  R t[3], mn[3], h[3];  // (1+r)/4, min(t, r), clamp(mn)
  R om[3], g[3];        // 1 - |s| dt/d, |s| (1 - |s| dt/d)
  R al[3];              // max(s, 0) - g h
};
template <bool kL3Product, typename R>
__device__ __forceinline__ void limited_flux(const IfaceT<R>& f, R n1, R n2, R up1, R up2, R up3,
                                             R dtd, R P[3], R M[3], LimitT<R>& v) {
#pragma clang fp contract(off)
  const WavesT<R>& w = f.w;
  const R n[3] = {n1, n2, w.a3 * w.a3};
  const R up[3] = {up1, up2, up3}, L[3] = {f.L1, f.L2, f.L3};
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    v.rn[p] = rcp(n[p]);
    v.r[p] = up[p] * v.rn[p];
    limit_half(v.r[p], v.t[p], v.mn[p], v.h[p]);
    const R s = fabs(L[p]);
    v.om[p] = fma_(-s, dtd, R(1));
    v.g[p] = s * v.om[p];
    v.al[p] = fma_(-v.g[p], v.h[p], fmax2(L[p], R(0)));
  }
  // al_p = max(s_p, 0) - c_p; be_p = min(s_p, 0) + c_p = s_p - al_p
  const R al1 = v.al[0], al2 = v.al[1], al3 = v.al[2];
  const R be1 = f.L1 - al1, be2 = f.L2 - al2;
  const R be3 = kL3Product ? fma_(f.s2, f.rS, -al3) : f.L3 - al3;
  P[0] = fma_(al1, w.a1, al2 * w.a2);
  P[1] = fma_(al1, w.w21, al2 * w.w22);
  P[2] = fma_(al3, w.a3, fma_(al1, w.w31, al2 * w.w32));
  M[0] = fma_(be1, w.a1, be2 * w.a2);
  M[1] = fma_(be1, w.w21, be2 * w.w22);
  M[2] = fma_(be3, w.a3, fma_(be1, w.w31, be2 * w.w32));
}
template <bool kL3Product, typename R>
__device__ __forceinline__ void limited_flux(const IfaceT<R>& f, R n1, R n2, R up1, R up2, R up3,
                                             R dtd, R P[3], R M[3]) {
  LimitT<R> v;
  limited_flux<kL3Product>(f, n1, n2, up1, up2, up3, dtd, P, M, v);
}

}  // namespace fvna

#endif  // FIVONAGI_APPS_NA_SOLVER_H
