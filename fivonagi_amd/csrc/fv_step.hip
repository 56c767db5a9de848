// fv_step.hip -- the fused FiVoNAGI time step for gfx950 (MI355X).
//
// One launch = one step attempt of every active instance.  It replaces the
// reference's per-step sequence (common/main.cu:310-635): texCpy, boundary,
// getWavesSpeedsCFL_y, step_y, calcLimiters_y, writeLimiters_y, the same four
// in x, 21 reduceCFL launches, reduceCFL2, source, update_T, update_dt and the
// seven blocking device->host copies.
//
// Work decomposition ("march"): one wave64 per work item, up to four items of
// a strip, one above the other, per workgroup.  Lane l owns column x0 - 3 + l;
// the wave marches upward through the rows of its strip:
//   load row r+1 (prefetch; boundary rules applied when the row is consumed)
//   -> y-Riemann at interface r        (registers, same lane)
//   -> y-limiter at interface r-1      (3-interface register window)
//   -> q_y(r-2)                        (first + second order, fused)
//   -> x-Riemann/limiter on row r-2    (neighbours via DPP wave_shr/wave_shl)
//   -> q_xy(r-2)
//   -> source on row r-4               (3-row register window + DPP)
//   -> store row r-4 (lanes 3..60)
// The loop is unrolled three times so the period-3 register windows rotate
// by renaming instead of moves.
//
// Seams: output row y needs interfaces y-2 .. y+3, so a lone item of H rows
// solves H+5 y interfaces, H+3 y limiters and H+2 x rows.  Inside a workgroup
// nothing is solved twice: each wave leaves what its first rows make (the
// first interface, the next one's dot products and M, the first two rows of
// q_xy) in LDS, one barrier after its sixth row publishes it, and the wave
// below ends its march on those values.  Only the topmost wave of a workgroup
// marches the five rows past its last.
//
// The march is bound by VALU issue (about 250 instructions per row of a wave)
// and, on small grids, by the length of the longest wave's march, so both gain
// from rows not repeated: a wave of 18 rows marched 21.3 rows' worth alone and
// 18.8 in a group of four, and a group of 16 rows marches 6 steps where a lone
// item needed 17.  Per step, one wave per workgroup against groups of four:
// 4096x1024 40.7 -> 36.9 us, 2048x2048 43.2 -> 37.5, 1024x1024 20.9 -> 16.6,
// 400x400 16.4 -> 8.7 (FP32).  Waves per group: two gave 38.4 on 4096x1024.
// Then 13 VALU instructions fewer per row (neighbour operands by DPP, the CFL
// maximum under the mask, dt/d carried from row to row): 37.3 -> 36.1 us on
// 4096x1024, 64.7 -> 62.3 on 4096x2048, 237 -> 228 on 8192x4096.
//
// CFL and accept/reject: each wave reduces its cells' cfl to one float and
// folds it into its group's 128-byte line (8 groups per instance) with one
// relaxed agent-scope atomicMax that nothing waits for.  Attempt a's maxima
// are read by every wave of launch a+1, which decides accept/reject, dt, T
// and the ping-pong index of attempt a+1 itself (advance(), identical in
// every wave); one wave per instance stores the result for the launch after.
// The control blocks and reduction slots rotate with the attempt index
// (2 control blocks, 3 slot sets), so no launch reads what it writes and the
// step ends when its last wave ends -- no ticket chain, no fences.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../apps/apps.h"
#include "../apps/hifu-beam/data_collect.h"
#include "../apps/taylor-angle-xy/data_collect.h"
#include "../apps/na/solver.h"
#include "../apps/na/source.h"
#include "fv_lanes.h"
#include "fv_types.h"

namespace fv {

typedef __attribute__((address_space(1))) float gfloat;
typedef __attribute__((address_space(1))) const float cgfloat;
typedef __attribute__((address_space(4))) const float kfloat;   // read-only: scalar loads
typedef __attribute__((address_space(1))) double gdouble;
typedef __attribute__((address_space(1))) const double cgdouble;
typedef __attribute__((address_space(4))) const double kdouble;
// the same three per real type R (float: the FP32 path, double: FP64)
template <typename R> struct Mem;
template <> struct Mem<float> { typedef gfloat g; typedef cgfloat cg; typedef kfloat k; };
template <> struct Mem<double> { typedef gdouble g; typedef cgdouble cg; typedef kdouble k; };

typedef __attribute__((address_space(1))) char gchar;
typedef __attribute__((address_space(1))) const char cgchar;

// Loads/stores at a 32-bit byte offset from a uniform base: the base stays in
// scalar registers (global_load/store with saddr) and each lane carries one
// 32-bit offset instead of a 64-bit address per field.
__device__ __forceinline__ float ldg(cgfloat* base, uint32_t off) {
  return *(cgfloat*)((cgchar*)base + off);
}
__device__ __forceinline__ void stg(gfloat* base, uint32_t off, float v) {
  *(gfloat*)((gchar*)base + off) = v;
}
__device__ __forceinline__ double ldg(cgdouble* base, uint32_t off) {
  return *(cgdouble*)((cgchar*)base + off);
}
__device__ __forceinline__ void stg(gdouble* base, uint32_t off, double v) {
  *(gdouble*)((gchar*)base + off) = v;
}

// s_waitcnt vmcnt(0) lgkmcnt(0) with expcnt left at its maximum (gfx9 encoding)
constexpr int kWaitLoads = 0x0070;

__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t uni64(int64_t v) {
  const uint64_t u = (uint64_t)v;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ float unif(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ double unif(double v) {
  return __longlong_as_double(uni64(__double_as_longlong(v)));
}

// S <- max(S, |a|, |b|) (the largest speed: |L3| <= max(|L1|, |L2|), whose mean
// it is) on the lanes whose bit of the uniform mask is set: one
// VALU instruction under the mask as the execution mask (the march's lanes are
// all active around it), where a select and two maxima take three.
__device__ __forceinline__ void masked_max(uint64_t mask, float& S, float a, float b) {
  uint64_t keep;
  asm("s_and_saveexec_b64 %1, %4\n\t"
      "v_max3_f32 %0, %0, |%2|, |%3|\n\t"
      "s_mov_b64 exec, %1"
      : "+v"(S), "=&s"(keep)
      : "v"(a), "v"(b), "s"(mask)
      : "scc");
}
__device__ __forceinline__ void masked_max(uint64_t mask, double& S, double a, double b) {
  uint64_t keep;
  asm("s_and_saveexec_b64 %1, %4\n\t"
      "v_max_f64 %0, %0, |%2|\n\t"
      "v_max_f64 %0, %0, |%3|\n\t"
      "s_mov_b64 exec, %1"
      : "+v"(S), "=&s"(keep)
      : "v"(a), "v"(b), "s"(mask)
      : "scc");
}

// fvna::upwind of the x sweep: dl on the lanes with a positive speed, else the
// right neighbour's dl, whose move folds into the select; and fvna::norms, whose
// multiply-adds fill the two wait states a select needs after the comparison
// that writes its mask.
// (FP64: each half of the value by a select of its own.  With the masked maxima
// and the limiter's forms in solver.h 409 -> 376 VALU instructions per FP64 row,
// a step of 2048x1024 40.1 -> 38.4 us, of 4096x1024 70.0 -> 66.7.)
__device__ __forceinline__ void upwind_x(const fvna::IfaceT<float>& f, float dl1, float dl2,
                                         float dl3, float& up1, float& up2, float& up3, float& n1,
                                         float& n2) {
  asm("v_cmp_lt_f32_e32 vcc, 0, %5\n\t"
      "v_mul_f32_e32 %3, %13, %13\n\t"
      "v_mul_f32_e32 %4, %16, %16\n\t"
      "v_cndmask_b32_dpp %0, %8, %8, vcc wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "v_cmp_lt_f32_e32 vcc, 0, %6\n\t"
      "v_fmac_f32_e32 %3, %12, %12\n\t"
      "v_fmac_f32_e32 %4, %15, %15\n\t"
      "v_cndmask_b32_dpp %1, %9, %9, vcc wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
      "v_cmp_lt_f32_e32 vcc, 0, %7\n\t"
      "v_fmac_f32_e32 %3, %11, %11\n\t"
      "v_fmac_f32_e32 %4, %14, %14\n\t"
      "v_cndmask_b32_dpp %2, %10, %10, vcc wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1"
      : "=&v"(up1), "=&v"(up2), "=&v"(up3), "=&v"(n1), "=&v"(n2)
      : "v"(f.L1), "v"(f.L2), "v"(f.L3), "v"(dl1), "v"(dl2), "v"(dl3), "v"(f.w.a1), "v"(f.w.w21),
        "v"(f.w.w31), "v"(f.w.a2), "v"(f.w.w22), "v"(f.w.w32)
      : "vcc");
}
__device__ __forceinline__ uint32_t lo32(double v) {
  return (uint32_t)(uint64_t)__double_as_longlong(v);
}
__device__ __forceinline__ uint32_t hi32(double v) {
  return (uint32_t)((uint64_t)__double_as_longlong(v) >> 32);
}
__device__ __forceinline__ double join64(uint32_t lo, uint32_t hi) {
  return __longlong_as_double((long long)((uint64_t)hi << 32 | lo));
}
__device__ __forceinline__ void upwind_x(const fvna::IfaceT<double>& f, double dl1, double dl2,
                                         double dl3, double& up1, double& up2, double& up3,
                                         double& n1, double& n2) {
  uint32_t l1, h1, l2, h2, l3, h3;
#define FV_SEL(d, s) \
  "v_cndmask_b32_dpp " d ", " s ", " s ", vcc wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
  asm("v_cmp_lt_f64_e32 vcc, 0, %8\n\t"
      "v_mul_f64 %6, %19, %19\n\t"
      "v_mul_f64 %7, %22, %22\n\t"
      FV_SEL("%0", "%11") FV_SEL("%1", "%12")
      "v_cmp_lt_f64_e32 vcc, 0, %9\n\t"
      "v_fmac_f64_e32 %6, %18, %18\n\t"
      "v_fmac_f64_e32 %7, %21, %21\n\t"
      FV_SEL("%2", "%13") FV_SEL("%3", "%14")
      "v_cmp_lt_f64_e32 vcc, 0, %10\n\t"
      "v_fmac_f64_e32 %6, %17, %17\n\t"
      "v_fmac_f64_e32 %7, %20, %20\n\t"
      FV_SEL("%4", "%15") FV_SEL("%5", "%16")
      : "=&v"(l1), "=&v"(h1), "=&v"(l2), "=&v"(h2), "=&v"(l3), "=&v"(h3), "=&v"(n1), "=&v"(n2)
      : "v"(f.L1), "v"(f.L2), "v"(f.L3), "v"(lo32(dl1)), "v"(hi32(dl1)), "v"(lo32(dl2)),
        "v"(hi32(dl2)), "v"(lo32(dl3)), "v"(hi32(dl3)), "v"(f.w.a1), "v"(f.w.w21), "v"(f.w.w31),
        "v"(f.w.a2), "v"(f.w.w22), "v"(f.w.w32)
      : "vcc");
#undef FV_SEL
  up1 = join64(l1, h1);
  up2 = join64(l2, h2);
  up3 = join64(l3, h3);
}

// Pins a value in a register here: its computation cannot sink into a
// branch that follows, so a cross-lane move feeding it stays in its block
// and folds into its user.
__device__ __forceinline__ void pin(float& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin(double& v) { asm volatile("" : "+v"(v)); }

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ float fmax_(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double fmax_(double a, double b) { return fmax(a, b); }

__device__ __forceinline__ uint32_t amax_relaxed(uint32_t* p, uint32_t v) {
  return __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t aadd_relaxed(uint32_t* p, uint32_t v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t axchg_relaxed(uint32_t* p, uint32_t v) {
  return __hip_atomic_exchange(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The per-group cfl maximum of an instance, as float or double bits
// (non-negative values order like their bit patterns).
template <typename R> struct CflSlot;
template <> struct CflSlot<float> {
  typedef uint32_t bits;
  static __device__ __forceinline__ bits load(const GroupSlot& g) { return g.cfl_bits; }
  static __device__ __forceinline__ void clear(GroupSlot& g) { g.cfl_bits = 0u; }
  static __device__ __forceinline__ void fold_in(GroupSlot& g, float v) {
    __hip_atomic_fetch_max(&g.cfl_bits, __float_as_uint(v), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ float value(bits b) { return __uint_as_float(b); }
  static __device__ __forceinline__ bits lane_max(bits g) {
    uint32_t m = 0u;
#pragma unroll
    for (int k = 0; k < kGroups; ++k) m = max(m, (uint32_t)__builtin_amdgcn_readlane(g, k));
    return m;
  }
};
template <> struct CflSlot<double> {
  typedef uint64_t bits;
  static __device__ __forceinline__ bits load(const GroupSlot& g) { return g.cfl_bits64; }
  static __device__ __forceinline__ void clear(GroupSlot& g) { g.cfl_bits64 = 0ull; }
  static __device__ __forceinline__ void fold_in(GroupSlot& g, double v) {
    __hip_atomic_fetch_max(&g.cfl_bits64, (uint64_t)__double_as_longlong(v), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
  }
  static __device__ __forceinline__ double value(bits b) {
    return __longlong_as_double((long long)b);
  }
  static __device__ __forceinline__ bits lane_max(bits g) {
    uint64_t m = 0ull;
#pragma unroll
    for (int k = 0; k < kGroups; ++k) {
      const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)g, k);
      const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(g >> 32), k);
      m = max(m, ((uint64_t)hi << 32) | lo);
    }
    return m;
  }
};

// What attempt a's reduction slots say about it, with the control block it
// ran with.  fold_load issues every load before anything is decided, so the
// fold costs one memory round trip.
// R: the instance's real type (its cfl reduction is in R).
template <typename R>
struct FoldRaw {
  Ctl p;          // control block attempt a ran with
  uint32_t ran, errf;
  typename CflSlot<R>::bits gbits;
};
template <typename R>
struct Fold {
  Ctl p;
  R cfl;          // max cfl over the counted cells of attempt a
  int state;      // kFoldIdle, kFoldError, kFoldAccept, kFoldReject
};
constexpr int kFoldIdle = 0, kFoldError = 1, kFoldAccept = 2, kFoldReject = 3;

template <typename R>
__device__ __forceinline__ FoldRaw<R> fold_load(const Ctl* __restrict__ c,
                                                const SyncSlots* __restrict__ sl) {
  FoldRaw<R> r;
  Ctl& p = r.p;
  p.dt = c->dt; p.T = c->T; p.last_cfl = c->last_cfl;
  p.drive_s = c->drive_s; p.drive_c = c->drive_c;
  p.n_acc = c->n_acc; p.n_rej = c->n_rej; p.n_att = c->n_att;
  p.target_acc = c->target_acc;
  p.cur = c->cur; p.err = c->err;
  p.dtx = c->dtx; p.dty = c->dty; p.ddx2 = c->ddx2; p.ddy2 = c->ddy2;
  p.mdx = c->mdx; p.mdy = c->mdy; p.T_stop = c->T_stop;
  r.ran = sl->ran;
  r.errf = sl->err_flag;
  // the group maxima with one vector load (lane l reads group l % kGroups)
  // rather than kGroups scalar loads
  r.gbits = CflSlot<R>::load(sl->grp[__lane_id() & (kGroups - 1)]);
  return r;
}

template <typename R>
__device__ __forceinline__ Fold<R> fold_decide(const FoldRaw<R>& r, double cfl_max, bool presc) {
  Fold<R> f;
  f.p = r.p;
  f.p.n_acc = uni64(r.p.n_acc); f.p.n_rej = uni64(r.p.n_rej); f.p.n_att = uni64(r.p.n_att);
  f.p.target_acc = uni64(r.p.target_acc);
  f.p.cur = uni(r.p.cur); f.p.err = uni(r.p.err);
  f.p.mdx = uni(r.p.mdx); f.p.mdy = uni(r.p.mdy);
  const R cfl = CflSlot<R>::value(CflSlot<R>::lane_max(r.gbits));
  f.cfl = cfl;
  const bool acc = presc || ((double)cfl < cfl_max);
  f.state = !uni(r.ran) ? kFoldIdle
                        : (uni(r.errf) ? kFoldError : (acc ? kFoldAccept : kFoldReject));
  return f;
}

// Ping-pong index attempt a+1 reads (known before the rest of advance()).
template <typename R>
__device__ __forceinline__ int next_cur(const Fold<R>& f) {
  return f.state == kFoldAccept ? (f.p.cur ^ 1) : f.p.cur;
}

using fvbc::md_shift;

// Control block of attempt a+1 from attempt a's fold: common/main.cu:199-230
// with a clean retry on rejection.  log: record the control block an accepted
// step ran with (adjoint runs: its recompute and reverse pass replay it); every
// writer records the same values.
template <typename R>
__device__ Ctl advance(const InstDesc& D, const Fold<R>& f, bool log) {
  const Ctl& p = f.p;
  Ctl o = p;
  if (f.state == kFoldIdle) return o;   // attempt a did not run (instance done or stopped)
  if (f.state == kFoldError) {
    o.err = 2;                         // imaginary eigenvalue: step discarded, instance stops
    return o;
  }
  const double cfl = (double)f.cfl;
  const bool presc = D.dt_seq != nullptr;
  const bool acc = f.state == kFoldAccept;
  const int64_t att = p.n_att + 1;
  o.n_att = att;
  o.last_cfl = cfl;
  double T = p.T;
  if (acc) {
    if (log && D.ctl_log && __lane_id() == 0) {
      const int64_t idx = p.n_acc - D.log_base;
      if (idx >= 0 && idx < D.log_len) D.ctl_log[idx] = p;
    }
    T = p.T + p.dt;
    o.T = T;
    o.n_acc = p.n_acc + 1;
    o.cur = p.cur ^ 1;
    if (D.md_on) {
      o.mdx = p.mdx + md_shift(T, D.md_t, D.md_vx, D.dx, p.mdx);
      o.mdy = p.mdy + md_shift(T, D.md_t, D.md_vy, D.dy, p.mdy);
    }
  } else {
    o.n_rej = p.n_rej + 1;
  }
  double ndt;
  if (presc) {
    // attempt att uses dt[att]; past the end the dt is kept, and an attempt
    // that would run with it is refused (prescribed_exhausted)
    ndt = (att < D.dt_seq_len) ? D.dt_seq[att] : p.dt;
  } else {
    ndt = p.dt * D.cfl_wish / cfl;
    if (!acc && ndt > p.dt * 0.9) ndt = p.dt * 0.9;
  }
  o.dt = ndt;
  o.dtx = (float)(ndt * D.inv_dx);
  o.dty = (float)(ndt * D.inv_dy);
  o.ddx2 = (float)(ndt * D.dif_x);
  o.ddy2 = (float)(ndt * D.dif_y);
  // drive phase omega*T in turns, reduced in double to [0, 1); the step uses
  // sin/cos in FP32
  const double turns = D.omega_turns * T;
  if (sizeof(R) == 4) {
    float fs, fc;
    sincospif((float)(2.0 * (turns - floor(turns))), &fs, &fc);
    o.drive_s = fs;
    o.drive_c = fc;
  } else {                      // FP64 instances: the drive phase in double
    double ds, dc;
    sincospi(2.0 * (turns - floor(turns)), &ds, &dc);
    o.drive_s = ds;
    o.drive_c = dc;
  }
  return o;
}

// An attempt that would run (instance not done, not stopped, no error) while
// its prescribed dt sequence has no entry for it: error 9 instead of running.
// The check sits where an attempt is about to run, not where the last entry
// is used, so a sequence of exactly n entries runs n steps.
__device__ __forceinline__ void prescribed_exhausted(const InstDesc& D, Ctl& P) {
  if (D.dt_seq != nullptr && P.err == 0 && P.n_att >= D.dt_seq_len &&
      P.n_acc < P.target_acc && P.T < P.T_stop)
    P.err = 9;
}

// Control block of the attempt a launch runs (phase = a mod 6), read-only.
template <typename R>
__device__ __forceinline__ Ctl current_t(const InstDesc& D, int phase, bool log) {
  Ctl P = advance(D,
                  fold_decide(fold_load<R>(D.ctl + (phase & 1), D.sync + (phase + 2) % 3),
                              D.cfl_max, D.dt_seq != nullptr),
                  log);
  prescribed_exhausted(D, P);
  return P;
}
__device__ __forceinline__ Ctl current(const InstDesc& D, int phase, bool log) {
  return D.fp64 ? current_t<double>(D, phase, log) : current_t<float>(D, phase, log);
}

// The fold of attempt a-1 as the launch of attempt a (phase) forms it.
template <typename R>
__device__ __forceinline__ Fold<R> fold_prev(const InstDesc& D, int phase) {
  return fold_decide(fold_load<R>(D.ctl + (phase & 1), D.sync + (phase + 2) % 3), D.cfl_max,
                     D.dt_seq != nullptr);
}

// Data collection of an attempt (phase, its fold F): if it was accepted, record
// its new T and its cfl (row 0 and row 1, entry n - 1 - n0frame) and the app's
// measurement (collect_hifu, collect_taylor) into the instance's measurement
// grid (data_collect.h of either app).  Thread tid = column.
template <typename R>
__device__ void collect_attempt(const InstDesc& D, const Fold<R>& F, int phase, int tid) {
  typename Mem<R>::g* __restrict__ m = (typename Mem<R>::g*)D.measure;
  if (m == nullptr || F.state != kFoldAccept) return;
  const Ctl& P = F.p;
  const double T = P.T + P.dt;                       // update_T
  const int nx = D.nx;
  // While T <= 0 the reference zeroes the whole grid every step and records
  // nothing (data_collect.h:22-30, both apps).  Here the grid is zeroed when
  // collection is switched on, and nothing writes it while T <= 0, so it is
  // already zero: the pass over the grid is skipped.
  if (T <= 0.0) return;
  const int64_t nf = P.n_acc - D.n0frame;          // n - 1 - n0frame, n = n_acc + 1
  if (nf >= nx) {                                   // simError 4
    if (tid == 0) aadd_relaxed(D.collect_err, 4u);
    return;
  }
  if (tid == 0) {                                   // T and cfl of the step
    m[nf] = R(T);
    m[nf + nx] = F.cfl;
  }
  if (D.bc == kBcTaylor)
    fvbc::collect_taylor<R>(D, P, T, (R*)m, tid);
  else
    fvbc::collect_hifu<R>(D, P, (const R*)D.stage + (phase & 1) * nx, T, nf, (R*)m, tid);
}

// Closed-form ghost ring of a Taylor-shock instance (apps/taylor-angle-xy/
// boundary.h:38-55) at T and window offset (mdx, mdy), into the ring of its
// buffer b, or its grid.  The values depend on the cell and on T only, never on
// the state.  Cells k0, k0 + dk, ... of the ring (2 cells wide).
__device__ __forceinline__ void taylor_ring(const InstDesc& D, double T, int b, int mdx, int mdy,
                                            bool to_ring, int k0, int dk) {
  const int nx = D.nx, ny = D.ny;
  const int ring = 4 * nx + 4 * (ny - 4);
  for (int k = k0; k < ring; k += dk) {
    int i, j;
    if (k < 4 * nx) {            // rows 0, 1, ny-2, ny-1
      const int rr = k / nx;
      i = k - rr * nx;
      j = rr < 2 ? rr : ny - 4 + rr;
    } else {                     // columns 0, 1, nx-2, nx-1 of rows 2..ny-3
      const int kk = k - 4 * nx;
      const int cc = kk / (ny - 4);
      j = 2 + (kk - cc * (ny - 4));
      i = cc < 2 ? cc : nx - 4 + cc;
    }
    // the closed form is taken at the cell's position in the unmoved frame
    // (apps/taylor-angle-xy/boundary.h:45-49: i + MDX, j + MDY)
    const size_t size = D.fp64 ? sizeof(double) : sizeof(float);
    const size_t o = to_ring ? D.ring + size * (size_t)k
                             : size * ((size_t)j * (size_t)nx + (size_t)i);
    if (D.fp64) {
      fvbc::Cell<double> c;
      fvbc::Taylor::prepass(D, T, i + mdx, j + mdy, c);
      *(double*)((char*)D.q[b][0] + o) = c.q1;
      *(double*)((char*)D.q[b][1] + o) = c.q2;
      *(double*)((char*)D.q[b][2] + o) = c.q3;
    } else {
      fvbc::Cell<float> c;
      fvbc::Taylor::prepass(D, T, i + mdx, j + mdy, c);
      *(float*)((char*)D.q[b][0] + o) = c.q1;
      *(float*)((char*)D.q[b][1] + o) = c.q2;
      *(float*)((char*)D.q[b][2] + o) = c.q3;
    }
  }
}

// What a step launch does beside the step, in workgroups of its own: the data
// collection of the attempt before it (collect), whose fold is known now and
// whose new state is this attempt's input, and the ghost ring of the attempt
// after it, for the T and window offset that follow if this one is accepted
// (else the ring this attempt reads stays the right one).  As launches of their
// own between the steps the two took 4.8 us each.
// part: the workgroup's place among its instance's `beside`, the first
// `collect` of them collect.
template <typename R>
__device__ __forceinline__ void beside_step(const InstDesc& D, int phase, int part, int beside,
                                            int collect) {
  const int threads = kLanes * kGroupWaves;
  const Fold<R> F = fold_prev<R>(D, phase);
  if (part < collect) {
    collect_attempt<R>(D, F, phase + 5, part * threads + (int)threadIdx.x);   // phase - 1 (mod 6)
    return;
  }
  if (D.bc != kBcTaylor || D.ring == 0) return;
  Ctl P = advance<R>(D, F, false);
  prescribed_exhausted(D, P);
  if (P.err != 0 || P.n_acc >= P.target_acc || !(P.T < P.T_stop)) return;
  const double T = P.T + P.dt;
  int mdx = P.mdx, mdy = P.mdy;
  if (D.md_on) {
    mdx += md_shift(T, D.md_t, D.md_vx, D.dx, P.mdx);
    mdy += md_shift(T, D.md_t, D.md_vy, D.dy, P.mdy);
  }
  taylor_ring(D, T, P.cur ^ 1, mdx, mdy, true, (part - collect) * threads + (int)threadIdx.x,
              (beside - collect) * threads);
}

template <typename R>
struct Row {         // one cell of a row as the y sweep sees it
  R q1, q2, q3;      // rho', rho u, rho v
  R un, ut;          // y normal velocity v = q3/rho, tangential u = q2/rho
  uint64_t cm;       // the row's CFL lane mask (uniform)
};

template <typename R>
struct YI {          // y interface with its limited flux towards the + cell
  fvna::IfaceT<R> f;
  R dl[3];           // W_p . W_p of the interface below (one per wave family)
  R P[3];            // apdq - fadd, in (density, normal, tangential) order
};

template <typename R>
struct XY {          // one cell of q_xy, with its velocities for the source
  R q1, q2, q3, u, v;
};

// What a wave hands to the wave below it, per lane: the waves and speeds of its
// first interface (y0-2), the dot products of the next (y0-1), that
// interface's M, and its first rows of q_xy (y0-1: the cell and its
// velocities; y0: the velocities).
constexpr int kSeamW = 0, kSeamL = 7, kSeamDl = 10, kSeamM = 13, kSeamX = 16, kSeamFields = 23;
template <typename R>
__device__ __forceinline__ void seam_put(R* s, int field, R v) {
  s[field * kLanes] = v;
}
template <typename R>
__device__ __forceinline__ R seam_get(const R* s, int field) {
  return s[field * kLanes];
}
// every wave's seam values are in LDS and visible to its workgroup (LDS only:
// the prefetched row stays in flight)
__device__ __forceinline__ void seam_publish() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
template <int kT>
using At = std::integral_constant<int, kT>;

// One work item of attempt `phase` (mod 6) of an instance whose ghost cells
// follow the boundary policy BC (apps/<app>/boundary.h).
// kOne: the launch covers a single instance.  The control blocks and reduction
// slots of this attempt are passed directly (ctl_in = the first instance's
// control block of attempt a = ctl + a % 2, sync_in = its slots of attempt a-1 =
// sync + (a + 2) % 3; the next instance's follow two and three on), so the
// fold's loads go out together with the work item's (kOne), or with the instance
// description's rather than after it (16 uneven instances 53.1 -> 52.7 us).
// kExt: some instance has a moving window or the HIFU boundary.
//  - Moving window: the shift that follows an accepted step (moveDomain,
//    common/main.cu:109-164) is folded into the stores: cell (i, j) of the new
//    state lands at (i - sx, j - sy), and also stays at (i, j) when
//    (i + sx, j + sy) is off the grid (moveDomain's else branch); every cell
//    of the output is written exactly once.  A rejected attempt's output is
//    discarded, as without the window.
//  - the HIFU app's packet and data collection staging.
// R: float (FP32 path) or double (FP64 instances: state, tables, arithmetic
// and the cfl reduction in double; the reference's PRECISION=2).
template <typename R, bool kOne, bool kExt, class BC>
__device__ __forceinline__ void step_impl(const InstDesc* __restrict__ insts, const WorkItem& it,
                                          const uint64_t* __restrict__ rowmask, int phase,
                                          const Ctl* __restrict__ ctl_in,
                                          const SyncSlots* __restrict__ sync_in,
                                          R (*seam)[kSeamFields][kLanes]) {
#pragma clang fp contract(off)
  const InstDesc& D = insts[kOne ? 0 : it.inst];
  const int local = it.local;
  const int lane = threadIdx.x & (kLanes - 1);

  // ---- the previous attempt's reduction, folded: accept/reject decides
  // which buffer this attempt reads, so its first row can be requested
  // before the rest of the control block (dt, T, drive phase) is formed ----
  // the instance's geometry and both buffers' pointers are requested with
  // the fold's loads; the asm barrier keeps the compiler from re-loading a
  // pointer by the buffer index once accept/reject is known
  const int nx = D.nx, ny = D.ny;
  typedef typename Mem<R>::g gR;
  typedef typename Mem<R>::cg cgR;
  R* qb[2][3];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int f = 0; f < 3; ++f) qb[h][f] = (R*)D.q[h][f];
  double cfl_max = D.cfl_max;
  const double* dt_seq = D.dt_seq;
  const int hist_state = kExt && sizeof(R) == 4 ? D.hist_state : 0;
  fvbc::Tables tb{D.edge_c, D.edge_s, D.hifu_tab};
  const FoldRaw<R> FR = fold_load<R>(ctl_in + (kOne ? 0 : 2 * it.inst),
                                     sync_in + (kOne ? 0 : 3 * it.inst));
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int f = 0; f < 3; ++f) asm volatile("" : "+s"(qb[h][f]));
  asm volatile("" : "+s"(cfl_max), "+s"(dt_seq));
  if (BC::kRowData) asm volatile("" : "+s"(tb.edge_c), "+s"(tb.edge_s));
  const Fold<R> F = fold_decide(FR, cfl_max, dt_seq != nullptr);
  const int cur = next_cur(F);

  cgR* __restrict__ in1 = (cgR*)(cur ? qb[1][0] : qb[0][0]);
  cgR* __restrict__ in2 = (cgR*)(cur ? qb[1][1] : qb[0][1]);
  cgR* __restrict__ in3 = (cgR*)(cur ? qb[1][2] : qb[0][2]);
  gR* __restrict__ o1 = (gR*)(cur ? qb[0][0] : qb[1][0]);
  gR* __restrict__ o2 = (gR*)(cur ? qb[0][1] : qb[1][1]);
  gR* __restrict__ o3 = (gR*)(cur ? qb[0][2] : qb[1][2]);
  if (hist_state) {
    // from the kept state to the next slot: one store per cell where a state
    // buffer and its kept copy take two (gradient of 200 steps of 2048x1024 19.1 ->
    // 18.7 ms)
    const size_t n = (size_t)nx * (size_t)ny;
    const uint32_t t = (uint32_t)(F.p.n_acc + (F.state == kFoldAccept ? 1 : 0) - D.log_base);
    R* const s = (R*)D.hist + (size_t)t * 3 * n;
    in1 = (cgR*)s;           o1 = (gR*)(s + 3 * n);
    in2 = (cgR*)(s + n);     o2 = (gR*)(s + 4 * n);
    in3 = (cgR*)(s + 2 * n); o3 = (gR*)(s + 5 * n);
  }

  const int i = it.x0 - kHalo + lane;
  const bool col_in = (i >= 0) && (i < nx);
  const bool col_x = col_in && (i >= 1);     // lane holds an x interface of the grid
  const int ic = min(max(i, 0), nx - 1);
  const bool col_int = (i >= 2) && (i <= nx - 3);
  const bool out_lane = (lane >= kHalo) && (lane < kLanes - kHalo) && (i < nx);
  const int y0 = it.y0, y1 = it.y1;
  // CFL lane masks of the strip's rows: cm[j], j in [0, ny)
  const uint64_t* __restrict__ cm = rowmask + (it.mrow - y0);

  // the lane's ghost-cell source columns (the app's boundary policy; Taylor
  // ghost cells are copies of the buffer's ghost ring, or of the grid)
  constexpr uint32_t kSz = sizeof(R);
  fvbc::LaneMap lm;
  lm.ring = D.ring;
  lm.ny = ny;
  BC::lane(ic, nx, lm, kSz);
  const uint32_t row_bytes = kSz * (uint32_t)nx;

  // raw (unpatched) load of row r, with its CFL lane mask and table entries; the
  // boundary patch is applied when the row is consumed one iteration later,
  // so the load latency overlaps a full step
  auto load_raw = [&](int r, R& a, R& b, R& c, uint64_t& k, fvbc::RowData<R>& h) {
    const int rc = min(max(r, 0), ny - 1);
    const uint32_t o = BC::offset(rc, ny, lm, row_bytes, kSz);
    a = ldg(in1, o);
    b = ldg(in2, o);
    c = ldg(in3, o);
    k = cm[rc];
    if (BC::kRowData) BC::template load_row<R>(tb, rc, h);
  };
  R n1, n2, n3;
  uint64_t nk;
  fvbc::RowData<R> nh{R(0), R(0), R(0), R(0), R(0), R(0)};
  load_raw(it.y0 - kHalo, n1, n2, n3, nk, nh);   // in flight during advance()

  // ---- control block of this attempt ----
  Ctl P = advance<R>(D, F, local == 0);
  prescribed_exhausted(D, P);
  const bool runs = P.err == 0 && P.n_acc < P.target_acc && P.T < P.T_stop;
  if (local == 0 && lane == 0) {
    // one wave per instance: publish the control block for the next launch,
    // clear the slots the next attempt reduces into, mark this attempt
    D.ctl[(phase + 1) & 1] = P;
    SyncSlots* nx_sl = D.sync + (phase + 1) % 3;
#pragma unroll
    for (int k = 0; k < kGroups; ++k) CflSlot<R>::clear(nx_sl->grp[k]);
    nx_sl->err_flag = 0u;
    nx_sl->ran = 0u;
    if (runs) D.sync[phase % 3].ran = 1u;
  }
  if (!runs) return;
  R dtx, dty, ddx2, ddy2, sin_t, cos_t, hbeta;
  if (sizeof(R) == 4) {     // the control block's FP32 forms
    dtx = unif(P.dtx); dty = unif(P.dty);
    ddx2 = unif(P.ddx2); ddy2 = unif(P.ddy2);
    sin_t = unif((float)P.drive_s); cos_t = unif((float)P.drive_c);
    hbeta = R(0.5f * D.beta2m2);            // BETA - 1
  } else {                  // FP64: the same quantities in double
    dtx = unif(R(P.dt * D.inv_dx)); dty = unif(R(P.dt * D.inv_dy));
    ddx2 = unif(R(P.dt * D.dif_x)); ddy2 = unif(R(P.dt * D.dif_y));
    sin_t = unif(R(P.drive_s)); cos_t = unif(R(P.drive_c));
    hbeta = R(D.hbeta_d);
  }
  // shift of the window after this attempt, if it is accepted
  int sx = 0, sy = 0;
  if (kExt && D.md_on) {
    const double Tn = P.T + P.dt;
    sx = uni(md_shift(Tn, D.md_t, D.md_vx, D.dx, P.mdx));
    sy = uni(md_shift(Tn, D.md_t, D.md_vy, D.dy, P.mdy));
  }
  const bool stage_on = kExt && D.stage != nullptr;
  typename Mem<R>::g* __restrict__ stage = (typename Mem<R>::g*)((R*)D.stage + (phase & 1) * nx);
  // adjoint forward runs: this attempt's output also goes to its history slot
  // where the count it makes if accepted is one of those kept.  A rejected attempt's copy is overwritten by the
  // retry, which has the same count, so the slot ends with the accepted
  // state (FP32 instances, extended instantiation only).
  gfloat* __restrict__ hs1 = nullptr;
  gfloat* __restrict__ hs2 = nullptr;
  gfloat* __restrict__ hs3 = nullptr;
  if constexpr (kExt && sizeof(R) == 4) {
    const int64_t t = P.n_acc + 1 - D.log_base;
    if (D.hist != nullptr && !hist_state && t >= 1 && t <= D.log_len) {
      const uint32_t every = (uint32_t)D.hist_every;
      const uint32_t slot = ((uint32_t)t + every - 1) / every;
      if (slot * every == (uint32_t)t || t == D.log_len) {
        const size_t n = (size_t)nx * (size_t)ny;
        hs1 = (gfloat*)(D.hist + (size_t)slot * 3 * n);
        hs2 = hs1 + n;
        hs3 = hs2 + n;
      }
    }
  }
  const bool hist_on = kExt && sizeof(R) == 4 && hs1 != nullptr;
  const int jcut = D.jcut;
  // what the boundary policy sees of this attempt; the moving window's MDX
  // only exists in the extended instantiation (else it is 0)
  fvbc::PatchCtx<R> pc;
  pc.sin_t = sin_t;
  pc.cos_t = cos_t;
  pc.T = P.T;
  pc.hk = sizeof(R) == 4 ? R(D.hifu_k) : R(D.hifu_k_d);
  pc.mdx = kExt ? P.mdx : 0;
  pc.x0 = it.x0;
  pc.nx = nx;
  pc.ny = ny;
  pc.ic = ic;
  pc.left = lm.left;
  pc.any_left = __builtin_amdgcn_ballot_w64(lm.left) != 0;
  auto patch = [&](Row<R>& q, const fvbc::RowData<R>& h, int r) {
    fvbc::Cell<R> c{q.q1, q.q2, q.q3};
    BC::patch(pc, min(max(r, 0), ny - 1), c, h);
    q.q1 = c.q1;
    q.q2 = c.q2;
    q.q3 = c.q3;
    const R ir = fvna::rcp(R(1) + q.q1);
    q.un = q.q3 * ir;
    q.ut = q.q2 * ir;
  };
  // source on row s (apps/na/source.h:86-104) from q_xy rows s-1, s, s+1,
  // then the store of row s (lanes 3..60)
  auto source_store = [&](int s, const XY<R>& lo, const XY<R>& mid, const XY<R>& hi) {
    const bool s_int = col_int && (s >= 2) && (s <= ny - 3);
    // u(i-1) + u(i+1): one cross-lane move, the other folds into the add
    const R uwe = shr1(mid.u) + shl1(mid.u);
    const R vwe = shr1(mid.v) + shl1(mid.v);
    // apps/na/source.h: x and y increments summed, then added to q once
    const R i2 = fvna::source_increment(ddx2, ddy2, mid.u, uwe, lo.u, hi.u);
    const R i3 = fvna::source_increment(ddx2, ddy2, mid.v, vwe, lo.v, hi.v);
    R r2 = fvna::apply_source(mid.q2, i2);
    R r3 = fvna::apply_source(mid.q3, i3);
    r2 = s_int ? r2 : mid.q2;
    r3 = s_int ? r3 : mid.q3;
    pin(r2);
    pin(r3);
    if (!kExt) {
      if (out_lane) {
        const uint32_t o = (uint32_t)s * row_bytes + kSz * (uint32_t)i;
        stg(o1, o, mid.q1);            // q1 passes the source unchanged
        stg(o2, o, r2);
        stg(o3, o, r3);
      }
    } else {
      // one cell of the output, at byte offset o, and of the history slot
      auto put = [&](uint32_t o) {
        stg(o1, o, mid.q1);
        stg(o2, o, r2);
        stg(o3, o, r3);
        if constexpr (sizeof(R) == 4) {
          if (hist_on) {
            stg(hs1, o, mid.q1);
            stg(hs2, o, r2);
            stg(hs3, o, r3);
          }
        }
      };
      if (out_lane && i >= sx && s >= sy)
        put((uint32_t)(s - sy) * row_bytes + kSz * (uint32_t)(i - sx));
      if (out_lane && (i + sx > nx - 1 || s + sy > ny - 1))
        put((uint32_t)s * row_bytes + kSz * (uint32_t)i);
      // data collection reads row jcut as it is before the shift
      if (stage_on && s == jcut && out_lane) stg(stage, kSz * (uint32_t)i, mid.q1);
    }
  };

  // dt/d on the lanes of interior columns, 0 on ghost columns
  const R dty_c = col_int ? dty : R(0), dtx_c = col_int ? dtx : R(0);
  // the same on the rows of interior cells, 0 on ghost rows: ghost cells keep
  // their value (the fluxes are finite wherever the attempt is valid, so
  // q - 0*flux == q exactly).  In FP32 the row's two are kept from row to row,
  // changed where the interior starts and ends; in FP64 they are selected anew
  // each row (four registers fewer: 70.2 against 70.7 us on 4096x1024).
  // Starts at row y0 - 1, the first one swept
  constexpr bool kCarryRow = sizeof(R) == 4;
  const bool first_int = y0 >= 3 && y0 <= ny - 2;
  R dtyu = first_int ? dty_c : R(0), dtxu = first_int ? dtx_c : R(0);
  R Sx = R(0), Sy = R(0);
  uint64_t err = 0;                          // lanes that met tmp3 < 0 (or NaN)
  const uint64_t in_mask = __builtin_amdgcn_ballot_w64(col_in);
  const uint64_t x_mask = __builtin_amdgcn_ballot_w64(col_x);

  // What this wave leaves for the wave below it, and finds of the wave above
  // (kSeam* fields, one value per lane).
  R* const s_out = &seam[it.role & kRoleIndex][0][lane];
  const R* const s_in = s_out + kSeamFields * kLanes;
  const bool above = (it.role & kRoleAbove) != 0;   // a wave above in the workgroup

  // One march step.  bn/bm/bo: q_b rows r, r-1, r-2; fn/fc/fl: y interfaces
  // r, r-1, r-2.  xn/xo/xm hold q_xy rows r-5, r-4, r-3 on entry; the x sweep
  // overwrites xn with row r-2.  n1..n3 (nh) hold the raw prefetched row r on
  // entry and row r+1 on exit.  Order: consume the prefetch, store row r-4,
  // issue the next prefetch -- so each store has a whole step to drain before
  // the next step waits for its prefetch (stores and loads share one in-order
  // counter).  kT: the step's place in the march.
  //   0..5    the first rows, r = y0 - 3 + kT: each stage starts where the
  //           item's first outputs need it, and what the wave below needs is
  //           left in LDS
  //   6       every later row
  //   7..9    the last three rows below a seam (r = y1-2, y1-1, y1): the
  //           interfaces y1-2 and up are the upper wave's
  auto body = [&](auto kTc, int r, Row<R>& bn, Row<R>& bm, Row<R>& bo, YI<R>& fn, YI<R>& fc,
                  YI<R>& fl, XY<R>& xn, XY<R>& xm, XY<R>& xo) {
    constexpr int kT = decltype(kTc)::value;
    if constexpr (kT <= 7) {
      // every load of the prefetch (and every store before it) is done: an
      // explicit vmcnt(0) here keeps the compiler's own wait for the prefetched
      // registers from landing after this step's stores, and lgkmcnt(0) its
      // wait for the row's scalars (which return in any order, so that it could
      // only wait for all) from landing after the next row's are requested
      __builtin_amdgcn_s_waitcnt(kWaitLoads);
      bn.q1 = n1; bn.q2 = n2; bn.q3 = n3; bn.cm = nk;
      patch(bn, nh, r);
    }
    if constexpr (kT >= 6) {
      if (r >= y0 + 4) source_store(r - 4, xn, xo, xm);
    }
    // row m = r-2 is the first interior row, or the first ghost row above
    if constexpr (kT >= 4 && kCarryRow) {
      if (r == 4 || r == ny) {
        dtyu = r == 4 ? dty_c : R(0);
        dtxu = r == 4 ? dtx_c : R(0);
      }
    }
    // the next row, also past the item's last row: the row index is clamped
    // to the grid, and an unconditional load needs no copy of the registers
    // it replaces
    if constexpr (kT <= 6) load_raw(r + 1, n1, n2, n3, nk, nh);
    if constexpr (kT == 0) return;
    const int m = r - 2;

    // ---- y interface r (rows r-1 | r): normal = q3, tangential = q2 ----
    if constexpr (kT <= 6) {
      // CFL lane mask of row r (its y interfaces).  Rows next to a workgroup's
      // own are counted there too: the same values, so the same maximum
      const uint64_t mY = (r >= 1 && r < ny) ? bn.cm : 0;
      fvna::riemann(fvna::jump(bm.q1, bm.q3, bm.q2, bm.un, bm.ut, bn.q1, bn.q3, bn.q2, bn.un,
                               bn.ut),
                    hbeta, fn.f);
      // branch-free (a branch here would split the block and stop the
      // cross-lane moves of the x sweep from folding into their users)
      err |= __builtin_amdgcn_ballot_w64(fn.f.bad) & ((r >= 1 && r < ny) ? in_mask : 0);
      masked_max(mY, Sy, fn.f.L1, fn.f.L2);
      if constexpr (kT == 1) {
        seam_put(s_out, kSeamW + 0, fn.f.w.a1);  seam_put(s_out, kSeamW + 1, fn.f.w.w21);
        seam_put(s_out, kSeamW + 2, fn.f.w.w31); seam_put(s_out, kSeamW + 3, fn.f.w.a2);
        seam_put(s_out, kSeamW + 4, fn.f.w.w22); seam_put(s_out, kSeamW + 5, fn.f.w.w32);
        seam_put(s_out, kSeamW + 6, fn.f.w.a3);
        seam_put(s_out, kSeamL + 0, fn.f.L1);
        seam_put(s_out, kSeamL + 1, fn.f.L2);
        seam_put(s_out, kSeamL + 2, fn.f.L3);
        return;
      }
    } else if constexpr (kT == 7) {
      fn.f.w.a1 = seam_get(s_in, kSeamW + 0);  fn.f.w.w21 = seam_get(s_in, kSeamW + 1);
      fn.f.w.w31 = seam_get(s_in, kSeamW + 2); fn.f.w.a2 = seam_get(s_in, kSeamW + 3);
      fn.f.w.w22 = seam_get(s_in, kSeamW + 4); fn.f.w.w32 = seam_get(s_in, kSeamW + 5);
      fn.f.w.a3 = seam_get(s_in, kSeamW + 6);
      fn.f.L1 = seam_get(s_in, kSeamL + 0);
      fn.f.L2 = seam_get(s_in, kSeamL + 1);
      fn.f.L3 = seam_get(s_in, kSeamL + 2);
    }

    // W(r).W(r-1): the left product of interface r, the right one of r-1
    if constexpr (kT <= 7) {
      fn.dl[0] = fvna::dot1(fn.f.w, fc.f.w);
      fn.dl[1] = fvna::dot2(fn.f.w, fc.f.w);
      fn.dl[2] = fn.f.w.a3 * fc.f.w.a3;
    } else if constexpr (kT == 8) {
#pragma unroll
      for (int p = 0; p < 3; ++p) fn.dl[p] = seam_get(s_in, kSeamDl + p);
    }
    if constexpr (kT == 2) {
#pragma unroll
      for (int p = 0; p < 3; ++p) seam_put(s_out, kSeamDl + p, fn.dl[p]);
      return;
    }

    // ---- y limiter at interface r-1 ----
    R M[3];
    if constexpr (kT <= 8) {
      R nw1, nw2;
      fvna::norms(fc.f.w, nw1, nw2);
      fvna::limited_flux<false>(fc.f, nw1, nw2, fvna::upwind(fc.f.L1, fc.dl[0], fn.dl[0]),
                                fvna::upwind(fc.f.L2, fc.dl[1], fn.dl[1]),
                                fvna::upwind(fc.f.L3, fc.dl[2], fn.dl[2]), dty, fc.P, M);
    } else {
#pragma unroll
      for (int p = 0; p < 3; ++p) M[p] = seam_get(s_in, kSeamM + p);
    }
    if constexpr (kT == 3) {
#pragma unroll
      for (int p = 0; p < 3; ++p) seam_put(s_out, kSeamM + p, M[p]);
      return;
    }

    // ---- q_y on row m = r-2 (components: density, normal=q3, tangential=q2)
    const uint64_t mX = (m >= 0 && m < ny) ? bo.cm : 0;
    if constexpr (!kCarryRow) {
      const bool row_int = (m >= 2) && (m <= ny - 3);
      dtyu = row_int ? dty_c : R(0);
      dtxu = row_int ? dtx_c : R(0);
    }
    const R y1q = fvna::sub_prod(bo.q1, dtyu, fl.P[0] + M[0]);
    const R y3q = fvna::sub_prod(bo.q3, dtyu, fl.P[1] + M[1]);
    const R y2q = fvna::sub_prod(bo.q2, dtyu, fl.P[2] + M[2]);

    // ---- x sweep on row m: normal = q2, tangential = q3 ----
    const R ir = fvna::rcp(R(1) + y1q);
    const R un = y2q * ir, ut = y3q * ir;
    const R l1 = shr1(y1q), l2 = shr1(y2q), l3 = shr1(y3q);
    const R lun = shr1(un), lut = shr1(ut);
    fvna::IfaceT<R> fx;
    // pinned together: the compiler folds a cross-lane move only into users
    // within a few instructions of it
    fvna::JumpT<R> jx = fvna::jump(l1, l2, l3, lun, lut, y1q, y2q, y3q, un, ut);
    pin(jx.s1); pin(jx.s2); pin(jx.s3); pin(jx.drho); pin(jx.dn); pin(jx.dtg);
    fvna::riemann(jx, hbeta, fx);
    err |= __builtin_amdgcn_ballot_w64(fx.bad) & ((m >= 0 && m < ny) ? x_mask : 0);
    masked_max(mX, Sx, fx.L1, fx.L2);
    // W(k).W(k-1), with the waves of the interface to the left
    R dl1, dl2, dl3;
    dots_left<false>(fx.w, dl1, dl2, dl3);
    // W(k).W(k+1) is the right neighbour's W(k+1).W(k)
    R up1, up2, up3, nw1, nw2;
    upwind_x(fx, dl1, dl2, dl3, up1, up2, up3, nw1, nw2);
    R PX[3], MX[3];
    fvna::limited_flux<true>(fx, nw1, nw2, up1, up2, up3, dtx, PX, MX);
    const R mr0 = shl1(MX[0]), mr1 = shl1(MX[1]), mr2 = shl1(MX[2]);
    xn.q1 = fvna::sub_prod(y1q, dtxu, mr0 + PX[0]);
    xn.q2 = fvna::sub_prod(y2q, dtxu, mr1 + PX[1]);
    xn.q3 = fvna::sub_prod(y3q, dtxu, mr2 + PX[2]);
    const R ir2 = fvna::rcp(R(1) + xn.q1);
    xn.u = xn.q2 * ir2;
    xn.v = xn.q3 * ir2;
    if constexpr (kT == 4) {
      seam_put(s_out, kSeamX + 0, xn.q1);
      seam_put(s_out, kSeamX + 1, xn.q2);
      seam_put(s_out, kSeamX + 2, xn.q3);
      seam_put(s_out, kSeamX + 3, xn.u);
      seam_put(s_out, kSeamX + 4, xn.v);
    }
    if constexpr (kT == 5) {
      seam_put(s_out, kSeamX + 5, xn.u);
      seam_put(s_out, kSeamX + 6, xn.v);
    }
  };

  // every window is written before it is read
  Row<R> B0, B1, B2;
  YI<R> F0, F1, F2;
  XY<R> X0, X1, X2;
  body(At<0>{}, y0 - 3, B0, B2, B1, F0, F2, F1, X0, X2, X1);
  body(At<1>{}, y0 - 2, B1, B0, B2, F1, F0, F2, X1, X0, X2);
  body(At<2>{}, y0 - 1, B2, B1, B0, F2, F1, F0, X2, X1, X0);
  body(At<3>{}, y0, B0, B2, B1, F0, F2, F1, X0, X2, X1);
  body(At<4>{}, y0 + 1, B1, B0, B2, F1, F0, F2, X1, X0, X2);
  body(At<5>{}, y0 + 2, B2, B1, B0, F2, F1, F0, X2, X1, X0);
  seam_publish();
  const int r_end = above ? y1 - 3 : y1 + 2;
  for (int r = y0 + 3; r <= r_end; r += 3) {
    body(At<6>{}, r, B0, B2, B1, F0, F2, F1, X0, X2, X1);
    if (r + 1 > r_end) break;
    body(At<6>{}, r + 1, B1, B0, B2, F1, F0, F2, X1, X0, X2);
    if (r + 2 > r_end) break;
    body(At<6>{}, r + 2, B2, B1, B0, F2, F1, F0, X2, X1, X0);
  }
  if (above) {
    // the host gives the items below a seam heights of 2 mod 3 (>= 5), so the
    // loop ends with the windows in their first rotation
    body(At<7>{}, y1 - 2, B0, B2, B1, F0, F2, F1, X0, X2, X1);
    body(At<8>{}, y1 - 1, B1, B0, B2, F1, F0, F2, X1, X0, X2);
    body(At<9>{}, y1, B2, B1, B0, F2, F1, F0, X2, X1, X0);
    XY<R> a0, a1;             // the upper wave's first two rows of q_xy, y1-1 and y1
    a0.q1 = seam_get(s_in, kSeamX + 0);
    a0.q2 = seam_get(s_in, kSeamX + 1);
    a0.q3 = seam_get(s_in, kSeamX + 2);
    a0.u = seam_get(s_in, kSeamX + 3);
    a0.v = seam_get(s_in, kSeamX + 4);
    a1 = a0;
    a1.u = seam_get(s_in, kSeamX + 5);
    a1.v = seam_get(s_in, kSeamX + 6);
    source_store(y1 - 3, X0, X1, X2);
    source_store(y1 - 2, X1, X2, a0);
    source_store(y1 - 1, X2, a0, a1);
  } else {
    // the last row, y1 - 1, with the window of the step r = y1 + 3 would see
    switch ((y1 - y0) % 3) {
      case 0: source_store(y1 - 1, X0, X1, X2); break;
      case 1: source_store(y1 - 1, X1, X2, X0); break;
      default: source_store(y1 - 1, X2, X0, X1); break;
    }
  }

  // ---- CFL / error reduction ----
  // per-cell cfl = |s| * dt/d (fv.h:148-180); max over the wave's cells,
  // folded into the group's slot of this attempt (read by the next launch)
  const R cflw = wave_max(fmax_(Sy * dty, Sx * dtx));
  if (lane != 0) return;
  SyncSlots* sl = D.sync + phase % 3;
  if (err != 0) aadd_relaxed(&sl->err_flag, 1u);
  CflSlot<R>::fold_in(sl->grp[local % kGroups], cflw);
}

// Marker for a step kernel that carries the march of every registered app
// (apps/apps.h) and runs, per work item, that of its instance's boundary kind
// (the item carries it, so the choice is made from the item alone): launches
// over several instances.  A single-instance launch takes its app's policy
// directly, a kernel with one march.
struct AnyApp {};

// The step kernel: one wave per work item, kGroupWaves items per workgroup
// (items[4 g .. 4 g + 3]; an unused slot has no rows); then `beside` workgroups
// per instance for beside_step.
template <typename R, bool kOne, bool kExt, class BC>
__global__ __launch_bounds__(kLanes * kGroupWaves) void fv_step_kernel(
    const InstDesc* __restrict__ insts, const WorkItem* __restrict__ items,
    const uint64_t* __restrict__ rowmask, int n_groups, int phase,
    const Ctl* __restrict__ ctl_in, const SyncSlots* __restrict__ sync_in, int beside,
    int collect) {
  // (the plain kernels of the other apps have nothing beside the step)
  constexpr bool kBeside = kExt || std::is_same<BC, AnyApp>::value ||
                           std::is_same<BC, fvbc::Taylor>::value;
  if (kBeside && (int)blockIdx.x >= n_groups) {
    const int e = blockIdx.x - n_groups, inst = uni(e / beside);
    beside_step<R>(insts[inst], phase, e - inst * beside, beside, collect);
    return;
  }
  __shared__ R seam[kGroupWaves][kSeamFields][kLanes];
  // XCD-aware order: workgroup b runs on XCD b % 8; give each XCD a contiguous
  // run of groups so vertically adjacent groups of a strip (which share
  // halo rows) hit the same L2.
  int group;
  {
    const int b = blockIdx.x;
    const int q = n_groups >> 3, rem = n_groups & 7, x = b & 7, k = b >> 3;
    group = x * q + min(x, rem) + k;
  }
  const WorkItem it = items[group * kGroupWaves + uni(threadIdx.x / kLanes)];
  if (it.y1 <= it.y0) return;      // the barrier counts the remaining waves only
  if constexpr (!std::is_same<BC, AnyApp>::value) {
    step_impl<R, kOne, kExt, BC>(insts, it, rowmask, phase, ctl_in, sync_in, seam);
    return;
  }
  switch (uni(it.bc)) {
#define FV_APP_CASE(P)                                                              \
  case P::kId:                                                                      \
    if constexpr (kExt || !P::kExtOnly)                                             \
      step_impl<R, kOne, kExt, P>(insts, it, rowmask, phase, ctl_in, sync_in, seam); \
    break;
    FIVONAGI_APPS(FV_APP_CASE)
#undef FV_APP_CASE
    default:
      break;
  }
}

// Control block after the last launched attempt (phase = index of the next
// attempt mod 6), stored where that attempt's launch will store it too, and
// into mirror (host memory, when given), which the host reads after a
// synchronisation.  One block per instance.
__global__ __launch_bounds__(64) void fv_settle_kernel(const InstDesc* __restrict__ insts,
                                                       int phase, Ctl* __restrict__ mirror) {
  const InstDesc& D = insts[blockIdx.x];
  const Ctl P = current(D, phase, true);
  if (threadIdx.x == 0) {
    D.ctl[(phase + 1) & 1] = P;
    if (mirror) mirror[blockIdx.x] = P;
  }
}

// Stop conditions of the attempts from phase on: the control block that
// attempt would form, with the new conditions, becomes the block it starts
// from, and the attempt before it is marked as folded in.  One block per
// instance; targets: host memory, or null for `target` itself.
__global__ __launch_bounds__(64) void fv_targets_kernel(const InstDesc* __restrict__ insts,
                                                        int phase,
                                                        const int64_t* __restrict__ targets,
                                                        int64_t target, double T_stop) {
  const InstDesc& D = insts[blockIdx.x];
  Ctl P = current(D, phase, true);
  if (threadIdx.x == 0) {
    P.target_acc = targets ? targets[blockIdx.x] : target;
    P.T_stop = T_stop;
    D.ctl[phase & 1] = P;
    D.sync[(phase + 2) % 3].ran = 0u;
  }
}

// Data collection of the attempt of phase `phase` alone, run after its launch
// (the last attempt of a run of launches; the others' comes with the launch
// after them, beside_step).  blockIdx.y = instance; threads cover the columns.
__global__ __launch_bounds__(256) void fv_collect_kernel(const InstDesc* __restrict__ insts,
                                                         int phase) {
  const InstDesc& D = insts[blockIdx.y];
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  if (D.fp64)
    collect_attempt<double>(D, fold_prev<double>(D, phase + 1), phase, tid);
  else
    collect_attempt<float>(D, fold_prev<float>(D, phase + 1), phase, tid);
}

// Ghost ring of the Taylor-shock instances for the attempt of phase `phase`
// (the first attempt of a run of launches, or every one where a buffer has no
// ring: then into the grid).  settle: instead, after that phase's last attempt:
// where the last attempt an instance ran was not accepted, the grid's ghost
// cells take the values it read, as if they had been written there.  blockIdx.y = instance; the ring is
// enumerated by a flat index.
__global__ __launch_bounds__(256) void fv_taylor_ghost_kernel(const InstDesc* __restrict__ insts,
                                                             int phase, int settle) {
  const InstDesc& D = insts[blockIdx.y];
  if (D.bc != kBcTaylor) return;
  const int k0 = blockIdx.x * blockDim.x + threadIdx.x, dk = gridDim.x * blockDim.x;
  if (settle) {
    if (D.ring == 0) return;
    int state;
    Ctl P;
    if (D.fp64) {
      const Fold<double> F = fold_prev<double>(D, phase);
      state = F.state;
      P = F.p;
    } else {
      const Fold<float> F = fold_prev<float>(D, phase);
      state = F.state;
      P = F.p;
    }
    // (an instance that an error stopped earlier in the run: still the ghost
    // cells of the attempt that failed, whose control block it keeps)
    if (state == kFoldReject || state == kFoldError || (state == kFoldIdle && P.err == 2))
      taylor_ring(D, P.T, P.cur, P.mdx, P.mdy, false, k0, dk);
    return;
  }
  const Ctl P = current(D, phase, false);
  if (P.err != 0 || P.n_acc >= P.target_acc || !(P.T < P.T_stop)) return;
  taylor_ring(D, P.T, P.cur, P.mdx, P.mdy, D.ring != 0, k0, dk);
}

}  // namespace fv

extern "C" hipError_t fv_launch_taylor_ghosts(const fv::InstDesc* insts, int n_inst,
                                              int max_ring, int phase, int settle,
                                              hipStream_t stream) {
  if (n_inst <= 0) return hipSuccess;
  const int blocks = (max_ring + 255) / 256;
  hipLaunchKernelGGL(fv::fv_taylor_ghost_kernel, dim3(blocks, n_inst), dim3(256), 0, stream,
                     insts, phase, settle);
  return hipGetLastError();
}

extern "C" hipError_t fv_launch_collect(const fv::InstDesc* insts, int n_inst, int max_nx,
                                        int phase, hipStream_t stream) {
  if (n_inst <= 0) return hipSuccess;
  hipLaunchKernelGGL(fv::fv_collect_kernel, dim3((max_nx + 255) / 256, n_inst), dim3(256), 0,
                     stream, insts, phase);
  return hipGetLastError();
}

extern "C" hipError_t fv_launch_settle(const fv::InstDesc* insts, int n_inst, int phase,
                                       fv::Ctl* mirror, hipStream_t stream) {
  if (n_inst <= 0) return hipSuccess;
  hipLaunchKernelGGL(fv::fv_settle_kernel, dim3(n_inst), dim3(64), 0, stream, insts, phase,
                     mirror);
  return hipGetLastError();
}

extern "C" hipError_t fv_launch_targets(const fv::InstDesc* insts, int n_inst, int phase,
                                        const int64_t* targets, int64_t target, double T_stop,
                                        hipStream_t stream) {
  if (n_inst <= 0) return hipSuccess;
  hipLaunchKernelGGL(fv::fv_targets_kernel, dim3(n_inst), dim3(64), 0, stream, insts, phase,
                     targets, target, T_stop);
  return hipGetLastError();
}

// Resident step waves per CU (occupancy of the step kernel on this device),
// of the FP64 kernel if fp64.  The lowest over the plain and extended
// kernels of several instances (every app's march: the most registers), so
// the split fits whichever kernel a context launches.
extern "C" hipError_t fv_step_waves_per_cu(int* waves, int fp64) {
  constexpr int kThreads = fv::kLanes * fv::kGroupWaves;
  int a = 0, b = 0;
  hipError_t e = fp64 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(
                            &a, fv::fv_step_kernel<double, false, false, fv::AnyApp>, kThreads, 0)
                      : hipOccupancyMaxActiveBlocksPerMultiprocessor(
                            &a, fv::fv_step_kernel<float, false, false, fv::AnyApp>, kThreads, 0);
  if (e != hipSuccess) return e;
  e = fp64 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(
                 &b, fv::fv_step_kernel<double, false, true, fv::AnyApp>, kThreads, 0)
           : hipOccupancyMaxActiveBlocksPerMultiprocessor(
                 &b, fv::fv_step_kernel<float, false, true, fv::AnyApp>, kThreads, 0);
  *waves = fv::kGroupWaves * (a < b ? a : b);
  return e;
}

namespace {
// the workgroups for beside_step: parts per instance
struct Beside {
  int n_inst, parts, collect;
};
template <typename R, bool kOne, bool kExt, class BC>
void launch_step_t(const fv::InstDesc* insts, const fv::WorkItem* items, const uint64_t* rowmask,
                   int n_groups, int phase, const fv::Ctl* c_in, const fv::SyncSlots* s_in,
                   const Beside& bs, hipStream_t stream) {
  hipLaunchKernelGGL((fv::fv_step_kernel<R, kOne, kExt, BC>),
                     dim3(n_groups + bs.n_inst * bs.parts), dim3(fv::kLanes * fv::kGroupWaves), 0,
                     stream, insts, items, rowmask, n_groups, phase, c_in, s_in, bs.parts,
                     bs.collect);
}
// a single instance: its app's own kernel (bc), else the dispatching one
template <typename R, bool kExt>
void launch_one(int bc, const fv::InstDesc* insts, const fv::WorkItem* items,
                const uint64_t* rowmask, int n_groups, int phase, const fv::Ctl* c_in,
                const fv::SyncSlots* s_in, const Beside& bs, hipStream_t stream) {
  switch (bc) {
#define FV_APP_LAUNCH(P)                                                                 \
  case P::kId:                                                                           \
    if constexpr (kExt || !P::kExtOnly) {                                                \
      launch_step_t<R, true, kExt, P>(insts, items, rowmask, n_groups, phase, c_in, s_in, \
                                      bs, stream);                                           \
      return;                                                                            \
    }                                                                                    \
    break;
    FIVONAGI_APPS(FV_APP_LAUNCH)
#undef FV_APP_LAUNCH
    default:
      break;
  }
  launch_step_t<R, true, kExt, fv::AnyApp>(insts, items, rowmask, n_groups, phase, c_in, s_in,
                                           bs, stream);
}
template <typename R>
void launch_step_r(bool one, bool ext, int bc, const fv::InstDesc* insts,
                   const fv::WorkItem* items, const uint64_t* rowmask, int n_groups, int phase,
                   const fv::Ctl* c_in, const fv::SyncSlots* s_in, const Beside& bs,
                   hipStream_t stream) {
  if (one && !ext)
    launch_one<R, false>(bc, insts, items, rowmask, n_groups, phase, c_in, s_in, bs, stream);
  else if (one)
    launch_one<R, true>(bc, insts, items, rowmask, n_groups, phase, c_in, s_in, bs, stream);
  else if (!ext)
    launch_step_t<R, false, false, fv::AnyApp>(insts, items, rowmask, n_groups, phase, c_in, s_in,
                                               bs, stream);
  else
    launch_step_t<R, false, true, fv::AnyApp>(insts, items, rowmask, n_groups, phase, c_in, s_in,
                                              bs, stream);
}
}  // namespace

// One step attempt of every instance: n_groups workgroups, items[4 g ..] each.
// ctl0/sync0: the control blocks (two per instance) and slot sets (three) of the
// instances, one instance after the other, where their descriptions point too;
// bc0: the boundary kind of an only instance; ext: some instance has a moving
// window, the HIFU boundary or data collection; fp64: the instances are FP64;
// beside, collect: workgroups per instance for beside_step, and how many of them
// collect the attempt before.
extern "C" hipError_t fv_launch_step(const fv::InstDesc* insts, const fv::WorkItem* items,
                                     const uint64_t* rowmask, int n_groups, int phase,
                                     int n_inst, fv::Ctl* ctl0, fv::SyncSlots* sync0, int bc0,
                                     int ext, int fp64, int beside, int collect,
                                     hipStream_t stream) {
  if (n_groups <= 0) return hipSuccess;
  const bool one = n_inst == 1;
  const fv::Ctl* c_in = ctl0 + (phase & 1);
  const fv::SyncSlots* s_in = sync0 + (phase + 2) % 3;
  const Beside bs{n_inst, beside, collect};
  if (fp64)
    launch_step_r<double>(one, ext != 0, bc0, insts, items, rowmask, n_groups, phase, c_in, s_in,
                          bs, stream);
  else
    launch_step_r<float>(one, ext != 0, bc0, insts, items, rowmask, n_groups, phase, c_in, s_in,
                         bs, stream);
  return hipGetLastError();
}
