// fv_lanes.h -- cross-lane operations of a wave64 that holds one row of a strip,
// a column per lane (device code; the step and the reverse march).
#ifndef FIVONAGI_FV_LANES_H
#define FIVONAGI_FV_LANES_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../apps/na/solver.h"

namespace fv {

// DPP cross-lane moves over the whole wave64 (gfx9 wave_shr:1 / wave_shl:1).
// shr1: lane l receives lane l-1's value (lane 0 receives 0).
// shl1: lane l receives lane l+1's value (lane 63 receives 0).
// bound_ctrl = 1: the missing source lane reads as 0, so no "old" value has
// to be materialised first.
__device__ __forceinline__ float shr1(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float shl1(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x130, 0xf, 0xf, true));
}
// 64-bit values move as two 32-bit halves
__device__ __forceinline__ double dpp64(double v, int ctrl_shr) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)(ctrl_shr ? __builtin_amdgcn_mov_dpp((int)(uint32_t)u, 0x138, 0xf, 0xf, true)
                                          : __builtin_amdgcn_mov_dpp((int)(uint32_t)u, 0x130, 0xf, 0xf, true));
  const uint32_t hi = (uint32_t)(ctrl_shr ? __builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), 0x138, 0xf, 0xf, true)
                                          : __builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), 0x130, 0xf, 0xf, true));
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
__device__ __forceinline__ double shr1(double v) { return dpp64(v, 1); }
__device__ __forceinline__ double shl1(double v) { return dpp64(v, 0); }

// Products with the left neighbour's waves: the same sums as fvna::dot1/dot2
// (a, shr1(a)), each multiply-add taking its neighbour operand by DPP.  The
// compiler folds a cross-lane move only into two-operand forms it has before
// register allocation, never into a multiply-add, so these are written out;
// s_nop covers the two wait states between a VALU write and a DPP read: before
// and, where the products are moved between lanes by what the compiler makes of
// the code behind (kMoved), behind.  (The step's only lane moves of them stand in
// upwind_x, behind three instructions of its own.)
#define FV_DOTS_LEFT(tail)                                                                        \
  asm("s_nop 1\n\t"                                                                               \
      "v_mul_f32_dpp %0, %5, %5 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"           \
      "v_mul_f32_dpp %1, %8, %8 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"           \
      "v_mul_f32_dpp %2, %9, %9 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"           \
      "v_fmac_f32_dpp %0, %4, %4 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"          \
      "v_fmac_f32_dpp %1, %7, %7 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"          \
      "v_fmac_f32_dpp %0, %3, %3 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"          \
      "v_fmac_f32_dpp %1, %6, %6 wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1" tail         \
      : "=&v"(d1), "=&v"(d2), "=&v"(d3)                                                           \
      : "v"(w.a1), "v"(w.w21), "v"(w.w31), "v"(w.a2), "v"(w.w22), "v"(w.w32), "v"(w.a3))
template <bool kMoved>
__device__ __forceinline__ void dots_left(const fvna::WavesT<float>& w, float& d1, float& d2,
                                          float& d3) {
  if constexpr (kMoved)
    FV_DOTS_LEFT("\n\ts_nop 1");
  else
    FV_DOTS_LEFT("");
}
#undef FV_DOTS_LEFT
template <bool kMoved>
__device__ __forceinline__ void dots_left(const fvna::WavesT<double>& w, double& d1, double& d2,
                                          double& d3) {
  fvna::WavesT<double> l;
  l.a1 = shr1(w.a1); l.w21 = shr1(w.w21); l.w31 = shr1(w.w31);
  l.a2 = shr1(w.a2); l.w22 = shr1(w.w22); l.w32 = shr1(w.w32);
  l.a3 = shr1(w.a3);
  d1 = fvna::dot1(w, l);
  d2 = fvna::dot2(w, l);
  d3 = w.a3 * l.a3;
}

}  // namespace fv

#endif  // FIVONAGI_FV_LANES_H
