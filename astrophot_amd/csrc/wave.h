// Sums over a wavefront without LDS.  The additions are those of the xor
// butterfly (partner at distance 32, 16, 8, 4, 2, 1), so the sum is the same
// in every lane and does not depend on how the partner's value arrives: by
// v_permlane32_swap / v_permlane16_swap for 32 and 16, and by DPP moves below
// (a rotation by 8 or 4 within a row of 16 lanes, quad permutations for 2 and
// 1; after the step at 8 the lanes of a row at distance 8 hold the same value,
// so the rotation by 4 brings the partner's).  ds_bpermute, which __shfl_xor
// compiles to, waits out an LDS round trip a step.
#pragma once

#include <hip/hip_runtime.h>

namespace apx {

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_move(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, false);
}

// v of the lane at distance O of this lane's butterfly step (32 and 16: the two
// halves' values come back as a pair whose sum is wanted)
__device__ __forceinline__ float butterfly_add32(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float butterfly_add16(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
template <int CTRL>
__device__ __forceinline__ float butterfly_add(float v) {
  return v + __uint_as_float(dpp_move<CTRL>(__float_as_uint(v)));
}
__device__ __forceinline__ double butterfly_add32(double v) {
  const uint32_t lo = (uint32_t)__double2loint(v), hi = (uint32_t)__double2hiint(v);
  const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
  return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
}
__device__ __forceinline__ double butterfly_add16(double v) {
  const uint32_t lo = (uint32_t)__double2loint(v), hi = (uint32_t)__double2hiint(v);
  const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
}
template <int CTRL>
__device__ __forceinline__ double butterfly_add(double v) {
  const uint32_t lo = (uint32_t)__double2loint(v), hi = (uint32_t)__double2hiint(v);
  return v + __hiloint2double((int)dpp_move<CTRL>(hi), (int)dpp_move<CTRL>(lo));
}

// sum over the row of 16 lanes, over 32 lanes, over the wave
template <typename T>
__device__ __forceinline__ T row_sum(T v) {
  v = butterfly_add<0x128>(v);     // row_ror:8
  v = butterfly_add<0x124>(v);     // row_ror:4
  v = butterfly_add<0x4e>(v);      // quad_perm 2,3,0,1
  return butterfly_add<0xb1>(v);   // quad_perm 1,0,3,2
}
template <typename T>
__device__ __forceinline__ T half_sum(T v) {
  return row_sum(butterfly_add16(v));
}
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  return half_sum(butterfly_add32(v));
}

// The wave sums of N values at once, to out[0 .. N) (LDS or global): the two
// widest steps halve the number of values in flight, as a swap of two registers'
// halves leaves one value's partial sums in one half and the other's in the
// other, so N values take about 3 N / 2 + 3 N instructions, not 18 N.
template <int N>
__device__ __forceinline__ void wave_sums(const double (&v)[N], double* out) {
  constexpr int H = (N + 1) / 2, Q = (H + 1) / 2;
  const int lane = threadIdx.x & 63, row = lane >> 4;
  double u[2 * Q];
#pragma unroll
  for (int j = 0; j < 2 * Q; ++j) {  // lanes 0-31: v[2 j], lanes 32-63: v[2 j + 1]
    const double a = 2 * j < N ? v[2 * j] : 0.0, b = 2 * j + 1 < N ? v[2 * j + 1] : 0.0;
    const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)__double2loint(a), (uint32_t)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)__double2hiint(a), (uint32_t)__double2hiint(b), false, false);
    u[j] = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
  }
#pragma unroll
  for (int m = 0; m < Q; ++m) {  // rows 0..3: v[4 m], v[4 m + 2], v[4 m + 1], v[4 m + 3]
    const double a = u[2 * m], b = u[2 * m + 1];
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)__double2loint(a), (uint32_t)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)__double2hiint(a), (uint32_t)__double2hiint(b), false, false);
    const double t = row_sum(__hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]));
    const int k = 4 * m + ((row & 1) << 1) + (row >> 1);
    if ((lane & 15) == 0 && k < N) out[k] = t;
  }
}

}  // namespace apx
