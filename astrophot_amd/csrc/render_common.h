// Per-pixel device code shared by the single-component render (render.hip)
// and the batched render (batch.hip): pixel offsets and quad:N sampling
// (utils/operations.py:105-147).
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/astrophot_hip.h"
#include "profile.h"
#include "wave.h"

namespace apx {

// offsets of a working pixel from the centre
template <typename T>
__device__ __forceinline__ void pixel_xy(const Prof<T>& p, int ci, int cj, int i, int j, T& X,
                                         T& Y) {
  const T di = (T)(i - ci);
  const T dj = (T)(j - cj);
  X = p.P00 * di + p.P01 * dj + p.fx;
  Y = p.P10 * di + p.P11 * dj + p.fy;
}
template <typename T>
__device__ __forceinline__ void pixel_xy(const Prof<T>& p, const apx_component& cp, int i, int j,
                                         T& X, T& Y) {
  pixel_xy(p, cp.ci, cp.cj, i, j, X, Y);
}

// quad:N sample of one pixel (operations.py:123-147): returns the weighted
// sum, `centre` the middle node; accumulates weighted slot gradients in g.
template <typename T, bool GRAD>
__device__ T quad_sample(const Prof<T>& p, const apx_component& cp, T X, T Y, int n,
                         const double* node, const double* weight, T scale, T hP00, T hP01,
                         T hP10, T hP11, T* g, T& centre) {
  T res = (T)0;
  T gl[APX_NSLOT];
  if (GRAD) {
#pragma unroll
    for (int k = 0; k < APX_NSLOT; ++k) g[k] = (T)0;
  }
  for (int k = 0; k < n * n; ++k) {
    const T u = (T)node[k % n], v = (T)node[k / n];
    const T w = (T)(weight[k % n] * weight[k / n] * 0.25);
    const T val = eval_profile<T, GRAD>(p, X + hP00 * u + hP01 * v, Y + hP10 * u + hP11 * v,
                                        scale, gl);
    res += w * val;
    if (k == (n * n) / 2) centre = val;
    if (GRAD) {
#pragma unroll
      for (int s = 0; s < APX_NSLOT; ++s) g[s] += w * gl[s];
    }
  }
  return res;
}


// Relative band around a threshold inside which a float32 test is taken again
// in float64 (float32 profile samples carry far less relative error).
constexpr double kSampleBand = 1e-4;

}  // namespace apx
