// Component render on gfx950: initial sampling, curvature-threshold selection
// and adaptive Gauss-Legendre supersampling of the selected pixels.
//
// Restates models/_model_methods.py:82-184 (_sample_init midpoint / quad:N,
// _sample_integrate threshold) and utils/operations.py:94-247
// (single_quad_integrate, grid_integrate) as three launches:
//   1. init     : one thread per working pixel, float32 profile value and
//                 Jacobian channels; a float64 per-block partial sum when the
//                 integrate reference is the mean sample.
//   2. select   : curvature (replicate-padded 5-point Laplacian) or |quad -
//                 centre node|, compared with tolerance * reference.  Pixels
//                 whose float32 test lies within a rounding band of the
//                 threshold are re-decided in float64, so the selected set is
//                 the float64 one.  Selected pixels are appended to a list with
//                 one atomic per wavefront.
//   3. integrate: one wavefront per listed pixel; the recursive quadrature
//                 (levels 1..max_depth, threshold x gridding^2 per level as in
//                 operations.py:241) runs in float64 and overwrites the
//                 pixel's value and Jacobian channels.
#include <hip/hip_runtime.h>

#include "capi_internal.h"
#include "profile.h"
#include "render_common.h"

namespace apx {

namespace {

constexpr int kInitBlock = 256;
constexpr int kIntegrateWaves = 2048;

// workspace layout (bytes)
struct RenderWs {
  int32_t* count;     // [0]: selected pixels
  double* reference;  // mean-sample reference (when mean_reference)
  double* partial;    // per-init-block sums
  int32_t* list;      // selected pixel indices
  float* centre;      // quad:N centre-node samples
  uint8_t* flags;     // 1 = pixel selected for integration
  double* vpart;      // per-integrate-block adjoint sums (8 per block)
};

__host__ __device__ inline int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }

__host__ __device__ inline int64_t init_blocks(int64_t npix) {
  return (npix + kInitBlock - 1) / kInitBlock;
}

__host__ inline RenderWs carve(void* ws, int64_t npix) {
  char* b = static_cast<char*>(ws);
  RenderWs w;
  w.count = reinterpret_cast<int32_t*>(b);
  w.reference = reinterpret_cast<double*>(b + 64);
  int64_t off = 256;
  w.partial = reinterpret_cast<double*>(b + off);
  off += align256(8 * 8 * init_blocks(npix));
  w.list = reinterpret_cast<int32_t*>(b + off);
  off += align256(4 * npix);
  w.centre = reinterpret_cast<float*>(b + off);
  off += align256(4 * npix);
  w.flags = reinterpret_cast<uint8_t*>(b + off);
  off += align256(npix);
  w.vpart = reinterpret_cast<double*>(b + off);
  return w;
}

template <bool GRAD>
__global__ __launch_bounds__(kInitBlock) void render_init_kernel(apx_component cp, float* planes,
                                                                 RenderWs ws) {
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const int64_t pix = (int64_t)blockIdx.x * kInitBlock + threadIdx.x;
  const Prof<float> p = make_prof<float>(cp);
  float value = 0.0f;
  if (pix < npix) {
    const int i = (int)(pix % cp.nx), j = (int)(pix / cp.nx);
    float X, Y;
    pixel_xy(p, cp, i, j, X, Y);
    float g[APX_NSLOT];
    if (cp.sampling != APX_SAMPLE_MIDPOINT) {
      float centre = 0.0f;
      value = quad_sample<float, GRAD>(p, cp, X, Y, cp.sample_quad, cp.sq_node, cp.sq_weight, 1.0f,
                                       0.5f * p.P00, 0.5f * p.P01, 0.5f * p.P10, 0.5f * p.P11, g,
                                       centre);
      ws.centre[pix] = centre;
    } else {
      value = eval_profile<float, GRAD>(p, X, Y, 1.0f, g);
    }
    planes[pix] = value;
    if (GRAD) {
      for (int c = 1; c < cp.nchan; ++c) {
        const int s = cp.chan_slot[c];
        planes[c * npix + pix] = g[s] * (float)cp.dvdr[s];
      }
    }
  }
  if (cp.mean_reference) {
    // deterministic float64 block sum of the initial samples
    __shared__ double red[kInitBlock / 64];
    double v = wave_sum((double)value);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int w = 0; w < kInitBlock / 64; ++w) t += red[w];
      ws.partial[blockIdx.x] = t;
    }
  }
}

__global__ __launch_bounds__(256) void mean_reference_kernel(RenderWs ws, int64_t nblocks,
                                                             int64_t npix) {
  __shared__ double red[4];
  double t = 0.0;
  for (int64_t b = threadIdx.x; b < nblocks; b += 256) t += ws.partial[b];
  t = wave_sum(t);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) {
    ws.reference[0] = (red[0] + red[1] + red[2] + red[3]) / (double)npix;
    ws.count[0] = 0;
  }
}

// float64 re-decision of one pixel's selection test
__device__ bool select_f64(const apx_component& cp, const Prof<double>& p, int i, int j,
                           double thr) {
  if (cp.sampling == APX_SAMPLE_QUAD) {
    double X, Y, centre = 0.0;
    pixel_xy(p, cp, i, j, X, Y);
    const double res = quad_sample<double, false>(p, cp, X, Y, cp.sample_quad, cp.sq_node,
                                                  cp.sq_weight, 1.0, 0.5 * p.P00, 0.5 * p.P01,
                                                  0.5 * p.P10, 0.5 * p.P11, nullptr, centre);
    return fabs(res - centre) > thr;
  }
  // midpoint: Laplacian of the pixel-centre values; trapezoid: of the means of
  // the pixel corners (_model_methods.py:121-139)
  const int ii = min(max(i, 1), cp.nx - 2), jj = min(max(j, 1), cp.ny - 2);
  double X, Y;
  auto at = [&](int a, int b) {
    pixel_xy(p, cp, a, b, X, Y);
    if (cp.sampling == APX_SAMPLE_TRAPEZOID) {
      double unused;
      return quad_sample<double, false>(p, cp, X, Y, cp.sample_quad, cp.sq_node, cp.sq_weight,
                                        1.0, 0.5 * p.P00, 0.5 * p.P01, 0.5 * p.P10, 0.5 * p.P11,
                                        nullptr, unused);
    }
    return eval_profile<double, false>(p, X, Y, 1.0, nullptr);
  };
  const double mc = at(ii, jj);
  const double curv = at(ii - 1, jj) + at(ii + 1, jj) + at(ii, jj - 1) + at(ii, jj + 1) - 4.0 * mc;
  const double mid = (i == ii && j == jj) ? mc : at(i, j);
  return fabs(mid - (mid + curv)) > thr;  // |deep - reference| (_model_methods.py:164-165)
}

__global__ __launch_bounds__(256) void render_select_kernel(apx_component cp, const float* planes,
                                                            RenderWs ws) {
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const int64_t pix = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const double thr = cp.tolerance * (cp.mean_reference ? ws.reference[0] : cp.reference);
  bool sel = false;
  if (cp.integrate == APX_INTEGRATE_RADIUS) {
    // pixels whose centre lies within the radius of the model centre
    if (pix < npix) {
      const Prof<double> p = make_prof<double>(cp);
      double X, Y;
      pixel_xy(p, cp, (int)(pix % cp.nx), (int)(pix / cp.nx), X, Y);
      // inclusive, with a 1e-9 relative margin: with the centre on a pixel
      // centre (psf_mode "full") lattice points lie exactly on the circle
      sel = X * X + Y * Y <= cp.integrate_radius * cp.integrate_radius * (1.0 + 1e-9);
    }
  } else if (pix < npix) {
    const int i = (int)(pix % cp.nx), j = (int)(pix / cp.nx);
    float metric, scale;
    if (cp.sampling == APX_SAMPLE_QUAD) {
      const float r = planes[pix], c = ws.centre[pix];
      metric = fabsf(r - c);
      scale = fabsf(r) + fabsf(c);
    } else {
      const int ii = min(max(i, 1), cp.nx - 2), jj = min(max(j, 1), cp.ny - 2);
      const float* v = planes + (int64_t)jj * cp.nx + ii;
      const float l = v[-1], r = v[1], u = v[-cp.nx], d = v[cp.nx], m = v[0];
      metric = fabsf(l + r + u + d - 4.0f * m);
      scale = fabsf(l) + fabsf(r) + fabsf(u) + fabsf(d) + 4.0f * fabsf(m);
    }
    // float32 profile values carry at most ~256 ulp of error; inside that band
    // the float64 test decides.
    const double band = 1.6e-5 * (double)scale + 2.0e-7 * thr;
    const double dm = (double)metric;
    if (dm > thr + band) {
      sel = true;
    } else if (dm >= thr - band) {
      const Prof<double> p = make_prof<double>(cp);
      sel = select_f64(cp, p, i, j, thr);
    }
  }
  if (pix < npix) ws.flags[pix] = sel ? 1 : 0;
  const uint64_t ballot = __ballot(sel);
  if (ballot) {
    const int lane = threadIdx.x & 63;
    int base = 0;
    if (lane == 0) base = atomicAdd(ws.count, (int)__popcll(ballot));
    base = __shfl(base, 0, 64);
    if (sel) {
      const uint64_t below = ballot & ((lane == 0) ? 0ull : (~0ull >> (64 - lane)));
      ws.list[base + (int)__popcll(below)] = (int32_t)pix;
    }
  }
}

// float64 adaptive quadrature of listed pixels, one wavefront per pixel
template <bool GRAD>
__global__ __launch_bounds__(256) void render_integrate_kernel(apx_component cp, float* planes,
                                                               RenderWs ws) {
  const int lane = threadIdx.x & 63;
  const int wave = (int)(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int nwaves = (int)(gridDim.x * 4);
  const int count = ws.count[0];
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const Prof<double> p = make_prof<double>(cp);
  const Prof<float> pf = make_prof<float>(cp);
  const double thr1 = cp.tolerance * (cp.mean_reference ? ws.reference[0] : cp.reference);
  for (int k = wave; k < count; k += nwaves) {
    const int32_t pix = ws.list[k];
    double out[1 + APX_NSLOT];
    integrate_pixel<GRAD>(cp, p, pf, cp.nx, cp.ci, cp.cj, pix, thr1, lane, out);
    if (lane == 0) {
      planes[pix] = (float)out[0];
      if (GRAD) {
        for (int c = 1; c < cp.nchan; ++c) {
          const int s = cp.chan_slot[c];
          planes[c * npix + pix] = (float)(out[1 + s] * cp.dvdr[s]);
        }
      }
    }
  }
}

// Adjoint of the render: sum over working pixels of B[q] * d deep[q] / d slot
// for the slots chan_slot[1 .. nchan-1].  Unselected pixels use the float32
// analytic partials (what the Jacobian channels hold); selected pixels
// recompute the forward quadrature (render_vjp_integrate_kernel).
__global__ __launch_bounds__(256) void render_vjp_kernel(apx_component cp,
                                                         const float* __restrict__ B, RenderWs ws,
                                                         int use_flags) {
  __shared__ double red[4][8];
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const int64_t pix = (int64_t)blockIdx.x * kInitBlock + threadIdx.x;
  double acc[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) acc[c] = 0.0;
  if (pix < npix && !(use_flags && ws.flags[pix])) {
    const Prof<float> p = make_prof<float>(cp);
    const int i = (int)(pix % cp.nx), j = (int)(pix / cp.nx);
    float X, Y, g[APX_NSLOT];
    pixel_xy(p, cp, i, j, X, Y);
    if (cp.sampling != APX_SAMPLE_MIDPOINT) {
      float centre;
      quad_sample<float, true>(p, cp, X, Y, cp.sample_quad, cp.sq_node, cp.sq_weight, 1.0f,
                               0.5f * p.P00, 0.5f * p.P01, 0.5f * p.P10, 0.5f * p.P11, g, centre);
    } else {
      eval_profile<float, true>(p, X, Y, 1.0f, g);
    }
    const double w = (double)B[pix];
    for (int c = 1; c < cp.nchan; ++c) acc[c] = w * (double)g[cp.chan_slot[c]];
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int c = 1; c < 8; ++c) {
    const double t = wave_sum(acc[c]);
    if (lane == 0) red[wv][c] = t;
  }
  __syncthreads();
  if (threadIdx.x >= 1 && threadIdx.x < 8)
    ws.partial[blockIdx.x * 8 + threadIdx.x] =
        red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
}

__global__ __launch_bounds__(256) void render_vjp_integrate_kernel(apx_component cp,
                                                                   const float* __restrict__ B,
                                                                   RenderWs ws) {
  __shared__ double red[4][8];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int wave = (int)(blockIdx.x * 4 + wv);
  const int nwaves = (int)(gridDim.x * 4);
  const int count = ws.count[0];
  const Prof<double> p = make_prof<double>(cp);
  const Prof<float> pf = make_prof<float>(cp);
  const double thr1 = cp.tolerance * (cp.mean_reference ? ws.reference[0] : cp.reference);
  double acc[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) acc[c] = 0.0;
  for (int k = wave; k < count; k += nwaves) {
    const int32_t pix = ws.list[k];
    double out[1 + APX_NSLOT];
    integrate_pixel<true>(cp, p, pf, cp.nx, cp.ci, cp.cj, pix, thr1, lane, out);
    const double w = (double)B[pix];
    for (int c = 1; c < cp.nchan; ++c) acc[c] += w * out[1 + cp.chan_slot[c]];
  }
  if (lane == 0)
    for (int c = 0; c < 8; ++c) red[wv][c] = acc[c];
  __syncthreads();
  if (threadIdx.x >= 1 && threadIdx.x < 8)
    ws.vpart[blockIdx.x * 8 + threadIdx.x] =
        red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
}

// One workgroup a slot, 256 partials in flight a step (a thread a slot read the
// 7,900 partials of a 1537 x 1201 image one after another: 1.24 ms; now 14 us).
__global__ __launch_bounds__(256) void render_vjp_final_kernel(apx_component cp, RenderWs ws,
                                                               int nb1, int nb2, double* grad) {
  __shared__ double red[4];
  const int c = blockIdx.x + 1;
  double t = 0.0;
  for (int b = threadIdx.x; b < nb1; b += 256) t += ws.partial[b * 8 + c];
  for (int b = threadIdx.x; b < nb2; b += 256) t += ws.vpart[b * 8 + c];
  t = wave_sum(t);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = t;
  __syncthreads();
  if (threadIdx.x == 0) grad[c - 1] = (red[0] + red[1] + red[2] + red[3]) * cp.dvdr[cp.chan_slot[c]];
}

__global__ void zero_count_kernel(RenderWs ws) { ws.count[0] = 0; }

// PSF_Model.sample's normalisation to unit sum (psf_model_object.py:255-257)
// applied to render planes: plane 0 becomes P / S with S = sum P, and each
// derivative plane dP becomes the derivative of P / S, dP / S - P (sum dP) / S^2.
// One workgroup of 16 wavefronts; float64 sums in a fixed order.
__global__ __launch_bounds__(1024) void normalize_planes_kernel(float* planes, int nchan,
                                                                int64_t npix) {
  __shared__ double red[APX_MAX_CHAN][16];
  __shared__ double tot[APX_MAX_CHAN];
  double s[APX_MAX_CHAN];
#pragma unroll
  for (int c = 0; c < APX_MAX_CHAN; ++c) s[c] = 0.0;
  for (int64_t p = threadIdx.x; p < npix; p += 1024) {
#pragma unroll
    for (int c = 0; c < APX_MAX_CHAN; ++c)
      if (c < nchan) s[c] += (double)planes[c * npix + p];
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int c = 0; c < APX_MAX_CHAN; ++c) {
    if (c < nchan) {
      const double v = wave_sum(s[c]);
      if (lane == 0) red[c][w] = v;
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < nchan) {
    double t = 0.0;
    for (int k = 0; k < 16; ++k) t += red[threadIdx.x][k];
    tot[threadIdx.x] = t;
  }
  __syncthreads();
  const double iS = 1.0 / tot[0];
  for (int64_t p = threadIdx.x; p < npix; p += 1024) {
    const double v = (double)planes[p];
    for (int c = 1; c < nchan; ++c)
      planes[c * npix + p] = (float)((double)planes[c * npix + p] * iS - v * tot[c] * iS * iS);
    planes[p] = (float)(v * iS);
  }
}

}  // namespace

int normalize_planes(float* planes, int32_t nchan, int64_t npix, hipStream_t stream) {
  if (!planes) return set_error(APX_E_INVALID, "normalize_planes: null pointer");
  if (nchan < 1 || nchan > APX_MAX_CHAN)
    return set_error(APX_E_INVALID, "normalize_planes: nchan out of range");
  if (npix < 1) return set_error(APX_E_INVALID, "normalize_planes: no pixels");
  hipLaunchKernelGGL(normalize_planes_kernel, dim3(1), dim3(1024), 0, stream, planes, nchan, npix);
  return check_launch("normalize_planes");
}

int64_t render_workspace_bytes(int64_t npix) {
  return 256 + align256(8 * 8 * init_blocks(npix)) + align256(4 * npix) + align256(4 * npix) +
         align256(npix) + align256(8 * 8 * (kIntegrateWaves / 4));
}

int render_component(const apx_component* cp_in, float* planes, void* workspace, int64_t ws_bytes,
                     hipStream_t stream) {
  if (!cp_in || !planes || !workspace) return set_error(APX_E_INVALID, "render: null pointer");
  apx_component cp = *cp_in;
  if (cp.integrate == APX_INTEGRATE_RADIUS) {
    if (!(cp.integrate_radius >= 0.0))
      return set_error(APX_E_INVALID, "render: integrate_radius must be >= 0");
    cp.max_depth = 1;  // one Gauss-Legendre level, no refinement
    cp.gridding = 1;
  } else if (cp.integrate != APX_INTEGRATE_NONE && cp.integrate != APX_INTEGRATE_THRESHOLD) {
    return set_error(APX_E_INVALID, "render: unknown integrate mode");
  }
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  if (cp.nx < 3 || cp.ny < 3) return set_error(APX_E_INVALID, "render: working grid below 3x3");
  if (npix > (int64_t)INT32_MAX) return set_error(APX_E_LIMIT, "render: grid too large");
  if (ws_bytes < render_workspace_bytes(npix))
    return set_error(APX_E_INVALID, "render: workspace too small");
  if (cp.profile < APX_SERSIC || cp.profile > APX_FLAT_SKY)
    return set_error(APX_E_INVALID, "render: unknown profile");
  if (cp.nchan < 1 || cp.nchan > APX_MAX_CHAN)
    return set_error(APX_E_INVALID, "render: nchan out of range");
  for (int c = 1; c < cp.nchan; ++c)
    if (cp.chan_slot[c] < 0 || cp.chan_slot[c] >= APX_NSLOT)
      return set_error(APX_E_INVALID, "render: bad channel slot");
  if (cp.sampling < APX_SAMPLE_MIDPOINT || cp.sampling > APX_SAMPLE_TRAPEZOID)
    return set_error(APX_E_INVALID, "render: unknown sampling mode");
  if (cp.sampling != APX_SAMPLE_MIDPOINT &&
      (cp.sample_quad < 1 || cp.sample_quad > APX_MAX_QUAD_LEVEL))
    return set_error(APX_E_LIMIT, "render: sampling quad level out of range");
  if (cp.integrate) {
    if (cp.quad_level < 1 || cp.quad_level > APX_MAX_QUAD_LEVEL)
      return set_error(APX_E_LIMIT, "render: integrate_quad_level out of range");
    if (cp.gridding < 1 || cp.gridding > APX_MAX_GRIDDING)
      return set_error(APX_E_LIMIT, "render: integrate_gridding out of range");
    if (cp.max_depth < 1 || cp.max_depth > APX_MAX_DEPTH)
      return set_error(APX_E_LIMIT, "render: integrate_max_depth out of range");
  }
  const RenderWs ws = carve(workspace, npix);
  const bool grad = cp.nchan > 1;
  const int64_t nb = init_blocks(npix);
  if (grad)
    hipLaunchKernelGGL(render_init_kernel<true>, dim3((unsigned)nb), dim3(kInitBlock), 0, stream,
                       cp, planes, ws);
  else
    hipLaunchKernelGGL(render_init_kernel<false>, dim3((unsigned)nb), dim3(kInitBlock), 0, stream,
                       cp, planes, ws);
  if (cp.mean_reference)
    hipLaunchKernelGGL(mean_reference_kernel, dim3(1), dim3(256), 0, stream, ws, nb, npix);
  else
    hipLaunchKernelGGL(zero_count_kernel, dim3(1), dim3(1), 0, stream, ws);
  if (cp.integrate) {
    hipLaunchKernelGGL(render_select_kernel, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0,
                       stream, cp, planes, ws);
    const int blocks = (int)std::min<int64_t>((npix + 3) / 4, kIntegrateWaves / 4);
    if (grad)
      hipLaunchKernelGGL(render_integrate_kernel<true>, dim3(blocks), dim3(256), 0, stream, cp,
                         planes, ws);
    else
      hipLaunchKernelGGL(render_integrate_kernel<false>, dim3(blocks), dim3(256), 0, stream, cp,
                         planes, ws);
  }
  return check_launch("render");
}

int render_vjp(const apx_component* cp_in, const float* weights, float* value_plane, double* grad,
               void* workspace, int64_t ws_bytes, hipStream_t stream) {
  if (!cp_in || !weights || !value_plane || !grad)
    return set_error(APX_E_INVALID, "render_vjp: null pointer");
  apx_component cp = *cp_in;
  if (cp.nchan < 2) return set_error(APX_E_INVALID, "render_vjp: no slots requested (nchan < 2)");
  if (cp.integrate == APX_INTEGRATE_RADIUS) {
    cp.max_depth = 1;
    cp.gridding = 1;
  }
  // the value render (supersamples recomputed) establishes the selection
  apx_component cv = cp;
  cv.nchan = 1;
  int rc = render_component(&cv, value_plane, workspace, ws_bytes, stream);
  if (rc) return rc;
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const RenderWs ws = carve(workspace, npix);
  const int64_t nb = init_blocks(npix);
  hipLaunchKernelGGL(render_vjp_kernel, dim3((unsigned)nb), dim3(kInitBlock), 0, stream, cp, weights,
                     ws, cp.integrate);
  int nb2 = 0;
  if (cp.integrate) {
    nb2 = (int)std::min<int64_t>((npix + 3) / 4, kIntegrateWaves / 4);
    hipLaunchKernelGGL(render_vjp_integrate_kernel, dim3(nb2), dim3(256), 0, stream, cp, weights, ws);
  }
  hipLaunchKernelGGL(render_vjp_final_kernel, dim3(cp.nchan - 1), dim3(256), 0, stream, cp, ws, (int)nb, nb2,
                     grad);
  return check_launch("render_vjp");
}

int render_selected_count(const void* workspace, hipStream_t stream, int32_t* count) {
  if (!workspace || !count) return set_error(APX_E_INVALID, "selected_count: null pointer");
  if (hipMemcpyAsync(count, workspace, sizeof(int32_t), hipMemcpyDeviceToHost, stream) !=
      hipSuccess)
    return set_error(APX_E_HIP, "selected_count: copy failed");
  if (hipStreamSynchronize(stream) != hipSuccess)
    return set_error(APX_E_HIP, "selected_count: sync failed");
  return APX_OK;
}

}  // namespace apx
