// Component render on gfx950: initial sampling, curvature-threshold selection
// and adaptive Gauss-Legendre supersampling of the selected pixels.
//
// Restates models/_model_methods.py:82-184 (_sample_init midpoint / quad:N,
// _sample_integrate threshold) and utils/operations.py:94-247
// (single_quad_integrate, grid_integrate) as four launches:
//   1. init     : one thread per working pixel, float32 profile value and
//                 Jacobian channels; a float64 per-block partial sum when the
//                 integrate reference is the mean sample.
//   2. select   : curvature (replicate-padded 5-point Laplacian) or |quad -
//                 centre node|, compared with tolerance * reference.  Pixels
//                 whose float32 test lies within a rounding band of the
//                 threshold are re-decided in float64, so the selected set is
//                 the float64 one.  Selected pixels are appended to a list with
//                 one atomic per wavefront.
//   3. level 1  : float64 Gauss-Legendre of the selected pixels, one lane a
//                 node; a pixel that needs refining goes to a second list.
//   4. deep     : levels 2 and 3 of those (threshold x gridding^2 per level as
//                 in operations.py:241), a workgroup a pixel; float32 samples
//                 summed in float64.
// The adjoint runs 3 and 4 again, reducing against its weights.
#include <hip/hip_runtime.h>

#include "capi_internal.h"
#include "profile.h"
#include "render_common.h"

namespace apx {

namespace {

constexpr int kInitBlock = 256;
constexpr int kLevelBlocks = 512;  // workgroups of the level-1 pass
constexpr int kDeepBlocks = 1024;  // workgroups of the deep pass

// workspace layout (bytes)
struct RenderWs {
  int32_t* count;     // [0]: selected pixels, [1]: those refined past level 1
  double* reference;  // mean-sample reference (when mean_reference)
  double* partial;    // per-init-block sums
  int32_t* list;      // selected pixel indices
  float* centre;      // quad:N centre-node samples
  int32_t* deep;      // refined pixel indices (in place of centre once the selection is made)
  uint8_t* flags;     // 1 = pixel selected for integration, 2 = refined past level 1
  double* vpart;      // adjoint sums of the level-1 and deep workgroups (8 per block)
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
  w.deep = reinterpret_cast<int32_t*>(b + off);
  off += align256(4 * npix);
  w.flags = reinterpret_cast<uint8_t*>(b + off);
  off += align256(npix);
  w.vpart = reinterpret_cast<double*>(b + off);
  return w;
}

template <bool GRAD>
__global__ __launch_bounds__(kInitBlock) void render_init_kernel(apx_component cp, RenderConst rc, float* planes,
                                                                 RenderWs ws) {
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const int64_t pix = (int64_t)blockIdx.x * kInitBlock + threadIdx.x;
  const Prof<float>& p = rc.f;
  if (blockIdx.x == 0 && threadIdx.x < 2) ws.count[threadIdx.x] = 0;
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
  if (cp.mean_reference && cp.integrate) {
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
  }
}

// float64 re-decision of one pixel's selection test under quad sampling
__device__ bool select_f64(const apx_component& cp, const Prof<double>& p, int i, int j,
                           double thr) {
  double X, Y, centre = 0.0;
  pixel_xy(p, cp, i, j, X, Y);
  const double res = quad_sample<double, false>(p, cp, X, Y, cp.sample_quad, cp.sq_node,
                                                cp.sq_weight, 1.0, 0.5 * p.P00, 0.5 * p.P01,
                                                0.5 * p.P10, 0.5 * p.P11, nullptr, centre);
  return fabs(res - centre) > thr;
}

// The same under midpoint sampling (the Laplacian of the pixel-centre values) and
// trapezoid sampling (of the means of the pixel corners, _model_methods.py:121-139),
// for the wave's pixels with `close`: the six float64 samples of a pixel go to six
// lanes, ten pixels at once.  One lane took them one after another, which set the
// time of the selection (512^2: 7.6 -> 5.8 us, 100^2: 7.0 -> 4.8).  Every lane of the wave calls it.
__device__ __forceinline__ bool select_close(const apx_component& cp, const Prof<double>& p, bool close, int i, int j,
                                             double thr) {
  const uint64_t todo = __ballot(close);
  if (!todo) return false;
  const int lane = threadIdx.x & 63, slot = lane / 6, pt = lane - 6 * slot, count = (int)__popcll(todo);
  const int rank = (int)__popcll(todo & ((1ull << lane) - 1ull));
  bool sel = false;
  for (int first = 0; first < count; first += 10) {
    uint64_t m = todo;
    for (int q = 0; q < first + slot; ++q) m &= m - 1ull;
    const int owner = m ? __ffsll((unsigned long long)m) - 1 : 0;
    const int oi = __shfl(i, owner, 64), oj = __shfl(j, owner, 64);
    double val = 0.0;
    if (slot < 10 && m) {  // the centre, its left, right, upper and lower neighbours, the pixel
      const int ii = min(max(oi, 1), cp.nx - 2), jj = min(max(oj, 1), cp.ny - 2);
      const int a = pt == 1 ? ii - 1 : pt == 2 ? ii + 1 : pt == 5 ? oi : ii;
      const int b = pt == 3 ? jj - 1 : pt == 4 ? jj + 1 : pt == 5 ? oj : jj;
      double X, Y;
      pixel_xy(p, cp, a, b, X, Y);
      if (cp.sampling == APX_SAMPLE_TRAPEZOID) {
        double unused;
        val = quad_sample<double, false>(p, cp, X, Y, cp.sample_quad, cp.sq_node, cp.sq_weight,
                                         1.0, 0.5 * p.P00, 0.5 * p.P01, 0.5 * p.P10, 0.5 * p.P11,
                                         nullptr, unused);
      } else {
        val = eval_profile<double, false>(p, X, Y, 1.0, nullptr);
      }
    }
    const bool mine = close && rank >= first && rank < first + 10;
    const int base = mine ? 6 * (rank - first) : 0;
    double at[6];
#pragma unroll
    for (int q = 0; q < 6; ++q) at[q] = __shfl(val, base + q, 64);
    if (mine) {
      const double curv = at[1] + at[2] + at[3] + at[4] - 4.0 * at[0];
      const double mid = at[5];
      sel = fabs(mid - (mid + curv)) > thr;  // |deep - reference| (_model_methods.py:164-165)
    }
  }
  return sel;
}

__global__ __launch_bounds__(256) void render_select_kernel(apx_component cp, RenderConst rc, const float* planes,
                                                            RenderWs ws) {
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const int64_t pix = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const double thr = cp.tolerance * (cp.mean_reference ? ws.reference[0] : cp.reference);
  // a list entry is an int32, so a pixel index fits 32 bits
  const int j = (int)((uint32_t)pix / (uint32_t)cp.nx), i = (int)((uint32_t)pix - (uint32_t)j * (uint32_t)cp.nx);
  bool sel = false, close = false;
  if (cp.integrate == APX_INTEGRATE_RADIUS) {
    // pixels whose centre lies within the radius of the model centre
    if (pix < npix) {
      double X, Y;
      pixel_xy(rc.d, cp, i, j, X, Y);
      // inclusive, with a 1e-9 relative margin: with the centre on a pixel
      // centre (psf_mode "full") lattice points lie exactly on the circle
      sel = X * X + Y * Y <= cp.integrate_radius * cp.integrate_radius * (1.0 + 1e-9);
    }
  } else if (pix < npix) {
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
      close = cp.sampling != APX_SAMPLE_QUAD;
      if (!close) sel = select_f64(cp, rc.d, i, j, thr);
    }
  }
  if (select_close(cp, rc.d, close, i, j, thr)) sel = true;
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

// What the quadrature passes do with a pixel's sums: write the value, the value
// and the channels, or (adjoint) add them, weighted, to the workgroup's sums.
enum : int { Q_VALUE = 0, Q_GRAD = 1, Q_VJP = 2 };

// the workgroup's adjoint sums of slots chan_slot[1 .. nchan-1] into part[0 .. 7]
__device__ __forceinline__ void vjp_part(const apx_component& cp, const double* acc, double* part) {
  __shared__ double red[4][8];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int s = 0; s < APX_NSLOT; ++s) {
    const double t = wave_sum(acc[s]);
    if (lane == 0) red[wv][s] = t;
  }
  __syncthreads();
  const int c = threadIdx.x;
  if (c >= 1 && c < cp.nchan) {
    const int s = cp.chan_slot[c];
    part[c] = red[0][s] + red[1][s] + red[2][s] + red[3][s];
  }
}

// Level 1 of the listed pixels (operations.py:210-228, area 1, float64, which
// is the value of every selected pixel that is not refined further): one lane a
// node, 64 / quad_level^2 pixels a wave (7 for the 3 x 3 rule), the nodes'
// terms added in node order by lane reads.  Bound by the latency of one float64
// sample and its sum.  A wave a pixel kept 9 lanes of 64 busy, and carried the
// pixel's deeper levels in the same wave (render_deep_kernel): 51 us for a 100^2
// cutout, 71 us for 1537 x 1201 (adjoint 114); 17 and 35 us (42) the two passes.
// ROW: lanes a pixel, summed by a butterfly, for rules of more than 9 nodes, whose
// many lane reads would take longer than their samples (level1_row).
template <int MODE, int ROW>
__global__ __launch_bounds__(256) void render_level1_kernel(apx_component cp, RenderConst rc, float* planes,
                                                            const float* __restrict__ B, RenderWs ws) {
  constexpr bool GRAD = MODE != Q_VALUE;
  const int lane = threadIdx.x & 63;
  const int n = cp.quad_level, nn = n * n, width = ROW ? ROW : nn, per = 64 / width;
  const int grp = lane / width, at = lane - grp * width, first = grp * width;
  const bool has = ROW == 0 || at < nn;  // this lane holds a node
  const int node = has ? at : 0;
  auto sum = [&](double v) {
    if constexpr (ROW == 64) return wave_sum(v);
    else if constexpr (ROW == 32) return half_sum(v);
    else if constexpr (ROW == 16) return row_sum(v);
    double r = 0.0;
    for (int j = 0; j < nn; ++j) r += __shfl(v, first + j, 64);
    return r;
  };
  const int wv = threadIdx.x >> 6, wave = (int)blockIdx.x * 4 + wv, nwaves = (int)(gridDim.x * 4);
  // The wave's refined pixels, appended to the list 64 at a time: where most pixels
  // are refined, an atomic a step on the one counter sets the time (512^2, 4 x 4
  // nodes, depth 2, tolerance 1e-4: 341 us, so 170).
  __shared__ int32_t pend[4][64];
  int npend = 0;
  auto flush = [&]() {
    if (npend == 0) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    int base = 0;
    if (lane == 0) base = atomicAdd(ws.count + 1, npend);
    base = __shfl(base, 0, 64);
    if (lane < npend) ws.deep[base + lane] = pend[wv][lane];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    npend = 0;
  };
  const int count = ws.count[0];
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const Prof<double>& p = rc.d;
  const double thr1 = cp.tolerance * (cp.mean_reference ? ws.reference[0] : cp.reference);
  const double u = cp.gl_node[node % n], v = cp.gl_node[node / n];
  const double w = cp.gl_weight[node % n] * cp.gl_weight[node / n] * 0.25;
  const double ox = 0.5 * (p.P00 * u + p.P01 * v), oy = 0.5 * (p.P10 * u + p.P11 * v);
  double adj[APX_NSLOT];
#pragma unroll
  for (int s = 0; s < APX_NSLOT; ++s) adj[s] = 0.0;
  for (int k0 = wave * per; k0 < count; k0 += nwaves * per) {
    const int k = k0 + grp;
    const bool on = grp < per && k < count;
    const int32_t pix = on ? ws.list[k] : 0;
    if (MODE == Q_VJP && (!on || !has || ws.flags[pix] == 2)) continue;  // no lane reads below
    double X0, Y0, gl[APX_NSLOT];
    pixel_xy(p, cp, pix % cp.nx, pix / cp.nx, X0, Y0);
    const double v1 = eval_profile<double, GRAD>(p, X0 + ox, Y0 + oy, 1.0, gl);
    if (MODE == Q_VJP) {
      const double wb = w * (double)B[pix];
#pragma unroll
      for (int s = 0; s < APX_NSLOT; ++s) adj[s] += wb * gl[s];
      continue;
    }
    const double res = sum(has ? w * v1 : 0.0);
    const double centre = __shfl(v1, first + nn / 2, 64);
    const bool refine = on && cp.max_depth > 1 && fabs(res - centre) > thr1;
    double gs[APX_NSLOT];
    if (GRAD) {
#pragma unroll
      for (int s = 0; s < APX_NSLOT; ++s) gs[s] = sum(has ? w * gl[s] : 0.0);
    }
    const bool lead = on && at == 0;
    if (lead && !refine) {
      planes[pix] = (float)res;
      if (GRAD)
        for (int c = 1; c < cp.nchan; ++c) {
          const int s = cp.chan_slot[c];
          planes[c * npix + pix] = (float)(gs[s] * cp.dvdr[s]);
        }
    }
    const uint64_t ballot = __ballot(lead && refine);
    if (ballot) {
      const int c = (int)__popcll(ballot);
      if (npend + c > 64) flush();
      if (lead && refine) {
        pend[wv][npend + (int)__popcll(ballot & ((1ull << lane) - 1ull))] = pix;
        ws.flags[pix] = 2;
      }
      npend += c;
    }
  }
  if (MODE != Q_VJP) flush();
  if (MODE == Q_VJP) vjp_part(cp, adj, ws.vpart + 8 * blockIdx.x);
}

// Levels 2 and 3 of the refined pixels (operations.py:229-247), a workgroup a
// pixel.  Samples are float32, sums float64; a level-2 test whose float32 value
// lies within kSampleBand of its threshold is taken again from float64 samples,
// so the sub-pixels refined are the ones float64 arithmetic picks.  The samples
// of every flagged sub-pixel form one run that the 256 threads share, so that a
// cuspy centre pixel, up to 25 x 225 samples, is not one wave's serial chain.
// FAST: the default 3 x 3 rule on 5 x 5 sub-pixels, whose 225 level-2 samples
// take a thread each (summed per sub-pixel in node order); else each sub-pixel's
// nodes are dealt out to `slices` threads, as many as fit, whose partial sums one
// thread adds; and where more pixels are listed than workgroups were launched (a
// rule without a central node refines every selected pixel) a workgroup takes four
// at once, level 2 of each by a wave of its own: 512^2, 4 x 4 nodes, depth 2,
// tolerance 1e-4, Jacobian 761 us a pixel at a time, 265 so (with the
// list of render_level1_kernel).
template <int MODE, bool FAST>
__global__ __launch_bounds__(256) void render_deep_kernel(apx_component cp, RenderConst rc, float* planes,
                                                          const float* __restrict__ B, RenderWs ws, int voff) {
  constexpr bool GRAD = MODE != Q_VALUE;
  constexpr int NV = GRAD ? 1 + APX_NSLOT : 1;
  constexpr int NS = FAST ? 225 : 1, NG = FAST ? 1 : 64;
  __shared__ float sample[NV][FAST ? NS : 256], middle[NG];
  __shared__ double sx[(FAST ? 1 : 4) * 64], sy[(FAST ? 1 : 4) * 64];  // flagged sub-pixels (of up to four pixels)
  __shared__ double ox3[NS], oy3[NS], w3[NS];
  __shared__ double nodeu[NG], nodev[NG], nodew[NG], suba[NG], subb[NG];  // node q; sub-pixel's place in its pixel
  __shared__ double red[4][NV];
  __shared__ double red3[FAST ? 1 : 4][4][NV];
  __shared__ int nflag, nflags[4], pixel[4];
  const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
  const int n = FAST ? 3 : cp.quad_level, nn = n * n, g = FAST ? 5 : cp.gridding, gg = g * g;
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const Prof<double>& p = rc.d;
  const Prof<float>& pf = rc.f;
  const double thr1 = cp.tolerance * (cp.mean_reference ? ws.reference[0] : cp.reference);
  const double ig = 1.0 / (double)g, sub0 = -(double)(g - 1) / (2.0 * g), subd = ig;
  const double sc2 = ig * ig, thr2 = thr1 * (double)gg, sc3 = sc2 * ig * ig;
  const float h = (float)(0.5 * ig);
  // offset and weight of level-3 sample e of a sub-pixel: sub-sub-pixel e / nn, node e % nn
  auto offset3 = [&](int e, double& x, double& y, double& w) {
    const int q = e / nn, kk = e - q * nn;
    const double a = (FAST ? sub0 + subd * (q % g) : suba[q]) * ig, b = (FAST ? sub0 + subd * (q / g) : subb[q]) * ig;
    const double hu = a + 0.5 * ig * ig * (FAST ? cp.gl_node[kk % n] : nodeu[kk]);
    const double hv = b + 0.5 * ig * ig * (FAST ? cp.gl_node[kk / n] : nodev[kk]);
    x = p.P00 * hu + p.P01 * hv;
    y = p.P10 * hu + p.P11 * hv;
    w = FAST ? cp.gl_weight[kk % n] * cp.gl_weight[kk / n] * 0.25 : nodew[kk];
  };
  const int count = ws.count[1];
  double adj[APX_NSLOT];
#pragma unroll
  for (int s = 0; s < APX_NSLOT; ++s) adj[s] = 0.0;
  if (FAST) {  // ahead of the first use of count, which is on its way
    if (t < NS) offset3(t, ox3[t], oy3[t], w3[t]);
  } else {
    if (t < nn) {
      nodeu[t] = cp.gl_node[t % n];
      nodev[t] = cp.gl_node[t / n];
      nodew[t] = cp.gl_weight[t % n] * cp.gl_weight[t / n] * 0.25;
    }
    if (t < gg) {
      suba[t] = sub0 + subd * (t % g);
      subb[t] = sub0 + subd * (t / g);
    }
    __syncthreads();
  }
  if ((int)blockIdx.x >= count) {  // no pixel for this workgroup
    if (MODE == Q_VJP) vjp_part(cp, adj, ws.vpart + 8 * (voff + blockIdx.x));
    return;
  }
  // sub-pixel and (first) node of this thread at level 2
  const int slices = FAST ? 9 : min(nn, 256 / gg);
  const int sub = FAST ? t / 9 : t % gg, k2 = FAST ? t - 9 * sub : t / gg;
  const double sa = sub0 + subd * (sub % g), sb = sub0 + subd * (sub / g);
  const double sdx = p.P00 * sa + p.P01 * sb, sdy = p.P10 * sa + p.P11 * sb;
  const float nu = FAST ? (float)cp.gl_node[k2 % 3] : 0.0f, nv = FAST ? (float)cp.gl_node[k2 / 3] : 0.0f;
  auto weight2 = [&](int q) { return (float)(cp.gl_weight[q % 3] * cp.gl_weight[q / 3] * 0.25); };
  // does float64 arithmetic refine the sub-pixel at (x2, y2) with float32 value r2, centre node `centre`
  auto refine = [&](double x2, double y2, float r2, float centre) {
    const double D = fabs((double)r2 - (double)centre);
    const double band = kSampleBand * (fabs((double)r2) + fabs((double)centre)) + 1e-7 * thr2;
    if (D > thr2 + band) return true;
    if (!(D >= thr2 - band)) return false;
    double cd = 0.0;
    const double rd = quad_sample<double, false>(p, cp, x2, y2, n, cp.gl_node, cp.gl_weight, sc2, 0.5 * ig * p.P00,
                                                 0.5 * ig * p.P01, 0.5 * ig * p.P10, 0.5 * ig * p.P11, nullptr, cd);
    return fabs(rd - cd) > thr2;
  };
  // weighted level-2 samples of nodes q0, q0 + step, .. of the sub-pixel at (x2, y2), added to part
  auto nodes2 = [&](float x2, float y2, int q0, int step, float (&part)[NV], float& centre) {
    for (int q = q0; q < nn; q += step) {
      const float u = (float)nodeu[q], v = (float)nodev[q], w = (float)nodew[q];
      float gl[APX_NSLOT];
      const float val = eval_profile<float, GRAD>(pf, x2 + h * pf.P00 * u + h * pf.P01 * v,
                                                  y2 + h * pf.P10 * u + h * pf.P11 * v, (float)sc2, gl);
      part[0] += w * val;
      if (q == nn / 2) centre = val;
      if (GRAD) {
#pragma unroll
        for (int s = 0; s < APX_NSLOT; ++s) part[1 + s] += w * gl[s];
      }
    }
  };
  // level 3: the samples of nf flagged sub-pixels, one run over the workgroup, added to acc
  auto level3 = [&](const double* xs, const double* ys, int nf, double (&acc)[NV]) {
    const int per3 = gg * nn, total3 = nf * per3;
    for (int e = t; e < total3; e += 256) {
      const int f = e / per3, q = e - f * per3;
      double dx, dy, w;
      if (FAST) {
        dx = ox3[q];
        dy = oy3[q];
        w = w3[q];
      } else {
        offset3(q, dx, dy, w);
      }
      float gl[APX_NSLOT];
      const float val = eval_profile<float, GRAD>(pf, (float)(xs[f] + dx), (float)(ys[f] + dy), (float)sc3, gl);
      acc[0] += w * (double)val;
      if (GRAD) {
#pragma unroll
        for (int s = 0; s < APX_NSLOT; ++s) acc[1 + s] += w * (double)gl[s];
      }
    }
  };
  const bool many = !FAST && count > (int)gridDim.x;
  if (many) {
    const int deal = min(nn, 64 / gg), mine = lane % gg, q0 = lane / gg;
    for (int k0 = blockIdx.x; k0 < count; k0 += 4 * (int)gridDim.x) {
      const int k = k0 + wv * (int)gridDim.x;
      const bool on = k < count;
      const int32_t pix = on ? ws.deep[k] : 0;
      double X0, Y0;
      pixel_xy(p, cp, pix % cp.nx, pix / cp.nx, X0, Y0);
      const double x2 = X0 + p.P00 * suba[mine] + p.P01 * subb[mine], y2 = Y0 + p.P10 * suba[mine] + p.P11 * subb[mine];
      float part[NV], own = 0.0f;
#pragma unroll
      for (int s = 0; s < NV; ++s) part[s] = 0.0f;
      if (on && q0 < deal) nodes2((float)x2, (float)y2, q0, deal, part, own);
      const float centre = __shfl(own, (nn / 2) % deal * gg + mine, 64);
      float r2 = 0.0f;
      double acc[NV];
#pragma unroll
      for (int s = 0; s < NV; ++s) {
        float v = 0.0f;
        for (int j = 0; j < deal; ++j) v += __shfl(part[s], j * gg + mine, 64);
        if (s == 0) r2 = v;
        acc[s] = (double)v;
      }
      const bool deeper = on && lane < gg && cp.max_depth > 2 && refine(x2, y2, r2, centre);
      if (lane >= gg || deeper) {
#pragma unroll
        for (int s = 0; s < NV; ++s) acc[s] = 0.0;
      }
      const uint64_t flags = __ballot(deeper);
      if (deeper) {
        const int at = 64 * wv + (int)__popcll(flags & ((1ull << lane) - 1ull));
        sx[at] = x2;
        sy[at] = y2;
      }
      if (lane == 0) {
        nflags[wv] = (int)__popcll(flags);
        pixel[wv] = pix;
      }
      if (MODE == Q_VJP) {
        const double wb = on ? (double)B[pix] : 0.0;
#pragma unroll
        for (int s = 0; s < APX_NSLOT; ++s) adj[s] += wb * acc[1 + s];
      } else {
#pragma unroll
        for (int s = 0; s < NV; ++s) {
          const double a = wave_sum(acc[s]);
          if (lane == 0) red[wv][s] = a;
        }
      }
      __syncthreads();
      // level 3 of each wave's pixel by the whole workgroup
      for (int j = 0; j < 4; ++j) {
        const int nf = nflags[j];
        if (nf == 0) continue;
        double a3[NV];
#pragma unroll
        for (int s = 0; s < NV; ++s) a3[s] = 0.0;
        level3(sx + 64 * j, sy + 64 * j, nf, a3);
        if (MODE == Q_VJP) {
          const double wb = (double)B[pixel[j]];
#pragma unroll
          for (int s = 0; s < APX_NSLOT; ++s) adj[s] += wb * a3[1 + s];
        } else {
#pragma unroll
          for (int s = 0; s < NV; ++s) {
            const double a = wave_sum(a3[s]);
            if (lane == 0) red3[j][wv][s] = a;
          }
        }
      }
      __syncthreads();
      if (MODE != Q_VJP && on && lane < cp.nchan && (GRAD || lane == 0)) {
        const int s = lane == 0 ? 0 : 1 + cp.chan_slot[lane];
        double a = red[wv][s];
        if (nflags[wv] > 0) a += red3[wv][0][s] + red3[wv][1][s] + red3[wv][2][s] + red3[wv][3][s];
        planes[lane * npix + pix] = (float)(lane == 0 ? a : a * cp.dvdr[s - 1]);
      }
      __syncthreads();  // the next pixels write sx, sy, red and red3 again
    }
  }
  for (int k = many ? count : (int)blockIdx.x; k < count; k += gridDim.x) {
    const int32_t pix = ws.deep[k];
    double X0, Y0;
    pixel_xy(p, cp, pix % cp.nx, pix / cp.nx, X0, Y0);
    double acc[NV];
#pragma unroll
    for (int s = 0; s < NV; ++s) acc[s] = 0.0;
    if (FAST) {
      if (t < NS) {
        float gl[APX_NSLOT];
        const float val = eval_profile<float, GRAD>(pf, (float)(X0 + sdx) + h * pf.P00 * nu + h * pf.P01 * nv,
                                                    (float)(Y0 + sdy) + h * pf.P10 * nu + h * pf.P11 * nv, (float)sc2, gl);
        sample[0][t] = val;
        if (GRAD) {
#pragma unroll
          for (int s = 0; s < APX_NSLOT; ++s) sample[1 + s][t] = gl[s];
        }
      }
    } else if (k2 < slices) {
      float part[NV], centre = 0.0f;
#pragma unroll
      for (int s = 0; s < NV; ++s) part[s] = 0.0f;
      nodes2((float)(X0 + sdx), (float)(Y0 + sdy), k2, slices, part, centre);
      if (k2 == (nn / 2) % slices) middle[sub] = centre;
#pragma unroll
      for (int s = 0; s < NV; ++s) sample[s][t] = part[s];
    }
    __syncthreads();
    // level 2: thread t < gg sums sub-pixel t and tests it
    if (t < 64) {
      bool deeper = false;
      double x2 = 0.0, y2 = 0.0;
      if (t < gg) {
        const double a = sub0 + subd * (t % g), b = sub0 + subd * (t / g);
        x2 = X0 + p.P00 * a + p.P01 * b;
        y2 = Y0 + p.P10 * a + p.P11 * b;
        float gs[APX_NSLOT], centre = 0.0f, r2 = 0.0f;
        if (FAST) {
#pragma unroll
          for (int q = 0; q < 9; ++q) r2 += weight2(q) * sample[0][9 * t + q];
          centre = sample[0][9 * t + 4];
          if (GRAD) {
#pragma unroll
            for (int s = 0; s < APX_NSLOT; ++s) {
              gs[s] = 0.0f;
#pragma unroll
              for (int q = 0; q < 9; ++q) gs[s] += weight2(q) * sample[1 + s][9 * t + q];
            }
          }
        } else {
          for (int q = 0; q < slices; ++q) r2 += sample[0][q * gg + t];
          centre = middle[t];
          if (GRAD) {
#pragma unroll
            for (int s = 0; s < APX_NSLOT; ++s) {
              gs[s] = 0.0f;
              for (int q = 0; q < slices; ++q) gs[s] += sample[1 + s][q * gg + t];
            }
          }
        }
        if (cp.max_depth > 2) deeper = refine(x2, y2, r2, centre);
        if (!deeper) {
          acc[0] = (double)r2;
          if (GRAD) {
#pragma unroll
            for (int s = 0; s < APX_NSLOT; ++s) acc[1 + s] = (double)gs[s];
          }
        }
      }
      const uint64_t flags = __ballot(deeper);
      if (deeper) {
        const int at = (int)__popcll(flags & ((lane == 0) ? 0ull : (~0ull >> (64 - lane))));
        sx[at] = x2;
        sy[at] = y2;
      }
      if (t == 0) nflag = (int)__popcll(flags);
    }
    __syncthreads();
    level3(sx, sy, nflag, acc);
    if (MODE == Q_VJP) {
      const double wb = (double)B[pix];
#pragma unroll
      for (int s = 0; s < APX_NSLOT; ++s) adj[s] += wb * acc[1 + s];
    } else {
#pragma unroll
      for (int s = 0; s < NV; ++s) {
        const double a = wave_sum(acc[s]);
        if (lane == 0) red[wv][s] = a;
      }
      __syncthreads();
      if (t < cp.nchan && (GRAD || t == 0)) {
        const int s = t == 0 ? 0 : 1 + cp.chan_slot[t];
        const double a = red[0][s] + red[1][s] + red[2][s] + red[3][s];
        planes[t * npix + pix] = (float)(t == 0 ? a : a * cp.dvdr[s - 1]);
      }
    }
    __syncthreads();  // the next pixel writes sample, sx, sy and red again
  }
  if (MODE == Q_VJP) vjp_part(cp, adj, ws.vpart + 8 * (voff + blockIdx.x));
}

// Adjoint of the render: sum over working pixels of B[q] * d deep[q] / d slot
// for the slots chan_slot[1 .. nchan-1].  Unselected pixels use the float32
// analytic partials (what the Jacobian channels hold); selected pixels
// recompute the forward quadrature (the level-1 and deep passes).
__global__ __launch_bounds__(256) void render_vjp_kernel(apx_component cp, RenderConst rc,
                                                         const float* __restrict__ B, RenderWs ws,
                                                         int use_flags) {
  __shared__ double red[4][8];
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const int64_t pix = (int64_t)blockIdx.x * kInitBlock + threadIdx.x;
  double acc[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) acc[c] = 0.0;
  if (pix < npix && !(use_flags && ws.flags[pix])) {
    const Prof<float>& p = rc.f;
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

// Lanes a pixel of the level-1 pass whose terms a butterfly adds; 0: nn lanes, added
// in node order by nn lane reads a channel.  The reads take 20 instructions a pixel
// and channel for the 3 x 3 rule (7 pixels a wave) and 784 for 7 x 7, a butterfly 5
// to 18.  512^2, tolerance 1e-4, Jacobian without the deeper levels: 5 x 5 nodes by
// lane reads 229 us, so 73; 7 x 7 751 and 119.
int level1_row(int nn) { return nn <= 9 ? 0 : nn <= 16 ? 16 : nn <= 32 ? 32 : 64; }

// workgroups of the two passes over npix pixels: no more than could find work
int level_blocks(const apx_component& cp, int64_t npix) {
  const int nn = cp.quad_level * cp.quad_level, row = level1_row(nn);
  const int per = 4 * (64 / (row ? row : nn));
  return (int)std::min<int64_t>(kLevelBlocks, (npix + per - 1) / per);
}
int deep_blocks(const apx_component& cp, int64_t npix) {
  return cp.max_depth < 2 ? 0 : (int)std::min<int64_t>(kDeepBlocks, npix);
}

// the level-1 and deep passes of a component
template <int MODE>
void integrate(const apx_component& cp, const RenderConst& rc, float* planes, const float* B, const RenderWs& ws,
               hipStream_t stream) {
  const int64_t npix = (int64_t)cp.nx * cp.ny;
  const int nl = level_blocks(cp, npix), nd = deep_blocks(cp, npix);
#define APX_LEVEL1(ROW) \
  hipLaunchKernelGGL((render_level1_kernel<MODE, ROW>), dim3(nl), dim3(256), 0, stream, cp, rc, planes, B, ws)
  switch (level1_row(cp.quad_level * cp.quad_level)) {
    case 64: APX_LEVEL1(64); break;
    case 32: APX_LEVEL1(32); break;
    case 16: APX_LEVEL1(16); break;
    default: APX_LEVEL1(0);
  }
#undef APX_LEVEL1
  if (nd == 0) return;
  if (cp.quad_level == 3 && cp.gridding == 5)
    hipLaunchKernelGGL((render_deep_kernel<MODE, true>), dim3(nd), dim3(256), 0, stream, cp, rc, planes, B, ws, nl);
  else
    hipLaunchKernelGGL((render_deep_kernel<MODE, false>), dim3(nd), dim3(256), 0, stream, cp, rc, planes, B, ws, nl);
}

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
         align256(npix) + align256(8 * 8 * (kLevelBlocks + kDeepBlocks));
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
  const RenderConst rc = render_const(cp);
  if (grad)
    hipLaunchKernelGGL(render_init_kernel<true>, dim3((unsigned)nb), dim3(kInitBlock), 0, stream,
                       cp, rc, planes, ws);
  else
    hipLaunchKernelGGL(render_init_kernel<false>, dim3((unsigned)nb), dim3(kInitBlock), 0, stream,
                       cp, rc, planes, ws);
  if (cp.integrate) {
    if (cp.mean_reference)
      hipLaunchKernelGGL(mean_reference_kernel, dim3(1), dim3(256), 0, stream, ws, nb, npix);
    hipLaunchKernelGGL(render_select_kernel, dim3((unsigned)((npix + 255) / 256)), dim3(256), 0,
                       stream, cp, rc, planes, ws);
    if (grad) integrate<Q_GRAD>(cp, rc, planes, nullptr, ws, stream);
    else integrate<Q_VALUE>(cp, rc, planes, nullptr, ws, stream);
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
  const RenderConst rcst = render_const(cp);
  hipLaunchKernelGGL(render_vjp_kernel, dim3((unsigned)nb), dim3(kInitBlock), 0, stream, cp, rcst, weights,
                     ws, cp.integrate);
  int nb2 = 0;
  if (cp.integrate) {
    nb2 = level_blocks(cp, npix) + deep_blocks(cp, npix);  // the value render left the lists
    integrate<Q_VJP>(cp, rcst, nullptr, weights, ws, stream);
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
