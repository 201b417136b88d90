// Pixel reductions that feed Levenberg-Marquardt (fit/lm.py:373-406):
//   chi2             sum W (Y - m)^2 over unmasked pixels    (_chi2)
//   normal_equations J^T W J and -J^T W (m - Y)                (_hess, _grad)
//   rpp              J^T ((2/d)(W (m1 - m0)/d - W J h))         (_rpp)
// Each is a grid-stride pass that writes one float64 partial per workgroup,
// then a single-workgroup pass sums the partials in a fixed order, so repeated
// runs give identical bits.  J^T W J uses the gfx950 matrix cores
// (v_mfma_f32_16x16x4_f32: 4 pixels x 16 parameters per instruction, FP32
// accumulate, flushed to float64 every 64 instructions).
#include <hip/hip_runtime.h>

#include <mutex>

#include "capi_internal.h"
#include "wave.h"

namespace apx {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kBlocks = 512;
constexpr int kMaxNp = 16;

__host__ __device__ inline int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }

__global__ __launch_bounds__(256) void chi2_partial_kernel(const float* __restrict__ model,
                                                           const float* __restrict__ data,
                                                           const float* __restrict__ weight,
                                                           const uint8_t* __restrict__ mask,
                                                           int64_t npix, double* partial) {
  __shared__ double red[4];
  double acc = 0.0;
  for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < npix;
       p += (int64_t)gridDim.x * 256) {
    if (mask && mask[p]) continue;
    const double d = (double)data[p] - (double)model[p];
    acc += (weight ? (double)weight[p] : 1.0) * d * d;
  }
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// out[k] = sum_b partial[b * stride + k] for k < n, one wave an output: 64
// partials in flight a step and the lanes' sums folded in a fixed order.  A
// thread an output read its up to 512 partials one after another: 81 us each
// for chi2 and rpp, now 4.7 us.
__device__ __forceinline__ double partial_sum(const double* __restrict__ partial, int nblocks, int stride, int k) {
  double t = 0.0;
  for (int b = threadIdx.x & 63; b < nblocks; b += 64) t += partial[(int64_t)b * stride + k];
  return wave_sum(t);
}

__global__ __launch_bounds__(256) void sum_partials_kernel(const double* __restrict__ partial, int nblocks,
                                                           int stride, int n, double* out,
                                                           double scale) {
  const int k = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (k >= n) return;
  const double t = partial_sum(partial, nblocks, stride, k);
  if ((threadIdx.x & 63) == 0) out[k] = t * scale;
}

// J^T W J and J^T W (Y - m): one 16x16x4 MFMA per 4 pixels per wavefront.
// Lane l holds parameter r = l % 16 of pixel base + l / 16:
//   A[r][k] = J[p_k][r], B[k][c] = W_p J[p_k][c], D[4(l/16)+i][l%16] (reg i).
// Bound by HBM (J, model, data and weight read once).  A wave has the loads of
// kStep steps in flight: with one step's it waited out a memory round trip
// every 4 pixels, 308 us for 2048^2 x 13 (268 MB); with 8 steps' 102 us, with 16 97.
constexpr int kStep = 16;  // divides 64, the steps between two flushes
__global__ __launch_bounds__(256) void normal_eq_kernel(const float* __restrict__ J,
                                                        const float* __restrict__ model,
                                                        const float* __restrict__ data,
                                                        const float* __restrict__ weight,
                                                        const uint8_t* __restrict__ mask,
                                                        int64_t npix, int np, double* partial) {
  __shared__ double redH[4][256];
  __shared__ double redg[4][16];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int r = lane & 15, k = lane >> 4;
  const int64_t gwave = (int64_t)blockIdx.x * 4 + wv;
  const int64_t nwave = (int64_t)gridDim.x * 4;
  v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
  double accd[4] = {0.0, 0.0, 0.0, 0.0};
  double gacc = 0.0;
  float gpart = 0.0f;
  int since = 0;
  for (int64_t base = gwave * 4; base < npix; base += kStep * nwave * 4) {
    // the loads of kStep steps (unconditional, at pixel 0 and column 0 where
    // there is nothing to read, so that none waits for another), then their
    // products in step order; what is not kept is zero and adds nothing
    float a[kStep], w[kStep], res[kStep], y[kStep], m[kStep];
    uint8_t drop[kStep];
#pragma unroll
    for (int u = 0; u < kStep; ++u) {
      const int64_t p = base + u * nwave * 4 + k, q = p < npix ? p : 0;
      drop[u] = mask ? mask[q] : (uint8_t)0;
      a[u] = J[q * np + (r < np ? r : 0)];
      w[u] = weight ? weight[q] : 1.0f;
      y[u] = data[q];
      m[u] = model[q];
    }
#pragma unroll
    for (int u = 0; u < kStep; ++u) {
      const bool keep = base + u * nwave * 4 + k < npix && r < np && !drop[u];
      a[u] = keep ? a[u] : 0.0f;
      w[u] = keep ? w[u] : 0.0f;
      res[u] = keep ? y[u] - m[u] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kStep; ++u) {
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], w[u] * a[u], acc, 0, 0, 0);
      gpart = fmaf(a[u] * w[u], res[u], gpart);
    }
    since += kStep;
    if (since == 64) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        accd[i] += (double)acc[i];
        acc[i] = 0.0f;
      }
      gacc += (double)gpart;
      gpart = 0.0f;
      since = 0;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) accd[i] += (double)acc[i];
  gacc += (double)gpart;
  // H element of (lane, reg i): row 4*(lane/16)+i, col lane%16
#pragma unroll
  for (int i = 0; i < 4; ++i) redH[wv][(4 * (lane >> 4) + i) * 16 + (lane & 15)] = accd[i];
  gacc += __shfl_xor(gacc, 16, 64);
  gacc += __shfl_xor(gacc, 32, 64);
  if (lane < 16) redg[wv][lane] = gacc;
  __syncthreads();
  const int stride = kMaxNp * kMaxNp + kMaxNp;
  double* out = partial + (int64_t)blockIdx.x * stride;
  for (int e = threadIdx.x; e < 256; e += 256)
    out[e] = redH[0][e] + redH[1][e] + redH[2][e] + redH[3][e];
  if (threadIdx.x < 16)
    out[256 + threadIdx.x] = redg[0][threadIdx.x] + redg[1][threadIdx.x] + redg[2][threadIdx.x] +
                             redg[3][threadIdx.x];
}

// unpack 16x16 padded partial sums into np x np hess and np grad (one wave an
// entry, as sum_partials_kernel; 125 us with a thread an entry, 4.8 us now)
__global__ __launch_bounds__(256) void normal_eq_final_kernel(const double* __restrict__ partial, int nblocks,
                                                              int np, double* hess, double* grad) {
  const int stride = kMaxNp * kMaxNp + kMaxNp;
  const int e = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (e >= np * np + np) return;
  const double t = partial_sum(partial, nblocks, stride, e < np * np ? (e / np) * kMaxNp + (e % np) : 256 + (e - np * np));
  if ((threadIdx.x & 63) == 0) {
    if (e < np * np)
      hess[e] = t;
    else
      grad[e - np * np] = t;
  }
}

// One pixel a thread, 256 pixels a workgroup step.  Their rows of J are one
// contiguous run: it is read coalesced, a float a thread at a time, and passed
// through LDS, and the next step's run is requested before this one's sums.
// Bound by HBM.  Each thread reading its own row (13 floats, 52 bytes apart
// from its neighbour's) took 116 us for 2048^2 x 13, this 86 us.
__global__ __launch_bounds__(256) void rpp_kernel(const float* __restrict__ J,
                                                  const float* __restrict__ m0,
                                                  const float* __restrict__ m1,
                                                  const float* __restrict__ weight,
                                                  const uint8_t* __restrict__ mask, int64_t npix,
                                                  int np, const double* __restrict__ h, double d,
                                                  double* partial) {
  __shared__ float rows[256 * kMaxNp];
  __shared__ double red[4][kMaxNp];
  const int t = threadIdx.x;
  double hv[kMaxNp], acc[kMaxNp];
#pragma unroll
  for (int r = 0; r < kMaxNp; ++r) {
    hv[r] = r < np ? h[r] : 0.0;
    acc[r] = 0.0;
  }
  const int64_t step = (int64_t)gridDim.x * 256, total = npix * np;
  float next[kMaxNp];  // floats t, t + 256, ... of the step's run
  auto request = [&](int64_t base) {
#pragma unroll
    for (int r = 0; r < kMaxNp; ++r) {
      const int64_t e = base * np + r * 256 + t;
      next[r] = (r < np && e < total) ? J[e] : 0.0f;
    }
  };
  request((int64_t)blockIdx.x * 256);
  for (int64_t base = (int64_t)blockIdx.x * 256; base < npix; base += step) {
    __syncthreads();  // the previous step's rows are read
#pragma unroll
    for (int r = 0; r < kMaxNp; ++r)
      if (r < np) rows[r * 256 + t] = next[r];
    __syncthreads();
    if (base + step < npix) request(base + step);
    const int64_t p = base + t;
    if (p >= npix || (mask && mask[p])) continue;
    float jr[kMaxNp];
    double jh = 0.0;
#pragma unroll
    for (int r = 0; r < kMaxNp; ++r) {
      jr[r] = r < np ? rows[t * np + r] : 0.0f;
      jh += (double)jr[r] * hv[r];
    }
    const double w = weight ? (double)weight[p] : 1.0;
    const double v = (2.0 / d) * (w * (double)(m1[p] - m0[p]) / d - w * jh);
#pragma unroll
    for (int r = 0; r < kMaxNp; ++r) acc[r] += (double)jr[r] * v;
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int r = 0; r < kMaxNp; ++r) {
    const double s = wave_sum(acc[r]);
    if (lane == 0) red[wv][r] = s;
  }
  __syncthreads();
  if (threadIdx.x < kMaxNp)
    partial[(int64_t)blockIdx.x * kMaxNp + threadIdx.x] =
        red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
}

int nblocks_for(int64_t npix) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(kBlocks, (npix + 1023) / 1024));
}

}  // namespace

// Partial sums of normal_equations_noalloc: one (16 x 16 + 16) float64 block
// per workgroup, at most kBlocks workgroups (1,114,112 bytes).  Each GPU the
// library runs on holds its own copy until the process ends.  Host code never
// names this array: its per-device address comes from hipGetSymbolAddress.
constexpr int64_t kScratchBytes = 8 * (int64_t)kBlocks * (kMaxNp * kMaxNp + kMaxNp);
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up once per
// device (with that device current) and kept.
int scratch_address(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess)
    return set_error(APX_E_HIP, "normal_equations_noalloc: hipGetDevice failed");
  if (dev < 0 || dev >= kMaxDevices)
    return set_error(APX_E_LIMIT, "normal_equations_noalloc: device index beyond 63");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_error(APX_E_HIP, "normal_equations_noalloc: hipGetSymbolAddress(scratch) failed");
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return APX_OK;
}

}  // namespace

int64_t reduce_workspace_bytes(int64_t npix, int32_t np) {
  (void)np;
  return align256(8 * (int64_t)kBlocks * (kMaxNp * kMaxNp + kMaxNp));
}

int chi2(const float* model, const float* data, const float* weight, const uint8_t* mask,
         int64_t npix, double* out, void* ws, int64_t ws_bytes, hipStream_t stream) {
  if (!model || !data || !out || !ws) return set_error(APX_E_INVALID, "chi2: null pointer");
  if (npix < 0) return set_error(APX_E_INVALID, "chi2: negative size");
  if (ws_bytes < reduce_workspace_bytes(npix, 1))
    return set_error(APX_E_INVALID, "chi2: workspace too small");
  const int nb = nblocks_for(npix);
  double* partial = static_cast<double*>(ws);
  hipLaunchKernelGGL(chi2_partial_kernel, dim3(nb), dim3(256), 0, stream, model, data, weight,
                     mask, npix, partial);
  hipLaunchKernelGGL(sum_partials_kernel, dim3(1), dim3(256), 0, stream, partial, nb, 1, 1, out,
                     1.0);
  return check_launch("chi2");
}

int normal_equations(const float* J, const float* model, const float* data, const float* weight,
                     const uint8_t* mask, int64_t npix, int32_t np, double* hess, double* grad,
                     void* ws, int64_t ws_bytes, hipStream_t stream) {
  if (!J || !model || !data || !hess || !grad || !ws)
    return set_error(APX_E_INVALID, "normal_equations: null pointer");
  if (np < 1 || np > kMaxNp) return set_error(APX_E_LIMIT, "normal_equations: np must be 1..16");
  if (ws_bytes < reduce_workspace_bytes(npix, np))
    return set_error(APX_E_INVALID, "normal_equations: workspace too small");
  const int nb = nblocks_for(npix);
  double* partial = static_cast<double*>(ws);
  hipLaunchKernelGGL(normal_eq_kernel, dim3(nb), dim3(256), 0, stream, J, model, data, weight,
                     mask, npix, np, partial);
  hipLaunchKernelGGL(normal_eq_final_kernel, dim3((np * np + np + 3) / 4), dim3(256), 0, stream, partial, nb, np, hess,
                     grad);
  return check_launch("normal_equations");
}

int rpp(const float* J, const float* m0, const float* m1, const float* weight, const uint8_t* mask,
        int64_t npix, int32_t np, const double* h, double d, double* out, void* ws,
        int64_t ws_bytes, hipStream_t stream) {
  if (!J || !m0 || !m1 || !h || !out || !ws) return set_error(APX_E_INVALID, "rpp: null pointer");
  if (np < 1 || np > kMaxNp) return set_error(APX_E_LIMIT, "rpp: np must be 1..16");
  if (ws_bytes < reduce_workspace_bytes(npix, np))
    return set_error(APX_E_INVALID, "rpp: workspace too small");
  const int nb = nblocks_for(npix);
  double* partial = static_cast<double*>(ws);
  hipLaunchKernelGGL(rpp_kernel, dim3(nb), dim3(256), 0, stream, J, m0, m1, weight, mask, npix, np,
                     h, d, partial);
  hipLaunchKernelGGL(sum_partials_kernel, dim3((np + 3) / 4), dim3(256), 0, stream, partial, nb, kMaxNp, np,
                     out, 1.0);
  return check_launch("rpp");
}

int normal_equations_noalloc(const float* J, const float* model, const float* data,
                             const float* weight, const uint8_t* mask, int64_t npix, int32_t np,
                             double* hess, double* grad, hipStream_t stream) {
  if (!J || !model || !data || !hess || !grad)
    return set_error(APX_E_INVALID, "normal_equations_noalloc: null pointer");
  if (npix < 0) return set_error(APX_E_INVALID, "normal_equations_noalloc: negative size");
  if (np < 1 || np > kMaxNp)
    return set_error(APX_E_LIMIT, "normal_equations_noalloc: np must be 1..16");
  const int nb = nblocks_for(npix);
  // the partial sums of nb workgroups must fit the static scratch (they always
  // do: nb <= kBlocks for every npix)
  if (8 * (int64_t)nb * (kMaxNp * kMaxNp + kMaxNp) > kScratchBytes)
    return set_error(APX_E_LIMIT, "normal_equations_noalloc: partial sums exceed the 1,114,112-byte scratch");
  void* ws = nullptr;
  const int rc = scratch_address(&ws);
  if (rc != APX_OK) return rc;
  double* partial = static_cast<double*>(ws);
  // every workgroup overwrites its whole partial block, so nothing is cleared
  hipLaunchKernelGGL(normal_eq_kernel, dim3(nb), dim3(256), 0, stream, J, model, data, weight,
                     mask, npix, np, partial);
  hipLaunchKernelGGL(normal_eq_final_kernel, dim3((np * np + np + 3) / 4), dim3(256), 0, stream, partial, nb, np, hess,
                     grad);
  return check_launch("normal_equations_noalloc");
}

}  // namespace apx
