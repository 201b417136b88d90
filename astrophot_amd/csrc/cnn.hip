// The learned initialiser's network on gfx950: a BF16 MFMA GEMM (float32
// accumulate) with a bias / ReLU epilogue, and the small kernels around it
// that make convolutions, their gradients and an Adam step out of GEMMs.
//
// Layout: activations NHWC (row = one output pixel of one cutout, column =
// channel), so a 3x3 / stride-2 / pad-1 convolution is
//   Y[M = B*Ho*Wo, Cout] = im2col(X)[M, Kp] * W[Kp, Cout]      (K = 9 Cin)
// with K ordered (ky, kx, ci) and zero-padded to a multiple of 32; its
// gradients are
//   dW = im2col(X)^T dZ,   dcol = dZ W^T,   dX = col2im(dcol)  (a gather).
// Bf16 values are stored as uint16 (round to nearest even from float32).
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "capi_internal.h"

namespace apx {

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint16_t to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// ---------------------------------------------------------------------------
// C[M, N] = A[M, K] B[K, N] (+ bias[N], ReLU), bf16 in, float32 accumulate.
// Element (m, k) of A at A[m * sam + k * sak]; (k, n) of B at B[k * sbk + n * sbn]
// (so a transposed operand is a stride swap).  Workgroup tile 64 x 64,
// k-step 32, 4 waves of 32 x 32 (2 x 2 MFMA 16x16x32 blocks).  MFMA lane
// layout: A row l % 16, k 8 (l / 16) .. + 7; B column l % 16, same k;
// D[4 (l / 16) + r][l % 16] in acc[r].
constexpr int BM = 64, BN = 64, BK = 32, LDK = BK + 8;  // LDS row pitch (bf16), padded

// Implicit im2col operand of a 3x3 / stride-2 / pad-1 convolution over X
// (B, H, W, Cin) NHWC bf16: row m = (b, oy, ox), column k = (ky * 3 + kx) *
// Cin + ci, zero beyond 9 Cin and outside the image.
struct ConvA {
  const uint16_t* X;
  int H, W, Cin, Ho, Wo;
};

// How an operand tile is read (OP_CONV: A only).  Every form brings 8 values a
// thread as one uint4, so that the next k-step's tile is in registers while the
// current one is multiplied:
//   OP_ANY    8 separate 2-byte loads along k: any strides, any alignment
//   OP_KROW   k contiguous: one 16-byte load of 8 k of a row (row pitch and
//             depth multiples of 8, base on 16 bytes)
//   OP_RROW   rows contiguous: one 16-byte load of 8 rows at one k, stored
//             transposed (row count and k pitch multiples of 8, base on 16 bytes)
// A training step on 256 cutouts spent 1.56 ms in its 17 GEMMs reading 2 bytes
// a load with nothing in flight across a k-step; see launch_gemm.
enum : int { OP_ANY = 0, OP_KROW = 1, OP_RROW = 2, OP_CONV = 3 };

// this thread's 8 values of the 64-row x BK tile at (r0, k0) of an R x K operand
template <int OP>
__device__ __forceinline__ uint4 load_operand(const uint16_t* X, int64_t sr, int64_t sk, int R, int kend, int r0, int k0) {
  if (OP == OP_RROW) {
    const int r = r0 + 8 * (threadIdx.x & 7), k = k0 + (threadIdx.x >> 3);
    return r < R && k < kend ? *reinterpret_cast<const uint4*>(X + (int64_t)k * sk + r) : make_uint4(0u, 0u, 0u, 0u);
  }
  const int r = r0 + (threadIdx.x >> 2), k = k0 + 8 * (threadIdx.x & 3);
  if (OP == OP_KROW)
    return r < R && k < kend ? *reinterpret_cast<const uint4*>(X + (int64_t)r * sr + k) : make_uint4(0u, 0u, 0u, 0u);
  uint16_t e[8];
#pragma unroll
  for (int q = 0; q < 8; ++q)
    e[q] = (r < R && k + q < kend) ? X[(int64_t)r * sr + (int64_t)(k + q) * sk] : (uint16_t)0;
  return make_uint4((uint32_t)e[0] | ((uint32_t)e[1] << 16), (uint32_t)e[2] | ((uint32_t)e[3] << 16),
                    (uint32_t)e[4] | ((uint32_t)e[5] << 16), (uint32_t)e[6] | ((uint32_t)e[7] << 16));
}

// the loaded values into the tile T[row][k]
template <int OP>
__device__ __forceinline__ void store_operand(uint16_t* T, uint4 v) {
  if (OP == OP_RROW) {
    uint16_t* o = T + 8 * (threadIdx.x & 7) * LDK + (threadIdx.x >> 3);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      o[(2 * q) * LDK] = (uint16_t)w[q];
      o[(2 * q + 1) * LDK] = (uint16_t)(w[q] >> 16);
    }
  } else {
    *reinterpret_cast<uint4*>(T + (threadIdx.x >> 2) * LDK + 8 * (threadIdx.x & 3)) = v;
  }
}

// this thread's 8 values of the implicit im2col row (b, oy, ox)
__device__ __forceinline__ uint4 load_patch(const ConvA& cv, bool in, int cb, int coy, int cox, int k, int kend) {
  uint4 v = make_uint4(0u, 0u, 0u, 0u);
  if (!in || k >= kend) return v;
  if ((cv.Cin & 7) == 0) {
    // 8 consecutive channels of one tap: one 16-byte load
    const int tap = k / cv.Cin, ci = k - tap * cv.Cin;
    const int iy = 2 * coy + tap / 3 - 1, ix = 2 * cox + tap % 3 - 1;
    if (tap < 9 && iy >= 0 && iy < cv.H && ix >= 0 && ix < cv.W)
      v = *reinterpret_cast<const uint4*>(cv.X + (((int64_t)cb * cv.H + iy) * cv.W + ix) * cv.Cin + ci);
    return v;
  }
  uint16_t e[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int kq = k + q, tap = kq / cv.Cin, ci = kq - tap * cv.Cin;
    const int iy = 2 * coy + tap / 3 - 1, ix = 2 * cox + tap % 3 - 1;
    e[q] = (kq < kend && tap < 9 && iy >= 0 && iy < cv.H && ix >= 0 && ix < cv.W)
               ? cv.X[(((int64_t)cb * cv.H + iy) * cv.W + ix) * cv.Cin + ci]
               : (uint16_t)0;
  }
  return make_uint4((uint32_t)e[0] | ((uint32_t)e[1] << 16), (uint32_t)e[2] | ((uint32_t)e[3] << 16),
                    (uint32_t)e[4] | ((uint32_t)e[5] << 16), (uint32_t)e[6] | ((uint32_t)e[7] << 16));
}

template <int AOP, int BOP>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(int M, int N, int K, const uint16_t* A,
                                                        int64_t sam, int64_t sak, const uint16_t* B,
                                                        int64_t sbk, int64_t sbn, float* C,
                                                        int64_t ldc, const float* bias, int relu,
                                                        uint16_t* Cb, int accumulate, float* P,
                                                        int kchunk, ConvA cv) {
  __shared__ __attribute__((aligned(16))) uint16_t As[BM * LDK];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[BN * LDK];  // Bs[n][k]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = w >> 1, wn = w & 1;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
  v4f acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
  const int kbeg = blockIdx.z * kchunk, kend = min(K, kbeg + kchunk);
  // OP_CONV: the output pixel of this thread's A row
  const int sr = threadIdx.x >> 2, sk = (threadIdx.x & 3) * 8;
  int cb = 0, coy = 0, cox = 0;
  if (AOP == OP_CONV && m0 + sr < M) {
    const int m = m0 + sr;
    cox = m % cv.Wo;
    coy = (m / cv.Wo) % cv.Ho;
    cb = m / (cv.Wo * cv.Ho);
  }
  auto load_a = [&](int k0) {
    if constexpr (AOP == OP_CONV) return load_patch(cv, m0 + sr < M, cb, coy, cox, k0 + sk, kend);
    else return load_operand<AOP>(A, sam, sak, M, kend, m0, k0);
  };
  uint4 va = load_a(kbeg), vb = load_operand<BOP>(B, sbn, sbk, N, kend, n0, kbeg);
  for (int k0 = kbeg; k0 < kend; k0 += BK) {
    __syncthreads();
    store_operand<AOP>(As, va);
    store_operand<BOP>(Bs, vb);
    __syncthreads();
    if (k0 + BK < kend) {  // the next tile arrives during this one's products
      va = load_a(k0 + BK);
      vb = load_operand<BOP>(B, sbn, sbk, N, kend, n0, k0 + BK);
    }
    const int kq = (lane >> 4) * 8;
    v8bf a[2], bb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = wm * 32 + i * 16 + (lane & 15);
      a[i] = *reinterpret_cast<const v8bf*>(&As[r * LDK + kq]);
      const int c = wn * 32 + i * 16 + (lane & 15);
      bb[i] = *reinterpret_cast<const v8bf*>(&Bs[c * LDK + kq]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], bb[j], acc[i][j], 0, 0, 0);
  }
  // epilogue
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm * 32 + i * 16 + (lane >> 4) * 4 + r;
        const int n = n0 + wn * 32 + j * 16 + (lane & 15);
        if (m >= M || n >= N) continue;
        float v = acc[i][j][r];
        if (P) {  // split-K partial, summed by splitk_sum_kernel
          P[((int64_t)blockIdx.z * M + m) * N + n] = v;
          continue;
        }
        if (accumulate) v += C[(int64_t)m * ldc + n];
        if (bias) v += bias[n];
        if (relu) v = fmaxf(v, 0.0f);
        C[(int64_t)m * ldc + n] = v;
        if (Cb) Cb[(int64_t)m * ldc + n] = to_bf16(v);
      }
}

// C = sum over the split-K partials (in split order) (+ C, bias, ReLU).  Bound by
// latency: a weight gradient has some 10,000 entries and up to 256 partials each,
// so eight partials are loaded ahead of their additions (12.5 -> 5.2 us a layer).
__global__ __launch_bounds__(256) void splitk_sum_kernel(const float* P, int splits, int M, int N,
                                                         float* C, int64_t ldc, const float* bias,
                                                         int relu, uint16_t* Cb, int accumulate) {
  const int64_t total = (int64_t)M * N;
  for (int64_t e = blockIdx.x * 256ll + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
    const int m = (int)(e / N), n = (int)(e % N);
    float v = 0.0f;
    const float* p = P + e;
    int z = 0;
    for (; z + 8 <= splits; z += 8, p += 8 * total) {
      float t[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) t[q] = p[q * total];
#pragma unroll
      for (int q = 0; q < 8; ++q) v += t[q];
    }
    for (; z < splits; ++z, p += total) v += *p;
    if (accumulate) v += C[(int64_t)m * ldc + n];
    if (bias) v += bias[n];
    if (relu) v = fmaxf(v, 0.0f);
    C[(int64_t)m * ldc + n] = v;
    if (Cb) Cb[(int64_t)m * ldc + n] = to_bf16(v);
  }
}

// weighted mean-squared error over B x N outputs: loss[0] = sum_bj w_j (y - t)^2 / B,
// dy = 2 w_j (y - t) / B (one workgroup, fixed summation order)
__global__ __launch_bounds__(256) void mse_kernel(const float* y, const float* t, const float* wj, int Bn,
                                                  int N, float* dy, float* loss) {
  __shared__ float red[4];
  float s = 0.0f;
  for (int e = threadIdx.x; e < Bn * N; e += 256) {
    const float d = y[e] - t[e], w = wj[e % N];
    dy[e] = 2.0f * w * d / (float)Bn;
    s += w * d * d;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) loss[0] = (red[0] + red[1] + red[2] + red[3]) / (float)Bn;
}

// im2col of a 3x3 / stride-2 / pad-1 convolution: X (B, H, W, Cin) bf16 ->
// col (B * Ho * Wo, Kp) bf16, column (ky * 3 + kx) * Cin + ci, zero beyond K
__global__ __launch_bounds__(256) void im2col_kernel(const uint16_t* X, int Bn, int H, int W, int Cin,
                                                     int Kp, uint16_t* col) {
  const int Ho = (H + 1) / 2, Wo = (W + 1) / 2;
  const int64_t total = (int64_t)Bn * Ho * Wo * Kp;
  for (int64_t e = blockIdx.x * 256ll + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
    const int k = (int)(e % Kp);
    const int64_t m = e / Kp;
    uint16_t v = 0;
    if (k < 9 * Cin) {
      const int ci = k % Cin, t = k / Cin, ky = t / 3, kx = t % 3;
      const int ox = (int)(m % Wo), oy = (int)((m / Wo) % Ho), b = (int)(m / ((int64_t)Wo * Ho));
      const int iy = 2 * oy + ky - 1, ix = 2 * ox + kx - 1;
      if (iy >= 0 && iy < H && ix >= 0 && ix < W) v = X[(((int64_t)b * H + iy) * W + ix) * Cin + ci];
    }
    col[e] = v;
  }
}

// im2col_kernel 8 columns a thread: one 16-byte store, and one 16-byte load where
// they are 8 channels of one tap (Cin a multiple of 8).  Bound by the store of
// col; an element a thread spent its time on 64-bit divisions (the four layers of
// 256 cutouts: 128 -> 41 us).
__global__ __launch_bounds__(256) void im2col8_kernel(const uint16_t* __restrict__ X, int H, int W, int Cin, int Kp,
                                                      uint32_t total, uint16_t* __restrict__ col) {
  const int Ho = (H + 1) / 2, Wo = (W + 1) / 2;
  const uint32_t K8 = (uint32_t)Kp / 8;
  for (uint32_t e = blockIdx.x * 256u + threadIdx.x; e < total; e += gridDim.x * 256u) {
    const uint32_t m = e / K8, q = m / (uint32_t)Wo;
    const int k = 8 * (int)(e - m * K8), ox = (int)(m - q * (uint32_t)Wo);
    const uint32_t b = q / (uint32_t)Ho;
    const ConvA cv{X, H, W, Cin, Ho, Wo};
    *reinterpret_cast<uint4*>(col + (int64_t)e * 8) =
        load_patch(cv, true, (int)b, (int)(q - b * (uint32_t)Ho), ox, k, 9 * Cin);
  }
}

// dX (B, H, W, Cin) float32 = col2im(dcol (B * Ho * Wo, Kp)): each input
// element gathers the (oy, ky) x (ox, kx) pairs that read it
__global__ __launch_bounds__(256) void col2im_kernel(const float* dcol, int Bn, int H, int W, int Cin,
                                                     int Kp, float* dX) {
  const int Ho = (H + 1) / 2, Wo = (W + 1) / 2;
  const int64_t total = (int64_t)Bn * H * W * Cin;
  for (int64_t e = blockIdx.x * 256ll + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
    const int ci = (int)(e % Cin);
    const int ix = (int)((e / Cin) % W), iy = (int)((e / ((int64_t)Cin * W)) % H);
    const int b = (int)(e / ((int64_t)Cin * W * H));
    float s = 0.0f;
#pragma unroll
    for (int ky = 0; ky < 3; ++ky) {
      const int ty = iy + 1 - ky;  // = 2 oy
      if (ty < 0 || (ty & 1) || ty / 2 >= Ho) continue;
#pragma unroll
      for (int kx = 0; kx < 3; ++kx) {
        const int tx = ix + 1 - kx;
        if (tx < 0 || (tx & 1) || tx / 2 >= Wo) continue;
        const int64_t m = ((int64_t)b * Ho + ty / 2) * Wo + tx / 2;
        s += dcol[m * Kp + (ky * 3 + kx) * Cin + ci];
      }
    }
    dX[e] = s;
  }
}

// col2im_kernel 4 channels a thread (16-byte loads, 32-bit divisions): the three
// layers of 256 cutouts 83 -> 32 us
__global__ __launch_bounds__(256) void col2im4_kernel(const float* __restrict__ dcol, int H, int W, int Cin, int Kp,
                                                      uint32_t total, float* __restrict__ dX) {
  const int Ho = (H + 1) / 2, Wo = (W + 1) / 2;
  const uint32_t C4 = (uint32_t)Cin / 4;
  for (uint32_t e = blockIdx.x * 256u + threadIdx.x; e < total; e += gridDim.x * 256u) {
    const uint32_t pix = e / C4, q = pix / (uint32_t)W, b = q / (uint32_t)H;
    const int ci = 4 * (int)(e - pix * C4), ix = (int)(pix - q * (uint32_t)W), iy = (int)(q - b * (uint32_t)H);
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int ky = 0; ky < 3; ++ky) {
      const int ty = iy + 1 - ky;  // = 2 oy
      if (ty < 0 || (ty & 1) || ty / 2 >= Ho) continue;
#pragma unroll
      for (int kx = 0; kx < 3; ++kx) {
        const int tx = ix + 1 - kx;
        if (tx < 0 || (tx & 1) || tx / 2 >= Wo) continue;
        const int64_t m = ((int64_t)b * Ho + ty / 2) * Wo + tx / 2;
        const float4 v = *reinterpret_cast<const float4*>(dcol + m * Kp + (ky * 3 + kx) * Cin + ci);
        s.x += v.x;
        s.y += v.y;
        s.z += v.z;
        s.w += v.w;
      }
    }
    *reinterpret_cast<float4*>(dX + (int64_t)e * 4) = s;
  }
}

// dst = bf16(src * (mask > 0)) (mask null: no ReLU gate)
__global__ __launch_bounds__(256) void cast_gate_kernel(const float* src, const float* mask, int64_t n,
                                                        uint16_t* dst, float* dstf) {
  for (int64_t e = blockIdx.x * 256ll + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
    float v = src[e];
    if (mask && !(mask[e] > 0.0f)) v = 0.0f;
    if (dstf) dstf[e] = v;
    dst[e] = to_bf16(v);
  }
}

// column sums of X (M, N) float32 into out (N): the bias gradient
__global__ __launch_bounds__(256) void colsum_kernel(const float* X, int M, int N, float* out) {
  __shared__ float red[4][64];
  const int n = blockIdx.x * 64 + (threadIdx.x & 63), part = threadIdx.x >> 6;
  float s = 0.0f;
  if (n < N)
    for (int m = part; m < M; m += 4) s += X[(int64_t)m * N + n];
  red[part][threadIdx.x & 63] = s;
  __syncthreads();
  if (part == 0 && n < N) out[n] = red[0][threadIdx.x] + red[1][threadIdx.x] + red[2][threadIdx.x] + red[3][threadIdx.x];
}

// The ReLU gate, the bf16 copy and the bias gradient of one layer in one pass:
// dst = bf16(v), v = src * (mask > 0), and per workgroup the column sums of v
// (M, N) into P[blockIdx.x][N]; column_final_kernel adds the workgroups'.
// Bound by HBM: 4 B (8 with a mask) read and 2 B written an element.  It stands
// in for a gate pass that also wrote v in float32 and a column sum of that copy
// on one workgroup per 64 columns, whose rows were read one after another: the
// six layers of a training step on 256 cutouts took 21.05 ms, and take 64 us
// (43 here, 20 in column_final_kernel).
// VEC: 4 consecutive columns a thread (16-byte loads); a workgroup covers
// 1024 / N whole rows a step, so a thread's columns never change.  Else: 64
// columns (blockIdx.y) x 4 rows a step, for any N.
template <bool VEC>
__global__ __launch_bounds__(256) void gate_colsum_kernel(const float* __restrict__ src, const float* __restrict__ mask,
                                                          int M, int N, uint16_t* __restrict__ dst, float* __restrict__ P) {
  __shared__ float red[1024];
  const int t = threadIdx.x;
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (VEC) {
    const int per = N >> 2;                // threads a row
    const int R = 256 / per, r0 = t / per; // rows a step, this thread's row in it
    const int64_t step = (int64_t)gridDim.x * R;
    const int c = 4 * (t - r0 * per);
    auto one = [&](int64_t m, float4 v, float4 g) {
      if (mask) {
        v.x = g.x > 0.0f ? v.x : 0.0f;
        v.y = g.y > 0.0f ? v.y : 0.0f;
        v.z = g.z > 0.0f ? v.z : 0.0f;
        v.w = g.w > 0.0f ? v.w : 0.0f;
      }
      s[0] += v.x;
      s[1] += v.y;
      s[2] += v.z;
      s[3] += v.w;
      ushort4 o;
      o.x = to_bf16(v.x);
      o.y = to_bf16(v.y);
      o.z = to_bf16(v.z);
      o.w = to_bf16(v.w);
      *reinterpret_cast<ushort4*>(dst + m * N + c) = o;
    };
    int64_t m = (int64_t)blockIdx.x * R + r0;
    const float4 none = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (; m + 3 * step < M; m += 4 * step) {  // 4 rows' loads in flight
      float4 v[4], g[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] = *reinterpret_cast<const float4*>(src + (m + q * step) * N + c);
        g[q] = mask ? *reinterpret_cast<const float4*>(mask + (m + q * step) * N + c) : none;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) one(m + q * step, v[q], g[q]);
    }
    for (; m < M; m += step)
      one(m, *reinterpret_cast<const float4*>(src + m * N + c),
          mask ? *reinterpret_cast<const float4*>(mask + m * N + c) : none);
    *reinterpret_cast<float4*>(red + 4 * t) = make_float4(s[0], s[1], s[2], s[3]);  // [row of the step][column]
    __syncthreads();
    for (int n = t; n < N; n += 256) {
      float a = 0.0f;
      for (int r = 0; r < R; ++r) a += red[r * N + n];
      P[(int64_t)blockIdx.x * N + n] = a;
    }
  } else {
    const int n = blockIdx.y * 64 + (t & 63), part = t >> 6;
    if (n < N)
      for (int64_t m = (int64_t)blockIdx.x * 4 + part; m < M; m += (int64_t)gridDim.x * 4) {
        float v = src[m * N + n];
        if (mask && !(mask[m * N + n] > 0.0f)) v = 0.0f;
        s[0] += v;
        dst[m * N + n] = to_bf16(v);
      }
    red[t] = s[0];
    __syncthreads();
    if (part == 0 && n < N) P[(int64_t)blockIdx.x * N + n] = red[t] + red[64 + t] + red[128 + t] + red[192 + t];
  }
}

// out[n] = sum of P[b][n] over b < nb, one wave a column
__global__ __launch_bounds__(256) void column_final_kernel(const float* __restrict__ P, int nb, int N, float* __restrict__ out) {
  const int n = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= N) return;
  float s = 0.0f;
  for (int b = lane; b < nb; b += 64) s += P[(int64_t)b * N + n];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) out[n] = s;
}

// Adam (Kingma & Ba 2015) on float32 master weights, refreshing their bf16 copy
__global__ __launch_bounds__(256) void adam_kernel(float* w, const float* g, float* m, float* v, int64_t n,
                                                   float lr, float b1, float b2, float eps, float c1,
                                                   float c2, uint16_t* wb) {
  for (int64_t e = blockIdx.x * 256ll + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
    const float gg = g[e];
    const float mm = b1 * m[e] + (1.0f - b1) * gg;
    const float vv = b2 * v[e] + (1.0f - b2) * gg * gg;
    m[e] = mm;
    v[e] = vv;
    const float ww = w[e] - lr * (mm / c1) / (sqrtf(vv / c2) + eps);
    w[e] = ww;
    if (wb) wb[e] = to_bf16(ww);
  }
}

// network input: asinh(x / sigma) of each 64 x 64 cutout (one sigma per cutout), bf16
__global__ __launch_bounds__(256) void asinh_input_kernel(const float* x, const float* sigma, int Bn,
                                                          int npx, uint16_t* out) {
  const int64_t total = (int64_t)Bn * npx;
  for (int64_t e = blockIdx.x * 256ll + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
    const int b = (int)(e / npx);
    out[e] = to_bf16(asinhf(x[e] / sigma[b]));
  }
}

// ---------------------------------------------------------------------------
// The network's input and its four convolutions of one cutout in one workgroup:
// asinh(x / sigma), 64 x 64 x 1 -> 32 x 32 x 32 -> 16 x 16 x 32 -> 8 x 8 x 64 ->
// 4 x 4 x 64, every activation in LDS.  A launch a layer wrote each activation in
// float32 (which only the gradients read) and bfloat16 and read it back, 3 GB for
// 8,192 cutouts, bound by HBM at 1.42 ms with the input pass; here a cutout's
// 16 kB come in and 2 kB go out: 0.25 ms, set by the waves' own instructions.
//
// A layer's products are those of gemm_bf16_kernel: K = (ky, kx, ci) in steps of
// 32 through one accumulator, so the outputs have the same bits.  The weights are
// the MFMA's A operand and the pixels its B, so a lane ends with 4 consecutive
// channels of a pixel: one 8-byte write.  A row of an activation holds its even
// columns, then its odd ones: the 16 pixels of an operand are neighbours in LDS
// for each tap of the stride-2 kernel (without bank conflicts, 64 bytes apart).
// LDS: 64 kB of layer 1 (then layer 3) and 16 kB of the input (then layer 2), so
// that two workgroups of 8 waves fit a CU.
constexpr int kFtWaves = 8, kFtThreads = 64 * kFtWaves;
constexpr int kFtIn = 36;                 // dwords a row of the input: columns -1 .. 64 as pairs, whole 16 bytes
constexpr int kFtBig = 32 * 1024;         // layer 1 (bf16 values)
constexpr size_t kFtLds = 2 * (kFtBig + 8 * 1024);
static_assert(65 * kFtIn * 4 <= 2 * 8 * 1024, "the input fits the second region");
// packed weights: layer, k-step, 16 channels, lane, 8 values
constexpr int kFtW[4] = {0, 32 * 32, 32 * 32 + 288 * 32, 32 * 32 + 288 * 32 + 288 * 64};
constexpr int kFtWeights = 32 * 32 + 288 * 32 + 288 * 64 + 576 * 64;

struct FeatureNet {
  const uint16_t* w[4];  // (K, Cout) bf16 of each convolution, K padded to 32
  const float* b[4];
};

// the four weight matrices in the order the lanes of a k-step read them: lane l
// of step s and channel block t holds W[32 s + 8 (l / 16) + j][16 t + l % 16]
__global__ __launch_bounds__(256) void pack_weights_kernel(FeatureNet net, uint16_t* __restrict__ out) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= kFtWeights) return;
  const int layer = e < kFtW[1] ? 0 : e < kFtW[2] ? 1 : e < kFtW[3] ? 2 : 3;
  const int N = layer < 2 ? 32 : 64;
  int r = e - (layer == 0 ? kFtW[0] : layer == 1 ? kFtW[1] : layer == 2 ? kFtW[2] : kFtW[3]);
  const int j = r & 7, l = (r >> 3) & 63;
  r >>= 9;
  const int t = r % (N / 16), s = r / (N / 16);
  const uint16_t* W = layer == 0 ? net.w[0] : layer == 1 ? net.w[1] : layer == 2 ? net.w[2] : net.w[3];
  out[e] = W[(int64_t)(32 * s + 8 * (l >> 4) + j) * N + 16 * t + (l & 15)];
}

__device__ __forceinline__ v8bf as_bf8(uint4 v) { return __builtin_bit_cast(v8bf, v); }

// two values as bf16 pair (round to nearest even, the first in the low half): the
// bits of to_bf16 but for a NaN's payload
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  typedef float v2f __attribute__((ext_vector_type(2)));
  typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(((v2f){a, b}), v2bf));
}

// bias, ReLU and bf16 of a lane's 4 channels, as 8 bytes
__device__ __forceinline__ uint2 finish4(v4f acc, float4 b) {
  return make_uint2(pack2(fmaxf(acc[0] + b.x, 0.0f), fmaxf(acc[1] + b.y, 0.0f)),
                    pack2(fmaxf(acc[2] + b.z, 0.0f), fmaxf(acc[3] + b.w, 0.0f)));
}

// 8 channels of a tap's pixel, zero outside the image (`in` false).  The read goes
// ahead all the same, at an address inside the activation: under a branch each
// read would wait for itself.
__device__ __forceinline__ v8bf tap8(const uint16_t* at, bool in) {
  const uint4 v = *reinterpret_cast<const uint4*>(at);
  const uint32_t m = in ? ~0u : 0u;
  return as_bf8(make_uint4(v.x & m, v.y & m, v.z & m, v.w & m));
}

__device__ __forceinline__ float4 bias4(const float* b, int c) { return make_float4(b[c], b[c + 1], b[c + 2], b[c + 3]); }

// asinh(z) to within kAsinhUlp of asinhf: the odd series below 1/4, log2 and sqrt
// units above.  `sure`: its bf16 rounding is that of asinhf, since no float within
// kAsinhMargin ulp rounds another way (the margin also covers z = x (1 / sigma)
// for x / sigma, 3 ulp); a pixel in 1,000 is not sure and takes asinhf itself,
// which is 230 instructions beside 25 here (20 us for 4,096 cutouts).
constexpr int kAsinhUlp = 12, kAsinhMargin = 2 * kAsinhUlp;
__device__ __forceinline__ float asinh_fast(float z, bool& sure) {
  const float a = fabsf(z), t = a * a;
  const float lo = fmaf(a * t, fmaf(t, fmaf(t, fmaf(t, 105.0f / 3456.0f, -15.0f / 336.0f), 3.0f / 40.0f), -1.0f / 6.0f), a);
  const float hi = 0.693147180559945309f * __builtin_amdgcn_logf(a + __builtin_amdgcn_sqrtf(fmaf(a, a, 1.0f)));
  const float y = a < 0.25f ? lo : hi;
  const int off = (int)(__float_as_uint(y) & 0xffffu) - 0x8000;
  sure = a >= 1e-30f && a <= 1e9f && (off > kAsinhMargin || off < -kAsinhMargin);
  return copysignf(y, z);
}

__global__ __launch_bounds__(kFtThreads, 4) void features_kernel(const float* __restrict__ images,
                                                                  const float* __restrict__ sigma, int B,
                                                                  FeatureNet net, const uint16_t* __restrict__ wp,
                                                                  uint16_t* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) uint16_t sm[];
  uint16_t* big = sm;             // layer 1 [y][x odd][x / 2][32], layer 3 [y][x odd][x / 2][64]
  uint16_t* low = sm + kFtBig;    // layer 2 [y][x odd][x / 2][32]
  uint32_t* in = reinterpret_cast<uint32_t*>(low);  // input: row y + 1, pair (x + 1) / 2
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, p = lane & 15, kq = lane >> 4;
  const uint4* w0 = reinterpret_cast<const uint4*>(wp);  // 64 x 16 bytes a block
  const v8bf w1[2] = {as_bf8(w0[lane]), as_bf8(w0[64 + lane])};
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  // this thread's pixels of a cutout: row y, columns 8 c ..
  const int y = t >> 3, c = t & 7;
  float px[8];
  auto load = [&](int b) {
    const float* src = images + (int64_t)b * 4096 + 8 * t;
#pragma unroll
    for (int q = 0; q < 8; ++q) px[q] = src[q];
  };
  if ((int)blockIdx.x < B) load(blockIdx.x);
  for (int b = blockIdx.x; b < B; b += gridDim.x) {
    // the weights of layers 2 to 4 are read for each cutout (from L2): held across
    // the loop, as the compiler would, they spill
    int keep = 0;
    asm volatile("" : "+s"(keep));
    const uint4* w4 = w0 + keep + lane;
    // ---- input
    {
      const float sg = sigma[b], rs = 1.0f / sg;
      const bool range = fabsf(sg) >= 1e-30f && fabsf(sg) <= 1e30f;
      float h[8];
      uint32_t left = 0;  // the pixels that take asinhf
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        bool sure;
        h[q] = asinh_fast(px[q] * rs, sure);
        if (px[q] == 0.0f) {
          h[q] = px[q] * copysignf(1.0f, sg);
          sure = true;
        }
        left |= (sure && range) ? 0u : 1u << q;
      }
      const float before = __shfl_up(h[7], 1, 64);  // every lane takes part
      uint32_t* row = in + (y + 1) * kFtIn + 4 * c;
      *reinterpret_cast<uint4*>(row) =
          make_uint4(pack2(c == 0 ? 0.0f : before, h[0]), pack2(h[1], h[2]), pack2(h[3], h[4]), pack2(h[5], h[6]));
      if (c == 7) row[4] = pack2(h[7], 0.0f);
      if (t < kFtIn) in[t] = 0u;  // the row above the image
      // the 2-byte writes below come after the 16-byte ones above (one wave's rows)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      while (__any(left != 0)) {
        if (left) {
          const int q = __ffs(left) - 1;
          left &= left - 1;
          reinterpret_cast<uint16_t*>(in)[(y + 1) * 2 * kFtIn + 1 + 8 * c + q] =
              to_bf16(asinhf(images[(int64_t)b * 4096 + 8 * t + q] / sg));
        }
      }
      if (b + (int)gridDim.x < B) load(b + gridDim.x);
    }
    __syncthreads();
    // ---- layer 1: a tile is 16 pixels of a row; K = the 9 taps
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int oy = w + kFtWaves * (q >> 1), ox = 16 * (q & 1) + p;
      const uint32_t* r0 = in + 2 * oy * kFtIn + ox;  // row 2 oy - 1, columns 2 ox - 1, 2 ox
      const uint32_t d0 = r0[0], d1 = r0[1], e0 = r0[kFtIn], e1 = r0[kFtIn + 1], f0 = r0[2 * kFtIn], f1 = r0[2 * kFtIn + 1];
      uint4 v = make_uint4(d0, (d1 & 0xffffu) | (e0 << 16), (e0 >> 16) | (e1 << 16), f0);
      if (kq == 1) v = make_uint4(f1 & 0xffffu, 0u, 0u, 0u);
      if (kq > 1) v = zero;
      uint16_t* o = big + oy * 1024 + (ox & 1) * 512 + (ox >> 1) * 32 + 4 * kq;
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const v4f acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[n], as_bf8(v), (v4f){0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
        *reinterpret_cast<uint2*>(o + 16 * n) = finish4(acc, bias4(net.b[0], 16 * n + 4 * kq));
      }
    }
    __syncthreads();
    // ---- layer 2: 16 channels and four rows of 16 pixels a wave
    {
      const int n = w & 1, oy0 = w >> 1;
      v4f acc[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int tap = 0; tap < 9; ++tap) {
        const int ky = tap / 3, kx = tap % 3;
        const v8bf a = as_bf8(w4[kFtW[1] / 8 + (tap * 2 + n) * 64]);
        const int col = (kx == 0 ? 512 - 32 : kx == 1 ? 0 : 512) + p * 32 + kq * 8;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int iy = 2 * (oy0 + 4 * i) + ky - 1;
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, tap8(big + max(iy, 0) * 1024 + col, !(i == 0 && ky == 0 && iy < 0) && !(kx == 0 && p == 0)), acc[i], 0, 0, 0);
        }
      }
      const float4 bb = bias4(net.b[1], 16 * n + 4 * kq);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<uint2*>(low + (oy0 + 4 * i) * 512 + (p & 1) * 256 + (p >> 1) * 32 + 16 * n + 4 * kq) =
            finish4(acc[i], bb);
    }
    __syncthreads();
    // ---- layer 3: 16 channels and twice two rows of 8 pixels a wave
    {
      const int n = w & 3, m0 = w >> 2, ox = p & 7;
      v4f acc[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int tap = 0; tap < 9; ++tap) {
        const int ky = tap / 3, kx = tap % 3;
        const v8bf a = as_bf8(w4[kFtW[2] / 8 + (tap * 4 + n) * 64]);
        const int col = (kx == 0 ? 256 - 32 : kx == 1 ? 0 : 256) + ox * 32 + kq * 8;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int iy = 2 * (2 * (m0 + 2 * i) + (p >> 3)) + ky - 1;
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, tap8(low + max(iy, 0) * 512 + col, !(i == 0 && ky == 0 && iy < 0) && !(kx == 0 && ox == 0)), acc[i], 0, 0, 0);
        }
      }
      const float4 bb = bias4(net.b[2], 16 * n + 4 * kq);
#pragma unroll
      for (int i = 0; i < 2; ++i)
        *reinterpret_cast<uint2*>(big + (2 * (m0 + 2 * i) + (p >> 3)) * 512 + (ox & 1) * 256 + (ox >> 1) * 64 + 16 * n +
                                  4 * kq) = finish4(acc[i], bb);
    }
    __syncthreads();
    // ---- layer 4: 16 channels of the 4 x 4 pixels a wave (the other waves go on
    // to the next cutout's input)
    if (w < 4) {
      const int oy = p >> 2, ox = p & 3;
      v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int s = 0; s < 18; ++s) {
        const int ky = (s >> 1) / 3, kx = (s >> 1) % 3;
        const v8bf a = as_bf8(w4[kFtW[3] / 8 + (s * 4 + w) * 64]);
        const int iy = 2 * oy + ky - 1;
        const uint16_t* at = big + max(iy, 0) * 512 + (kx == 0 ? 256 - 64 : kx == 1 ? 0 : 256) + ox * 64 + (s & 1) * 32 + kq * 8;
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, tap8(at, !(ky == 0 && iy < 0) && !(kx == 0 && ox == 0)), acc, 0, 0, 0);
      }
      *reinterpret_cast<uint2*>(out + (int64_t)b * 1024 + p * 64 + 16 * w + 4 * kq) =
          finish4(acc, bias4(net.b[3], 16 * w + 4 * kq));
    }
  }
}

// The form of an operand with element (r, k) at X[r * sr + k * sk] (R rows,
// depth K): 16-byte loads where one of the two strides is 1 and the other, the
// contiguous extent and the base keep every load whole and on 16 bytes.
inline int operand_form(const uint16_t* X, int64_t sr, int64_t sk, int R, int K) {
  if (reinterpret_cast<uintptr_t>(X) & 15) return OP_ANY;
  if (sk == 1 && sr % 8 == 0 && K % 8 == 0) return OP_KROW;
  if (sr == 1 && sk % 8 == 0 && R % 8 == 0) return OP_RROW;
  return OP_ANY;
}

// One GEMM launch with each operand in its form.  The forms give the same
// products in the same order, so the choice does not change a bit of the
// result.  With both operands read 2 bytes at a time the 17 GEMMs of a training
// step on 256 cutouts take 1.56 ms; with the 16-byte forms 0.395 ms.
void launch_gemm(dim3 grid, hipStream_t stream, int aop, int bop, int M, int N, int K, const uint16_t* A, int64_t sam,
                 int64_t sak, const uint16_t* B, int64_t sbk, int64_t sbn, float* C, int64_t ldc, const float* bias,
                 int relu, uint16_t* Cb, int accumulate, float* P, int kchunk, ConvA cv) {
#define APX_GEMM(AO, BO)                                                                                          \
  hipLaunchKernelGGL((gemm_bf16_kernel<AO, BO>), grid, dim3(256), 0, stream, M, N, K, A, sam, sak, B, sbk, sbn, C, \
                     ldc, bias, relu, Cb, accumulate, P, kchunk, cv)
#define APX_GEMM_B(AO)                                                                   \
  do {                                                                                   \
    if (bop == OP_KROW) APX_GEMM(AO, OP_KROW);                                           \
    else if (bop == OP_RROW) APX_GEMM(AO, OP_RROW);                                      \
    else APX_GEMM(AO, OP_ANY);                                                           \
  } while (0)
  if (aop == OP_KROW) APX_GEMM_B(OP_KROW);
  else if (aop == OP_RROW) APX_GEMM_B(OP_RROW);
  else if (aop == OP_CONV) APX_GEMM_B(OP_CONV);
  else APX_GEMM_B(OP_ANY);
#undef APX_GEMM_B
#undef APX_GEMM
}

inline dim3 grid_for(int64_t n) { return dim3((unsigned)std::min<int64_t>((n + 255) / 256, 8192)); }

}  // namespace

int gemm_bf16(int M, int N, int K, const uint16_t* A, int64_t sam, int64_t sak, const uint16_t* B,
              int64_t sbk, int64_t sbn, float* C, int64_t ldc, const float* bias, int relu,
              uint16_t* Cb, int accumulate, int splits, float* ws, int64_t ws_floats,
              hipStream_t stream) {
  if (M < 0 || N < 0 || K < 0 || !A || !B || !C || ldc < N || splits < 1)
    return set_error(APX_E_INVALID, "gemm_bf16: bad arguments");
  if (M == 0 || N == 0) return APX_OK;
  const dim3 grid((M + BM - 1) / BM, (N + BN - 1) / BN, splits);  // M tiles on x (up to 2^31 - 1)
  if (grid.y > 65535 || splits > 65535) return set_error(APX_E_LIMIT, "gemm_bf16: N or splits too large");
  // k range per split: a multiple of the k-step
  const int kchunk = splits == 1 ? std::max(K, 1) : ((K + splits - 1) / splits + BK - 1) / BK * BK;
  const int aop = operand_form(A, sam, sak, M, K), bop = operand_form(B, sbn, sbk, N, K);
  if (splits > 1) {
    if (!ws || ws_floats < (int64_t)splits * M * N)
      return set_error(APX_E_INVALID, "gemm_bf16: split-K workspace too small");
    launch_gemm(grid, stream, aop, bop, M, N, K, A, sam, sak, B, sbk, sbn, C, ldc, bias, relu, Cb, accumulate, ws, kchunk,
                ConvA{});
    hipLaunchKernelGGL(splitk_sum_kernel, grid_for((int64_t)M * N), dim3(256), 0, stream, ws, splits, M, N,
                       C, ldc, bias, relu, Cb, accumulate);
  } else {
    launch_gemm(grid, stream, aop, bop, M, N, K, A, sam, sak, B, sbk, sbn, C, ldc, bias, relu, Cb, accumulate, nullptr,
                kchunk, ConvA{});
  }
  return check_launch("gemm_bf16");
}

int conv_s2_bf16(const uint16_t* X, int Bn, int H, int W, int Cin, int Kp, const uint16_t* Wt, int N,
                 float* C, const float* bias, int relu, uint16_t* Cb, hipStream_t stream) {
  if (!X || !Wt || !C || Bn < 1 || H < 1 || W < 1 || Cin < 1 || N < 1 || Kp < 9 * Cin || Kp % BK != 0)
    return set_error(APX_E_INVALID, "conv_s2_bf16: bad arguments");
  const int Ho = (H + 1) / 2, Wo = (W + 1) / 2;
  const int64_t M64 = (int64_t)Bn * Ho * Wo;
  if (M64 > INT32_MAX) return set_error(APX_E_LIMIT, "conv_s2_bf16: too many output pixels");
  const int M = (int)M64;
  const dim3 grid((M + BM - 1) / BM, (N + BN - 1) / BN, 1);
  if (grid.y > 65535) return set_error(APX_E_LIMIT, "conv_s2_bf16: N too large");
  const ConvA cv{X, H, W, Cin, Ho, Wo};
  launch_gemm(grid, stream, OP_CONV, operand_form(Wt, 1, N, N, Kp), M, N, Kp, nullptr, 0, 0, Wt, N, 1, C, N, bias, relu, Cb,
              0, nullptr, Kp, cv);
  return check_launch("conv_s2_bf16");
}

int mse(const float* y, const float* t, const float* w, int Bn, int N, float* dy, float* loss,
        hipStream_t stream) {
  if (!y || !t || !w || !dy || !loss || Bn < 1 || N < 1) return set_error(APX_E_INVALID, "mse: bad arguments");
  hipLaunchKernelGGL(mse_kernel, dim3(1), dim3(256), 0, stream, y, t, w, Bn, N, dy, loss);
  return check_launch("mse");
}

int im2col_s2(const uint16_t* X, int Bn, int H, int W, int Cin, int Kp, uint16_t* col,
              hipStream_t stream) {
  if (!X || !col || Bn < 1 || H < 1 || W < 1 || Cin < 1 || Kp < 9 * Cin)
    return set_error(APX_E_INVALID, "im2col: bad arguments");
  const int64_t n = (int64_t)Bn * ((H + 1) / 2) * ((W + 1) / 2) * Kp;
  // 8 columns a thread where every row starts on 16 bytes (and so does each tap's
  // group of 8 channels); their count fits 32 bits with a grid's stride to spare
  const uintptr_t at = reinterpret_cast<uintptr_t>(col) | (Cin % 8 == 0 ? reinterpret_cast<uintptr_t>(X) : 0);
  if (Kp % 8 == 0 && (at & 15) == 0 && n / 8 < (int64_t)1 << 31)
    hipLaunchKernelGGL(im2col8_kernel, grid_for(n / 8), dim3(256), 0, stream, X, H, W, Cin, Kp, (uint32_t)(n / 8), col);
  else
    hipLaunchKernelGGL(im2col_kernel, grid_for(n), dim3(256), 0, stream, X, Bn, H, W, Cin, Kp, col);
  return check_launch("im2col");
}

int col2im_s2(const float* dcol, int Bn, int H, int W, int Cin, int Kp, float* dX, hipStream_t stream) {
  if (!dcol || !dX || Bn < 1 || H < 1 || W < 1 || Cin < 1 || Kp < 9 * Cin)
    return set_error(APX_E_INVALID, "col2im: bad arguments");
  const int64_t n = (int64_t)Bn * H * W * Cin;
  // 4 channels a thread where every row of dcol and of dX keeps them on 16 bytes
  if (Cin % 4 == 0 && Kp % 4 == 0 && ((reinterpret_cast<uintptr_t>(dcol) | reinterpret_cast<uintptr_t>(dX)) & 15) == 0 &&
      n / 4 < (int64_t)1 << 31)
    hipLaunchKernelGGL(col2im4_kernel, grid_for(n / 4), dim3(256), 0, stream, dcol, H, W, Cin, Kp, (uint32_t)(n / 4), dX);
  else
    hipLaunchKernelGGL(col2im_kernel, grid_for(n), dim3(256), 0, stream, dcol, Bn, H, W, Cin, Kp, dX);
  return check_launch("col2im");
}

int cast_gate(const float* src, const float* mask, int64_t n, uint16_t* dst, float* dstf,
              hipStream_t stream) {
  if (!src || !dst || n < 0) return set_error(APX_E_INVALID, "cast_gate: bad arguments");
  if (n == 0) return APX_OK;
  hipLaunchKernelGGL(cast_gate_kernel, grid_for(n), dim3(256), 0, stream, src, mask, n, dst, dstf);
  return check_launch("cast_gate");
}

int colsum(const float* X, int M, int N, float* out, hipStream_t stream) {
  if (!X || !out || M < 0 || N < 1) return set_error(APX_E_INVALID, "colsum: bad arguments");
  hipLaunchKernelGGL(colsum_kernel, dim3((N + 63) / 64), dim3(256), 0, stream, X, M, N, out);
  return check_launch("colsum");
}

int gate_colsum(const float* src, const float* mask, int M, int N, uint16_t* dst, float* out, float* ws,
                int64_t ws_floats, hipStream_t stream) {
  if (!src || !dst || !out || !ws || M < 0 || N < 1) return set_error(APX_E_INVALID, "gate_colsum: bad arguments");
  if (ws_floats < N) return set_error(APX_E_INVALID, "gate_colsum: workspace below N floats");
  // 16-byte loads of 4 columns where whole rows fill a step of the workgroup
  // (N = 4, 8, .., 1024) and every row starts on 16 bytes (8 in dst)
  const bool vec = N % 4 == 0 && N <= 1024 && 256 % (N / 4) == 0 &&
                   ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(mask)) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(dst) & 7) == 0;
  const int rows = vec ? 1024 / N : 4;  // rows a step
  // two workgroups a CU at most, and no more than the workspace holds partials for
  const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(512, ws_floats / N), ((int64_t)M + rows - 1) / rows));
  if (vec)
    hipLaunchKernelGGL(gate_colsum_kernel<true>, dim3(nb), dim3(256), 0, stream, src, mask, M, N, dst, ws);
  else
    hipLaunchKernelGGL(gate_colsum_kernel<false>, dim3(nb, (N + 63) / 64), dim3(256), 0, stream, src, mask, M, N, dst, ws);
  hipLaunchKernelGGL(column_final_kernel, dim3((N + 3) / 4), dim3(256), 0, stream, ws, nb, N, out);
  return check_launch("gate_colsum");
}

int adam(float* w, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2,
         float eps, int step, uint16_t* wb, hipStream_t stream) {
  if (!w || !g || !m || !v || n < 0 || step < 1) return set_error(APX_E_INVALID, "adam: bad arguments");
  if (n == 0) return APX_OK;
  const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
  hipLaunchKernelGGL(adam_kernel, grid_for(n), dim3(256), 0, stream, w, g, m, v, n, lr, b1, b2, eps, c1,
                     c2, wb);
  return check_launch("adam");
}

int64_t init_features_workspace_bytes() { return 2 * kFtWeights; }

int init_features(const float* images, const float* sigma, int Bn, const uint16_t* const* w, const float* const* b,
                  uint16_t* out, void* ws, int64_t ws_bytes, hipStream_t stream) {
  if (!images || !sigma || !w || !b || !out || !ws || Bn < 1) return set_error(APX_E_INVALID, "init_features: bad arguments");
  if (ws_bytes < init_features_workspace_bytes()) return set_error(APX_E_INVALID, "init_features: workspace too small");
  if ((reinterpret_cast<uintptr_t>(ws) & 15) || (reinterpret_cast<uintptr_t>(out) & 7))
    return set_error(APX_E_INVALID, "init_features: workspace not on 16 bytes or output not on 8");
  FeatureNet net;
  for (int k = 0; k < 4; ++k) {
    if (!w[k] || !b[k]) return set_error(APX_E_INVALID, "init_features: bad arguments");
    net.w[k] = w[k];
    net.b[k] = b[k];
  }
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(&features_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)kFtLds) != hipSuccess)
    return set_error(APX_E_HIP, "init_features: LDS size refused");
  uint16_t* wp = static_cast<uint16_t*>(ws);
  hipLaunchKernelGGL(pack_weights_kernel, dim3((kFtWeights + 255) / 256), dim3(256), 0, stream, net, wp);
  // two workgroups a CU, each cutout after cutout: the weights of layer 1 and the
  // next cutout's pixels stay in registers
  hipLaunchKernelGGL(features_kernel, dim3(std::min(Bn, 512)), dim3(kFtThreads), kFtLds, stream, images, sigma, Bn, net,
                     (const uint16_t*)wp, out);
  return check_launch("init_features");
}

int asinh_input(const float* x, const float* sigma, int Bn, int npx, uint16_t* out, hipStream_t stream) {
  if (!x || !sigma || !out || Bn < 1 || npx < 1) return set_error(APX_E_INVALID, "asinh_input: bad arguments");
  hipLaunchKernelGGL(asinh_input_kernel, grid_for((int64_t)Bn * npx), dim3(256), 0, stream, x, sigma, Bn,
                     npx, out);
  return check_launch("asinh_input");
}

}  // namespace apx
