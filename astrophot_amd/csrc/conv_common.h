// Direct-convolution pieces shared by the single-component convolution
// (convolve.hip) and the batched one (batch.hip).
//
// Taps are pre-arranged as KT[k][b][u] = K[u - 7][b] (zero outside the
// kernel), kts floats per tap column, so that the 8 output rows of a
// wavefront find the tap of (input row t, output row r) at u = t - r + 7.
#pragma once

#include <hip/hip_runtime.h>

namespace apx {

constexpr int kRYF = 8;       // output rows per workgroup (one accumulator each)
constexpr int kFastMax = 89;  // largest kernel side whose tile fits 64 KiB of LDS

__host__ __device__ inline int fast_nt(int kh) { return (kh + kRYF - 1 + 7) / 8; }
__host__ __device__ inline int fast_kts(int kh) { return 8 * fast_nt(kh) + 8; }

// Bilinear sample of the 1-px zero-padded PSF at (c - sx, r - sy) with the
// reference's clamped corners (utils/interpolate.py:282-329), and its
// derivatives with respect to the shift; at(y, x) is the padded PSF's value.
template <typename At>
__device__ __forceinline__ void bilinear_of(At&& at, int ph, int pw, int r, int c, double sx, double sy, double& val,
                                            double& dsx, double& dsy) {
  const int H2 = ph + 2, W2 = pw + 2;
  const double x = (double)c - sx, y = (double)r - sy;
  const int xf = (int)floor(x), yf = (int)floor(y);
  const int x0 = min(max(xf, 0), W2 - 2), x1 = min(max(xf + 1, 1), W2 - 1);
  const int y0 = min(max(yf, 0), H2 - 2), y1 = min(max(yf + 1, 1), H2 - 1);
  const double fa = at(y0, x0), fb = at(y1, x0), fc = at(y0, x1), fd = at(y1, x1);
  const double wx1 = (double)x1 - x, wx0 = x - (double)x0;
  const double wy1 = (double)y1 - y, wy0 = y - (double)y0;
  val = fa * wx1 * wy1 + fb * wx1 * wy0 + fc * wx0 * wy1 + fd * wx0 * wy0;
  dsx = -(-fa * wy1 - fb * wy0 + fc * wy1 + fd * wy0);  // d/ds_x = -d/dx
  dsy = -(-fa * wx1 + fb * wx1 - fc * wx0 + fd * wx0);  // d/ds_y = -d/dy
}

// the PSF in memory, without its border
__device__ __forceinline__ void bilinear(const float* psf, int ph, int pw, int r, int c, double sx,
                                         double sy, double& val, double& dsx, double& dsy) {
  bilinear_of([&](int yy, int xx) -> double {
    return (yy >= 1 && yy <= ph && xx >= 1 && xx <= pw) ? (double)psf[(yy - 1) * pw + (xx - 1)] : 0.0;
  }, ph, pw, r, c, sx, sy, val, dsx, dsy);
}

// The padded PSF in LDS ((ph + 2) x (pw + 2) floats), by the whole workgroup.  A
// sample reads four neighbours; from memory each is a conditional load that the
// next waits for.
__device__ __forceinline__ void pad_psf(const float* __restrict__ psf, int ph, int pw, float* lds) {
  const int W2 = pw + 2, n = (ph + 2) * W2;
  for (int e = threadIdx.x; e < n; e += blockDim.x) {
    const int r = e / W2 - 1, c = e % W2 - 1;
    lds[e] = (r >= 0 && r < ph && c >= 0 && c < pw) ? psf[r * pw + c] : 0.0f;
  }
}
__device__ __forceinline__ void bilinear_lds(const float* lds, int ph, int pw, int r, int c, double sx, double sy,
                                             double& val, double& dsx, double& dsy) {
  bilinear_of([&](int yy, int xx) -> double { return (double)lds[yy * (pw + 2) + xx]; }, ph, pw, r, c, sx, sy, val, dsx,
              dsy);
}

// One wavefront's share of a 64 x 8 output tile: input-row blocks j = wu,
// wu + 4, ... of the staged tile (row length LW), all tap columns, nk kernels
// (nk <= NKmax).  Taps go through the scalar cache in bursts of 16.
template <int NKmax>
__device__ __forceinline__ void conv_accumulate(const float* smem, int LW, int lane, int wu, int nT,
                                                int kw, int kts, int nk,
                                                const float* __restrict__ kt,
                                                float (&acc)[NKmax][kRYF]) {
  for (int j = wu; j < nT; j += 4) {
    const int t0 = 8 * j;
    const float* trow = smem + t0 * LW + lane;
    const float* ktj = kt + t0;
    for (int b = 0; b < kw; ++b) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = trow[i * LW + b];
#pragma unroll
      for (int k = 0; k < NKmax; ++k) {
        if (k < nk) {
          const float4* kp = reinterpret_cast<const float4*>(ktj + ((int64_t)k * kw + b) * kts);
          const float4 q0 = kp[0], q1 = kp[1], q2 = kp[2], q3 = kp[3];
          const float kk[16] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w,
                                q2.x, q2.y, q2.z, q2.w, q3.x, q3.y, q3.z, q3.w};
#pragma unroll
          for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int r = 0; r < kRYF; ++r) acc[k][r] = fmaf(kk[i - r + 7], v[i], acc[k][r]);
        }
      }
    }
  }
}


// ---------------------------------------------------------------------------
// Rows from HBM straight into LDS: row t of dst (rows x cols, pitch dpitch) gets
// src[(gy0 + t) * pitch + gx0 ..], zero where that lies outside nx x ny.  The
// workgroup's waves take the rows in turn, 64 floats a load, through a buffer
// resource of one source row from the tile's first column on: its range check gives
// the zeros (a column before the row is a huge unsigned offset, a row outside has an
// empty resource), so no register holds the data, nothing is divided and every load
// of the tile is in flight at once.  A resource has 32 bits of bytes: the rest of a
// longer row, which no tile reaches, is cut off.  Completion: vmcnt, then a barrier.
typedef __attribute__((address_space(3))) void* lds_ptr;
constexpr int kBufWord3 = 0x00020000;  // buffer resource word 3 on gfx9: 32-bit data

template <int NW = 4>  // waves of the workgroup
__device__ __forceinline__ void stage_rows(const float* src, int64_t pitch, int nx, int ny, int gx0, int gy0, int rows,
                                           int cols, float* dst, int dpitch) {
  const int lane = threadIdx.x & 63;
  const int bx = max(gx0, 0), bytes = min(max(nx - bx, 0), 1 << 28) * 4;
  for (int t = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); t < rows; t += NW) {
    const int gy = gy0 + t;
    const bool in = gy >= 0 && gy < ny;
    // every field of the resource is uniform: read from lane 0 so that it stays in SGPRs
    const uint64_t a = (uint64_t)(src + (int64_t)(in ? gy : 0) * pitch + bx);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), (short)0, __builtin_amdgcn_readfirstlane(in ? bytes : 0), kBufWord3);
    for (int c = 0; c < cols; c += 64)
      if (c + lane < cols)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)(dst + t * dpitch + c), 4, (gx0 - bx + c + lane) * 4, 0, 0, 0);
  }
}

// ---------------------------------------------------------------------------
// MFMA convolution by v_mfma_f32_16x16x4f32.  A wave computes a 16 x 16
// output block (16 columns x, kMfR rows r) as
//   out[r][x] = sum_kx sum_j A_kx[x][j] B_kx[j][r],
//   A_kx[x][j] = in[j][x + kx],  B_kx[j][r] = Kf[j - r][kx] (zero outside the kernel),
// j over the staged input rows in k-steps of 4.  A comes from the staged input
// tile, B from a per-kernel tap table tab[kx][dd] = Kf[dd - 15][kx], both in
// LDS.  A table column is mf_dd long and is read 15 entries further, into the
// next one's leading zeros.  Lane layout: A[l % 16][l / 16], B[l / 16][l % 16], and
// D[4 (l / 16) + i][l % 16] in acc[i] (x = 4 (l / 16) + i, r = l % 16).
// A kernel column needs kMfR + kh - 1 input rows, ceil of that / 4 k-steps
// (a compile-time count dispatched on the kernel height); the staged rows and
// the tap table are padded with zeros to whole k-steps.
typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int kMfR = 16;       // output rows of an MFMA block
constexpr int kMfmaWide = 67;  // tallest kernel mfma_block dispatches (21 k-steps)

__host__ __device__ constexpr int mf_nks(int kh) { return (kMfR + kh - 1 + 3) / 4; }  // k-steps per kx
__host__ __device__ constexpr int mf_rows(int kh) { return 4 * mf_nks(kh); }
// Row pitch of the staged input, one for every kernel width, so that an A
// operand's k-steps lie at immediate offsets.  144 floats hold the 64 + 67 - 1
// columns of the widest kernel and put the 4 rows x 16 columns of an operand
// (lanes l / 16, l % 16) in distinct LDS banks.
constexpr int kMfLW = 144;
__host__ __device__ constexpr int mf_dd(int kh) { return mf_rows(kh) + 1; }
__host__ __device__ constexpr int mf_tab(int kh, int kw) { return kw * mf_dd(kh) + 16; }  // the last column's zeros too
// LDS of one pass: the staged input of `blocks` 16-row output blocks and one tap table
__host__ constexpr size_t mfma_lds_bytes(int kh, int kw, int blocks = 1) {
  return sizeof(float) * ((size_t)(mf_rows(kh) + kMfR * (blocks - 1)) * kMfLW + (size_t)mf_tab(kh, kw));
}
__host__ constexpr size_t mfma_lds_bytes(int kmax) { return mfma_lds_bytes(kmax, kmax); }
// The single-image convolution may give two 16-row blocks to a workgroup of 8 waves,
// which share the halo rows and the tap table: two such workgroups fit a CU
// (kernels to 67: 80.4 kB of 80 KiB), 512 the chip, with 4 waves a SIMD in place of 2
// and half the staging an output.  It takes a full round of them (kMfTallMin): value
// plane, 768^2 (288 workgroups) 53 rows 51.0 -> 58.7 us, 1024^2 (512) 64.6 -> 59.0 and
// 21 rows 19.9 -> 19.2.  A Jacobian's columns also take kMfTallRows kernel rows: with
// fewer products a row their additions to interleaved memory weigh more, which more,
// smaller workgroups hide better.  Seven of 13 columns, 1024^2: 31 rows 201 -> 221 us,
// 39 rows 301 -> 276, 67 rows 723 -> 632; 512^2 (896): 31 rows 52.0 -> 58.4, 39 rows
// 80.5 -> 76.7, 53 rows 115.5 -> 116.8, and within a Jacobian of two components
// 112.5 -> 107.5.  (The batched convolution keeps one tile a workgroup: its tile pairs
// took 0.82 -> 0.88 ms over 256 uneven cutouts, where many last pairs are half empty.)
constexpr int kMfTallMin = 512, kMfTallRows = 37;

// All kernel columns of one output block: column kx needs NKS k-steps.  The
// operands of the next column are loaded between the MFMAs of the current one
// (two register sets of NKS A and B values): a wave issues in order and an MFMA
// holds its issue for 32 cycles, so loads placed ahead of a column's MFMAs
// would leave the matrix pipe idle while they issue (125 sources, 67 x 67
// kernels: 3.47 -> 2.78 ms; 512^2, 53 x 53: 32 -> 24.5 us a pass).
template <int NKS>
__device__ __forceinline__ v4f mfma_columns(const float* ta, const float* tb, int kw, int DD) {
  v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
  float a0[NKS], b0[NKS], a1[NKS], b1[NKS];
  // MFMAs of (a, b), the loads of column kx into (an, bn)
  auto step = [&](const float (&a)[NKS], const float (&b)[NKS], int kx, float (&an)[NKS], float (&bn)[NKS]) {
    const float* pa = ta + kx;
    const float* pb = tb + kx * DD;
#pragma unroll
    for (int t = 0; t < NKS; ++t) {
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t], b[t], acc, 0, 0, 0);
      an[t] = pa[4 * t * kMfLW];
      bn[t] = pb[4 * t];
    }
#pragma unroll
    for (int t = 0; t < NKS; ++t) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read (of two operands)
    }
  };
#pragma unroll
  for (int t = 0; t < NKS; ++t) {
    a0[t] = ta[4 * t * kMfLW];
    b0[t] = tb[4 * t];
  }
  int kx = 0;
  for (; kx + 1 < kw; kx += 2) {
    step(a0, b0, kx + 1, a1, b1);
    step(a1, b1, min(kx + 2, kw - 1), a0, b0);
  }
  if (kx < kw) {
#pragma unroll
    for (int t = 0; t < NKS; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[t], b0[t], acc, 0, 0, 0);
  }
  return acc;
}

// mfma_columns with the k-step count of the kernel height: 5 .. N k-steps,
// kernels of 1 .. 4 N - 15 rows (N = 21: kMfmaWide).  A launch whose register
// budget cannot hold 21-step operand sets instantiates a smaller N.
template <int N>
__device__ __forceinline__ v4f mfma_block_n(int nks, const float* ta, const float* tb, int kw, int DD) {
  if constexpr (N > 5) {
    if (nks < N) return mfma_block_n<N - 1>(nks, ta, tb, kw, DD);
  }
  return mfma_columns<N>(ta, tb, kw, DD);
}

__device__ __forceinline__ v4f mfma_block(int nks, const float* ta, const float* tb, int kw, int DD) {
  return mfma_block_n<21>(nks, ta, tb, kw, DD);
}

}  // namespace apx
