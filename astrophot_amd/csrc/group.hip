// A group model whose sources sit on windows of one image, with block-sparse
// Jacobian products for Levenberg-Marquardt (group_model_object.py:183-283,
// fit/lm.py:359-406).
//
// Each source is one cutout of an apx_batch (its window on the image), so
// its model and its 7 Jacobian columns live only on that window, in the
// batch's per-source buffers.  What LM needs from the whole group is built
// from those blocks without ever forming the dense (pixels x parameters) J:
//   image    sky + sum of the sources covering each pixel, in group order;
//   J^T W J  one 7 x 7 block per pair of overlapping windows, plus the sky
//            row (the sky's column is a constant on the image);
//   J^T v    per source over its window;  J h  per pixel over its sources.
// Pixels find their sources through a per-tile list (64 x 16 tiles) built on
// the host; every sum runs in a fixed order, so repeated runs give identical
// bits.  The damped normal equations are solved by a blocked float64
// Cholesky factorisation (right-looking, 32-column panels) and two blocked
// triangular solves.
#include <hip/hip_runtime.h>

#include "capi_internal.h"
#include "wave.h"

namespace apx {

namespace {

constexpr int kTW = 64, kTH = 16;  // image tile
constexpr int kNB = 32;            // Cholesky panel
constexpr int kUT = 64;            // trailing-update tile

// lane `src`'s v to every lane (src uniform): two v_readlane_b32 into SGPRs,
// no LDS round trip
__device__ __forceinline__ double lane_bcast(double v, int src) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), src);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), src);
  return __hiloint2double(hi, lo);
}

// Sum of the source values covering pixel (x, y), with the sky added where
// it stands in the group order.
template <typename F>
__device__ __forceinline__ double cover_sum(const apx_group& g, int x, int y, int tile, F&& value) {
  double v = 0.0;
  const int s0 = g.tile_ptr[tile], s1 = g.tile_ptr[tile + 1];
  bool sky_done = g.sky_after < 0;
  for (int e = s0; e < s1; ++e) {
    const int s = g.tile_src[e];
    if (!sky_done && s >= g.sky_after) {
      v += value(-1, 0);
      sky_done = true;
    }
    const int* w = g.win + 4 * s;
    const int dx = x - w[0], dy = y - w[1];
    if (dx >= 0 && dx < w[2] && dy >= 0 && dy < w[3])
      v += value(s, g.pix_off[s] + (int64_t)dy * w[2] + dx);
  }
  if (!sky_done) v += value(-1, 0);
  return v;
}

__global__ __launch_bounds__(256) void group_image_kernel(apx_group g, const float* __restrict__ src,
                                                          double sky, float* __restrict__ out) {
  const int tx = blockIdx.x % g.ntx, ty = blockIdx.x / g.ntx;
  const int x = tx * kTW + (threadIdx.x & 63);
  for (int r = threadIdx.x >> 6; r < kTH; r += 4) {
    const int y = ty * kTH + r;
    if (x >= g.nx || y >= g.ny) continue;
    const double v = cover_sum(g, x, y, blockIdx.x, [&](int s, int64_t p) -> double {
      return s < 0 ? sky : (double)src[p];
    });
    out[(int64_t)y * g.nx + x] = (float)v;
  }
}

// u = (2/d) (w (m1 - m0) / d - w (J h)) per pixel (zero where masked)
__global__ __launch_bounds__(256) void group_rpp_weights_kernel(apx_group g, const float* __restrict__ J,
                                                                const float* __restrict__ m0,
                                                                const float* __restrict__ m1,
                                                                const float* __restrict__ weight,
                                                                const uint8_t* __restrict__ mask,
                                                                const double* __restrict__ h, double d,
                                                                double sky_dcol, double* __restrict__ u) {
  const int tx = blockIdx.x % g.ntx, ty = blockIdx.x / g.ntx;
  const int x = tx * kTW + (threadIdx.x & 63);
  for (int r = threadIdx.x >> 6; r < kTH; r += 4) {
    const int y = ty * kTH + r;
    if (x >= g.nx || y >= g.ny) continue;
    const int64_t p = (int64_t)y * g.nx + x;
    const double jh = cover_sum(g, x, y, blockIdx.x, [&](int s, int64_t q) -> double {
      if (s < 0) return g.sky_col >= 0 ? sky_dcol * h[g.sky_col] : 0.0;
      const int c = g.col0[s];
      double t = 0.0;
#pragma unroll
      for (int k = 0; k < APX_BATCH_NP; ++k) t += (double)J[(int64_t)k * g.nsrcpix + q] * h[c + k];
      return t;
    });
    const double w = weight ? (double)weight[p] : 1.0;
    const bool keep = !(mask && mask[p]);
    u[p] = keep ? (2.0 / d) * (w * (double)(m1[p] - m0[p]) / d - w * jh) : 0.0;
  }
}

// A window (or an overlap of two) of n pixels goes to several workgroups: pieces
// of up to kPiece pixels, larger only where there would be more than S of them, so
// that the largest (400 x 400 beside a median overlap of 4,500 pixels) does not set
// the pass's time.  One workgroup a window: pairs, sources and J^T v of 500 sources
// on 2048^2 (3,051 pairs, 35 M pair pixels) took 0.94, 0.73 and 0.43 ms; in pieces
// 0.33, 0.16 and 0.12 ms.
constexpr int kPiece = 4096;

struct Piece {
  int x, y, dx, dy, w;  // this thread's pixel, and the step of 256 pixels
  int64_t e, e1;        // its index, and the end of the piece
  // piece s of at most S of a w x h rectangle; false: no such piece
  __device__ __forceinline__ bool open(int w_, int h, int s, int S) {
    const int64_t n = (int64_t)w_ * h;
    const int64_t np = min((int64_t)S, max((int64_t)1, (n + kPiece - 1) / kPiece)), len = (n + np - 1) / np;
    if (s >= np) return false;
    w = w_;
    e = s * len + threadIdx.x;
    e1 = min(n, (s + 1) * len);
    if (w > 0) {
      y = (int)(e / w);
      x = (int)(e - (int64_t)y * w);
      dy = 256 / w;
      dx = 256 - dy * w;
    }
    return true;
  }
  __device__ __forceinline__ void next() {
    e += 256;
    x += dx;
    y += dy;
    if (x >= w) {
      x -= w;
      ++y;
    }
  }
};
__device__ __forceinline__ int pieces_of(int64_t n, int S) {
  return (int)min((int64_t)S, max((int64_t)1, (n + kPiece - 1) / kPiece));
}
// The most pieces a window (or an overlap) gets when `count` of them share the
// chip.  Every one is launched, also those that small windows do not have, at some
// 10 ns each, so the launch is kept to 8,192 workgroups where that leaves 5 pieces
// or more (normal equations of 250 sources, 1,182 pairs: 372 us with 16, 285 with
// 8; of 30 sources, 185 pairs: 108 with 16, 127 with 8), and a group of small
// windows gets fewer: as many as one of three times the mean window has (1,000
// windows of 30 x 30: 362 us with 16, 142 with 1).  With one, the kernels write the
// result itself in place of a partial sum.
inline int max_pieces(const apx_group& g, int count) {
  const int64_t mean = g.nsrcpix / std::max(1, g.nsrc), n = std::max(1, count);
  return (int)std::max<int64_t>(1, std::min<int64_t>({16, std::max(8192 / n, std::min<int64_t>(5, 32768 / n)), 3 * mean / kPiece}));
}

// part[s S + piece][k] = sum over the piece of the window of J_k * v (v a double
// image); with S = 1 out[col0 + k] itself
__global__ __launch_bounds__(256) void group_jtv_kernel(apx_group g, const float* __restrict__ J,
                                                        const double* __restrict__ v, int S,
                                                        double* __restrict__ part, double* __restrict__ out) {
  __shared__ double red[4][APX_BATCH_NP];
  const int s = blockIdx.x / S;
  const int* w = g.win + 4 * s;
  const int w0 = w[0], w1 = w[1];
  Piece t;
  if (!t.open(w[2], w[3], blockIdx.x % S, S)) return;
  double acc[APX_BATCH_NP];
#pragma unroll
  for (int k = 0; k < APX_BATCH_NP; ++k) acc[k] = 0.0;
  const float* Js = J + g.pix_off[s];
  for (; t.e < t.e1; t.next()) {
    const double vv = v[(int64_t)(w1 + t.y) * g.nx + (w0 + t.x)];
#pragma unroll
    for (int k = 0; k < APX_BATCH_NP; ++k) acc[k] += (double)Js[(int64_t)k * g.nsrcpix + t.e] * vv;
  }
  wave_sums(acc, red[threadIdx.x >> 6]);
  __syncthreads();
  if (threadIdx.x < APX_BATCH_NP) {
    const int k = threadIdx.x;
    double* to = S == 1 ? out + g.col0[s] : part + (int64_t)blockIdx.x * APX_BATCH_NP;
    to[k] = red[0][k] + red[1][k] + red[2][k] + red[3][k];
  }
}

// out[col0 + k] = the sum of the source's pieces, in order
__global__ __launch_bounds__(256) void group_jtv_final_kernel(apx_group g, int S, const double* __restrict__ part,
                                                              double* __restrict__ out) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= g.nsrc * APX_BATCH_NP) return;
  const int s = e / APX_BATCH_NP, k = e % APX_BATCH_NP;
  const int np = pieces_of((int64_t)g.win[4 * s + 2] * g.win[4 * s + 3], S);
  double v = 0.0;
  for (int q = 0; q < np; ++q) v += part[((int64_t)s * S + q) * APX_BATCH_NP + k];
  out[g.col0[s] + k] = v;
}

// Image-wide float64 sums, one partial per workgroup (fixed order):
//   mode 0: part[b] = {sum w, sum w (data - model)}   (sky row of J^T W J, J^T W r)
//   mode 1: part[b] = {sum v, 0}                       (sky entry of J^T v)
__global__ __launch_bounds__(256) void group_image_sums_kernel(int64_t npix, int mode,
                                                               const float* __restrict__ model,
                                                               const float* __restrict__ data,
                                                               const float* __restrict__ weight,
                                                               const uint8_t* __restrict__ mask,
                                                               const double* __restrict__ v,
                                                               double* __restrict__ part) {
  __shared__ double red[2][4];
  double a = 0.0, b = 0.0;
  for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < npix; p += (int64_t)gridDim.x * 256) {
    if (mode == 1) {
      a += v[p];
      continue;
    }
    if (mask && mask[p]) continue;
    const double w = weight ? (double)weight[p] : 1.0;
    a += w;
    b += w * ((double)data[p] - (double)model[p]);
  }
  a = wave_sum(a);
  b = wave_sum(b);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][wv] = a;
    red[1][wv] = b;
  }
  __syncthreads();
  if (threadIdx.x < 2)
    part[2 * blockIdx.x + threadIdx.x] =
        red[threadIdx.x][0] + red[threadIdx.x][1] + red[threadIdx.x][2] + red[threadIdx.x][3];
}

// the sky entries from the image partials:
//   mode 0: H[sky][sky] = c^2 sum w, grad[sky] = c sum w r;  mode 1: out[sky] = c sum v
__global__ __launch_bounds__(256) void group_sky_final_kernel(int nblocks, int mode, int np, int sky, double c,
                                                              const double* __restrict__ part,
                                                              double* __restrict__ H, double* __restrict__ vec) {
  __shared__ double red[4][2];
  double ab[2] = {0.0, 0.0};
  for (int k = threadIdx.x; k < nblocks; k += 256) {
    ab[0] += part[2 * k];
    ab[1] += part[2 * k + 1];
  }
  wave_sums(ab, red[threadIdx.x >> 6]);
  __syncthreads();
  if (threadIdx.x != 0) return;
  const double a = red[0][0] + red[1][0] + red[2][0] + red[3][0];
  const double b = red[0][1] + red[1][1] + red[2][1] + red[3][1];
  if (mode == 0) {
    H[(int64_t)sky * np + sky] = c * c * a;
    vec[sky] = c * b;
  } else {
    vec[sky] = c * a;
  }
}

__global__ __launch_bounds__(256) void fill_kernel(double* __restrict__ a, int64_t n, double v) {
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) a[e] = v;
}

// Entry k of a source: grad[col0 + k] = v, and from k = NP on the sky column
// H[col0 + k - NP][sky] = H[sky][col0 + k - NP] = c v.
__device__ __forceinline__ void source_entry(const apx_group& g, int s, int k, double c, double v, double* H, double* grad) {
  constexpr int NP = APX_BATCH_NP;
  if (k < NP) {
    grad[g.col0[s] + k] = v;
  } else if (g.sky_col >= 0) {
    const int col = g.col0[s] + k - NP;
    H[(int64_t)col * g.np + g.sky_col] = c * v;
    H[(int64_t)g.sky_col * g.np + col] = c * v;
  }
}

// Per piece of a source's window: the sums of J_k w (data - model) and J_k w; kOne
// (S is 1): the entries themselves.
template <bool kOne>
__global__ __launch_bounds__(256) void group_source_kernel(apx_group g, const float* __restrict__ J,
                                                           const float* __restrict__ model,
                                                           const float* __restrict__ data,
                                                           const float* __restrict__ weight,
                                                           const uint8_t* __restrict__ mask, int S,
                                                           double* __restrict__ part, double c,
                                                           double* __restrict__ H, double* __restrict__ grad) {
  constexpr int NP = APX_BATCH_NP;
  __shared__ double red[4][2 * NP];
  const int s = blockIdx.x / S;
  const int* w = g.win + 4 * s;
  const int w0 = w[0], w1 = w[1];
  Piece t;
  if (!t.open(w[2], w[3], blockIdx.x % S, S)) return;
  double acc[2 * NP];
#pragma unroll
  for (int k = 0; k < 2 * NP; ++k) acc[k] = 0.0;
  const float* Js = J + g.pix_off[s];
  for (; t.e < t.e1; t.next()) {
    const int64_t p = (int64_t)(w1 + t.y) * g.nx + (w0 + t.x);
    if (mask && mask[p]) continue;
    const double ww = weight ? (double)weight[p] : 1.0;
    const double wr = ww * ((double)data[p] - (double)model[p]);
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const double j = (double)Js[(int64_t)k * g.nsrcpix + t.e];
      acc[k] += j * wr;
      acc[NP + k] += j * ww;
    }
  }
  wave_sums(acc, red[threadIdx.x >> 6]);
  __syncthreads();
  if (threadIdx.x < 2 * NP) {
    const int k = threadIdx.x;
    const double v = red[0][k] + red[1][k] + red[2][k] + red[3][k];
    if (kOne) source_entry(g, s, k, c, v, H, grad);
    else part[(int64_t)blockIdx.x * 2 * NP + k] = v;
  }
}

// the entries from the source's pieces, in order
__global__ __launch_bounds__(256) void group_source_final_kernel(apx_group g, int S, double c,
                                                                 const double* __restrict__ part,
                                                                 double* __restrict__ H,
                                                                 double* __restrict__ grad) {
  constexpr int NP = APX_BATCH_NP;
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= g.nsrc * 2 * NP) return;
  const int s = e / (2 * NP), k = e % (2 * NP);
  const int np = pieces_of((int64_t)g.win[4 * s + 2] * g.win[4 * s + 3], S);
  double v = 0.0;
  for (int q = 0; q < np; ++q) v += part[((int64_t)s * S + q) * 2 * NP + k];
  source_entry(g, s, k, c, v, H, grad);
}

// the overlap of windows a and b: corner (x0, y0), size ow x oh (not positive: none)
struct Overlap {
  int x0, y0, ow, oh;
  __device__ __forceinline__ Overlap(const int* wa, const int* wb) {
    x0 = max(wa[0], wb[0]);
    y0 = max(wa[1], wb[1]);
    ow = max(0, min(wa[0] + wa[2], wb[0] + wb[2]) - x0);
    oh = max(0, min(wa[1] + wa[3], wb[1] + wb[3]) - y0);
  }
};

// entry e of the pair's 7 x 7 block, at (a, b) and (b, a)
__device__ __forceinline__ void pair_entry(const apx_group& g, int a, int b, int e, double v, double* H) {
  const int ra = g.col0[a] + e / APX_BATCH_NP, rb = g.col0[b] + e % APX_BATCH_NP;
  H[(int64_t)ra * g.np + rb] = v;
  H[(int64_t)rb * g.np + ra] = v;
}

// One 7 x 7 block of J^T W J per pair of overlapping windows (a <= b): sum
// over the overlap of w J_a J_b^T, a piece a workgroup (kOne: S is 1, the block itself).  Bound by the J values of
// the pair pixels (56 bytes a pixel, most of them from the caches): the next
// pixel's loads are issued before the 49 multiply-adds of the current one.
template <bool kOne>
__global__ __launch_bounds__(256) void group_pair_kernel(apx_group g, const float* __restrict__ J,
                                                         const float* __restrict__ weight,
                                                         const uint8_t* __restrict__ mask, int S,
                                                         double* __restrict__ part, double* __restrict__ H) {
  constexpr int NP = APX_BATCH_NP, NN = NP * NP;
  __shared__ double red[4][NN];
  const int pr = blockIdx.x / S;
  const int a = g.pair[2 * pr], b = g.pair[2 * pr + 1];
  const int* wa = g.win + 4 * a;
  const int* wb = g.win + 4 * b;
  const Overlap o(wa, wb);
  const int sa = wa[2], sb = wb[2];
  Piece t;
  if (!t.open(o.ow, o.oh, blockIdx.x % S, S)) return;
  double acc[NN];
#pragma unroll
  for (int k = 0; k < NN; ++k) acc[k] = 0.0;
  const float* Ja = J + g.pix_off[a] + (int64_t)(o.y0 - wa[1]) * sa + (o.x0 - wa[0]);
  const float* Jb = J + g.pix_off[b] + (int64_t)(o.y0 - wb[1]) * sb + (o.x0 - wb[0]);
  const int64_t p0 = (int64_t)o.y0 * g.nx + o.x0;
  struct Px {
    float ja[NP], jb[NP], w;
    bool keep;
  };
  auto load = [&](Px& v) {
    v.keep = t.e < t.e1;
    const int x = v.keep ? t.x : 0, y = v.keep ? t.y : 0;  // past the end: the corner, read and not used
    const int64_t p = p0 + (int64_t)y * g.nx + x;
    const float* pa = Ja + (int64_t)y * sa + x;
    const float* pb = Jb + (int64_t)y * sb + x;
    v.w = weight ? weight[p] : 1.0f;
    if (mask) v.keep &= mask[p] == 0;
#pragma unroll
    for (int k = 0; k < NP; ++k) v.ja[k] = pa[(int64_t)k * g.nsrcpix];
#pragma unroll
    for (int k = 0; k < NP; ++k) v.jb[k] = pb[(int64_t)k * g.nsrcpix];
  };
  if (t.e1 > 0) {
    Px cur;
    load(cur);
    for (int64_t left = t.e1 - (t.e - threadIdx.x); left > 0; left -= 256) {
      t.next();
      Px nxt;
      load(nxt);
      if (cur.keep) {
#pragma unroll
        for (int k = 0; k < NP; ++k) {
          const double ja = (double)cur.w * (double)cur.ja[k];
#pragma unroll
          for (int l = 0; l < NP; ++l) acc[k * NP + l] += ja * (double)cur.jb[l];
        }
      }
      cur = nxt;
    }
  }
  wave_sums(acc, red[threadIdx.x >> 6]);
  __syncthreads();
  if (threadIdx.x < NN) {
    const int k = threadIdx.x;
    const double v = red[0][k] + red[1][k] + red[2][k] + red[3][k];
    if (kOne) pair_entry(g, a, b, k, v, H);
    else part[(int64_t)blockIdx.x * NN + k] = v;
  }
}

// the pair's pieces, in order
__global__ __launch_bounds__(64) void group_pair_final_kernel(apx_group g, int S, const double* __restrict__ part,
                                                              double* __restrict__ H) {
  constexpr int NP = APX_BATCH_NP, NN = NP * NP;
  if (threadIdx.x >= NN) return;
  const int a = g.pair[2 * blockIdx.x], b = g.pair[2 * blockIdx.x + 1];
  const Overlap o(g.win + 4 * a, g.win + 4 * b);
  const int np = pieces_of((int64_t)o.ow * o.oh, S);
  double v = 0.0;
  for (int q = 0; q < np; ++q) v += part[((int64_t)blockIdx.x * S + q) * NN + threadIdx.x];
  pair_entry(g, a, b, threadIdx.x, v, H);
}

// ---------------------------------------------------------------------------
// Dense float64 damped Cholesky: A(L)_ii = H_ii + L (1 + H_ii), A(L)_ij =
// H_ij / (1 + L) (fit/lm.py:359-371), factor A = L L^T in place (lower
// triangle), then solve L L^T x = b.

__global__ __launch_bounds__(256) void damp_kernel(const double* __restrict__ H, int n, double L,
                                                   double* __restrict__ A) {
  const int64_t nn = (int64_t)n * n;
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nn; e += (int64_t)gridDim.x * 256) {
    const int i = (int)(e / n), j = (int)(e % n);
    const double v = H[e];
    // the entry (k0, k0 + 1) of each diagonal block seeds its envelope slot
    A[e] = (i == j) ? v + L * (1.0 + v) : (j == i + 1 && i % kNB == 0) ? __hiloint2double(0, i) : v / (1.0 + L);
  }
}

// One launch a panel of kNB = 32 columns.  A panel's own chain (the diagonal
// block's factor, then the rows below) is serial, so the update of everything
// to its right runs beside the next panel: launch k takes panel k - 1 out of
// block column k and factors it (the first workgroups), and takes panel k - 1
// out of the block columns after it (the others).  Two launches a panel, with
// the rows solved after the diagonal factor and a division a step, took 20 + 11 us a
// panel (n = 3501, a band 658 wide: 3.45 ms a factor); this one 10.2 us (1.13 ms).
typedef double v4d __attribute__((ext_vector_type(4)));

// 16 x 16 blocks by v_mfma_f64_16x16x4_f64: lane l gives A[l % 16][l / 16] and
// B[l / 16][l % 16] of a k-step of 4, and holds D[4 r + l / 16][l % 16] in acc[r].
constexpr int kSteps = kNB / 4;  // k-steps of a panel

// k-step operands of rows r0 .. r0 + 15 of the panel at column p0 (zero past the matrix)
__device__ __forceinline__ void panel_operand(const double* __restrict__ A, int n, int r0, int p0, double (&o)[kSteps]) {
  const int lane = threadIdx.x & 63, row = r0 + (lane & 15);
#pragma unroll
  for (int t = 0; t < kSteps; ++t) o[t] = row < n ? A[(int64_t)row * n + p0 + 4 * t + (lane >> 4)] : 0.0;
}

// Rows of block column k0 with panel k0 - kNB taken out, into T: a wave's 16
// rows r0 .. (T rows 16 w ..) by the block's 32 columns.  Here and in
// trailing_tile a panel's 32 products are summed from zero and subtracted once:
// added into the entry itself, each would round at the entry's size, and
// |L L^T - A| grew with sqrt(n) in place of sqrt(n / 32) (dense, n = 701: 7.6e-16
// of |A| in place of 2.0e-16).
__device__ __forceinline__ void panel_rows(const double* __restrict__ A, int n, int k0, int nb, int r0, int w,
                                           double (*T)[kNB + 1]) {
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  v4d c[2];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = r0 + 4 * r + lk, col = 16 * q + li;
      // lower triangle: workgroup 0 of the launch writes the block's upper one
      c[q][r] = (row < n && col < nb && k0 + col <= row) ? A[(int64_t)row * n + k0 + col] : 0.0;
    }
  if (k0 > 0) {
    double a[kSteps], b[2][kSteps];
    panel_operand(A, n, r0, k0 - kNB, a);
    panel_operand(A, n, k0, k0 - kNB, b[0]);
    panel_operand(A, n, k0 + 16, k0 - kNB, b[1]);
    v4d sum[2] = {};
#pragma unroll
    for (int t = 0; t < kSteps; ++t)
#pragma unroll
      for (int q = 0; q < 2; ++q) sum[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b[q][t], sum[q], 0, 0, 0);
#pragma unroll
    for (int q = 0; q < 2; ++q) c[q] -= sum[q];
  }
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) T[16 * w + 4 * r + lk][16 * q + li] = c[q][r];
}

// Cholesky of a diagonal block and the solve of rows below it, in T (rows 0 ..
// 31 the block, the others rows further down), by a workgroup whose wave w holds
// T's rows 16 w ...  Wave 0 takes a row a lane: the rows below take the block's
// own steps (column j: divided by the pivot's root, then out of the later
// columns), so they cost nothing beyond the factor.  Column entries go lane to
// lane by v_readlane, two a multiply-add, so only the steps within 16 columns go
// this way; the first 16 columns leave the last 16 by MFMA, every wave its rows
// (all 32 columns by lane reads: 11.8 us a panel; this way 10.2).
// 1 / sqrt(pivot) is v_rsq_f64 (24 bits) and one third-order step, within 2 ulp,
// and a quotient takes one more step from it (rounded as a division's: without
// it |L L^T - A| of systems up to 16 wide is 4 to 10 % larger; it takes 1 % of
// the factor's time): a division and a square root a step, 60 dependent
// instructions, set the chain's length before.  T[i][k] = L[i][k] on return (k <= i).  A pivot that is
// not positive and finite gives NaN and sets *status to its 1-based column
// (first one only, when `report`).
constexpr int kHB = kNB / 2;

template <bool kFull>
__device__ __forceinline__ int potrf_half(int nb, int j0, double (&r)[kHB]) {
  const int lane = threadIdx.x & 63;
  int bad = -1;
#pragma unroll
  for (int j = 0; j < kHB; ++j) {
    if (kFull || j0 + j < nb) {  // uniform; constant trip counts keep r[] in registers
      const double piv = lane_bcast(r[j], j0 + j);
      const bool ok = piv > 0.0 && isfinite(piv);
      bad = (!ok && bad < 0) ? j0 + j : bad;
      const double p = ok ? piv : __builtin_nan("");
      double y = __builtin_amdgcn_rsq(p);
      const double e = fma(-p * y, y, 1.0);
      y = fma(y * e, fma(0.375, e, 0.5), y);
      double d = p * y;
      d = fma(fma(-d, d, p), 0.5 * y, d);
      const double q = r[j] * y;
      r[j] = lane == j0 + j ? d : fma(fma(-q, d, r[j]), y, q);
      // every lane updates every later column: entries above the diagonal
      // (k > lane) and columns past nb are never used, and only lower entries of
      // columns before k feed a lower entry
#pragma unroll
      for (int k = j + 1; k < kHB; ++k) r[k] = fma(-r[j], lane_bcast(r[j], j0 + k), r[k]);
    }
  }
  return bad;
}

template <bool kFull>
__device__ __forceinline__ void factor_rows(double (*T)[kNB + 1], int rows, int k0, int nb, int32_t* __restrict__ status,
                                            bool report) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  int bad = -1;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    __syncthreads();
    if (h == 1) {
      const double(*R)[kNB + 1] = T + 16 * w;
      v4d c, sum = {};
#pragma unroll
      for (int q = 0; q < 4; ++q) c[q] = R[4 * q + lk][kHB + li];
#pragma unroll
      for (int t = 0; t < kHB / 4; ++t)
        sum = __builtin_amdgcn_mfma_f64_16x16x4f64(R[li][4 * t + lk], T[kHB + li][4 * t + lk], sum, 0, 0, 0);
#pragma unroll
      for (int q = 0; q < 4; ++q) T[16 * w + 4 * q + lk][kHB + li] = c[q] - sum[q];
      __syncthreads();
    }
    if (w == 0) {
      double r[kHB];
#pragma unroll
      for (int k = 0; k < kHB; ++k) r[k] = lane < rows ? T[lane][kHB * h + k] : 0.0;
      const int b = potrf_half<kFull>(nb, kHB * h, r);
      bad = (b >= 0 && bad < 0) ? b : bad;
      if (lane < rows) {
#pragma unroll
        for (int k = 0; k < kHB; ++k) T[lane][kHB * h + k] = r[k];
      }
    }
  }
  __syncthreads();
  if (report && bad >= 0 && threadIdx.x == 0 && status[0] == 0) status[0] = k0 + bad + 1;
}

// 64 x 64 tile (ti, tj) of the update by panel p0 of the lower triangle from
// row and column `base` on: A[i][j] -= sum_t L[i][p0 + t] L[j][p0 + t]
__device__ __forceinline__ void trailing_tile(double* __restrict__ A, int n, int p0, int i0, int j0) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const int r0 = i0 + 16 * w;
  v4d c[4];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = r0 + 4 * r + lk, j = j0 + 16 * q + li;
      c[q][r] = (i < n && j <= i) ? A[(int64_t)i * n + j] : 0.0;
    }
  double a[kSteps], b[4][kSteps];
  panel_operand(A, n, r0, p0, a);
#pragma unroll
  for (int q = 0; q < 4; ++q) panel_operand(A, n, j0 + 16 * q, p0, b[q]);
  v4d sum[4] = {};
#pragma unroll
  for (int t = 0; t < kSteps; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) sum[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b[q][t], sum[q], 0, 0, 0);
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = r0 + 4 * r + lk, j = j0 + 16 * q + li;
      if (i < n && j <= i) A[(int64_t)i * n + j] = c[q][r] - sum[q][r];
    }
}

// Envelope of the damped matrix: for each 32-row block, the first column
// holding a nonzero entry of the block's rows (lower triangle).  A Cholesky
// factor has no fill before a row's first nonzero entry, so the block's rows of
// L are exactly zero in every earlier panel.  The column is kept as an int in
// the low half of the block's diagonal-block entry (k0, k0 + 1) of the upper
// triangle, which the factor neither reads nor writes before that block's own
// panel writes L^T there; damp_kernel seeds it with k0, and each workgroup of
// envelope_kernel (a block x a chunk of kEnvCols columns) lowers it to the
// first nonzero column of its chunk.  A block of one row has no such entry and
// counts as reaching every panel.  A NaN counts as nonzero.
constexpr int kEnvCols = 512;

__device__ __forceinline__ int* envelope_slot(double* A, int n, int k0) {
  return reinterpret_cast<int*>(A + (int64_t)k0 * n + k0 + 1);
}

__global__ __launch_bounds__(256) void envelope_kernel(double* __restrict__ A, int n) {
  __shared__ int wmin[4];
  const int k0 = blockIdx.x * kNB, nb = min(kNB, n - k0);
  const int c0 = blockIdx.y * kEnvCols;
  if (nb < 2 || c0 >= k0) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // thread: columns c0 + lane + 64 q, rows w + 4 r
  int best = 1 << 30;
#pragma unroll
  for (int q = 0; q < kEnvCols / 64; ++q) {
    const int c = c0 + lane + 64 * q;
#pragma unroll
    for (int r = 0; r < kNB / 4; ++r) {
      const int row = w + 4 * r;
      if (c < k0 && row < nb && A[(int64_t)(k0 + row) * n + c] != 0.0) best = min(best, c);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) best = min(best, __shfl_xor(best, o, 64));
  if (lane == 0) wmin[w] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    best = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3]));
    if (best < (1 << 30)) atomicMin(envelope_slot(A, n, k0), best);
  }
}

// first panel that block `blk`'s rows reach (envelope_kernel); past the
// matrix: never
__device__ __forceinline__ int block_reach(const double* __restrict__ A, int n, int blk) {
  const int k0 = blk * kNB;
  if (k0 >= n) return 1 << 30;
  if (n - k0 < 2) return 0;
  return *reinterpret_cast<const int*>(A + (int64_t)k0 * n + k0 + 1) / kNB;
}

// Launch of panel k0: workgroups 0 .. row_wgs - 1 take the diagonal block and 32
// rows below it each (every one factors the diagonal block itself, the same
// operations on the same input, instead of waiting a launch for it); the others
// take the tiles of the trailing update by the panel before, those whose rows
// and columns all reach it: the update of the rest is exactly zero.  The
// diagonal block's lower triangle is left as it is, since other workgroups may
// still be reading it; workgroup 0 writes L^T into its strict upper triangle
// (read by the forward solve along columns), and diag_writeback_kernel writes
// the lower triangle and the diagonal once the whole factor is done.
template <bool kFull>
__global__ __launch_bounds__(256) void panel_kernel(double* __restrict__ A, int n, int k0, int row_wgs, int ntiles,
                                                    int32_t* __restrict__ status) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int nb = kFull ? kNB : min(kNB, n - k0);
  if ((int)blockIdx.x >= row_wgs) {
    // tiles b0, b0 + step, ...: a lane looks at one, then the workgroup takes those that are reached
    const int step = (int)gridDim.x - row_wgs, base = k0 + kNB, pk = k0 / kNB - 1;
    for (int b0 = (int)blockIdx.x - row_wgs; b0 < ntiles; b0 += 64 * step) {
      const int b = b0 + lane * step;
      int ti = 0, tj = 0;
      bool hit = false;
      if (b < ntiles) {  // tile (ti, tj), tj <= ti, of the linear index
        ti = (int)((sqrt(8.0 * b + 1.0) - 1.0) * 0.5);
        while ((ti + 1) * (ti + 2) / 2 <= b) ++ti;
        while (ti * (ti + 1) / 2 > b) --ti;
        tj = b - ti * (ti + 1) / 2;
        const int bi = (base + ti * kUT) / kNB, bj = (base + tj * kUT) / kNB;
        hit = min(block_reach(A, n, bi), block_reach(A, n, bi + 1)) <= pk &&
              min(block_reach(A, n, bj), block_reach(A, n, bj + 1)) <= pk;
      }
      for (uint64_t m = __ballot(hit); m; m &= m - 1) {
        const int l = __ffsll((unsigned long long)m) - 1;
        trailing_tile(A, n, k0 - kNB, base + __builtin_amdgcn_readlane(ti, l) * kUT,
                      base + __builtin_amdgcn_readlane(tj, l) * kUT);
      }
    }
    return;
  }
  __shared__ double T[2 * kNB][kNB + 1];
  const int i0 = k0 + nb + (int)blockIdx.x * kNB;
  panel_rows(A, n, k0, nb, w < 2 ? k0 + 16 * w : i0 + 16 * (w - 2), w, T);
  factor_rows<kFull>(T, 2 * kNB, k0, nb, status, blockIdx.x == 0);
#pragma unroll
  for (int e = t; e < kNB * kNB; e += 256) {
    const int p = e / kNB, q = e % kNB;
    if (i0 + p < n && q < nb) A[(int64_t)(i0 + p) * n + k0 + q] = T[kNB + p][q];
    if (i0 + q < n && p < nb) A[(int64_t)(k0 + p) * n + i0 + q] = T[kNB + q][p];  // L^T in the upper triangle
    if (blockIdx.x == 0 && p < q && q < nb) A[(int64_t)(k0 + p) * n + k0 + q] = T[q][p];
  }
}

// Lower triangle and diagonal of every diagonal block, a workgroup of two waves
// a block, after the factor: each block still holds what its own launch read
// (no later panel's update reaches it), and is factored again to the same bits.
__global__ __launch_bounds__(128) void diag_writeback_kernel(double* __restrict__ A, int n) {
  __shared__ double T[kNB][kNB + 1];
  const int t = threadIdx.x, w = t >> 6;
  const int k0 = blockIdx.x * kNB, nb = min(kNB, n - k0);
  panel_rows(A, n, k0, nb, k0 + 16 * w, w, T);
  if (nb == kNB) factor_rows<true>(T, kNB, k0, nb, nullptr, false);
  else factor_rows<false>(T, kNB, k0, nb, nullptr, false);
  for (int e = t; e < kNB * kNB; e += 128) {
    const int p = e / kNB, q = e % kNB;
    if (q <= p && p < nb) A[(int64_t)(k0 + p) * n + k0 + q] = T[p][q];
  }
}

// Triangular solves, two block columns a launch.  A launch takes the terms of
// the two blocks solved last out of every entry still to be solved (forward:
// rows of L^T, which the factor keeps in its upper triangle; backward: rows of
// L; both read coalesced along x), and its first wave then solves the next two
// diagonal blocks on registers, lanes 0-31 the first and lanes 32-63 the
// second.  Every entry receives the terms of the blocks one at a time, in
// block order, each summed from its first column.  All loads of a launch are
// issued before its first wait.  A wave has at most 63 in flight, so the terms of
// the first wave's own 64 rows are the second wave's work and reach it through
// LDS: with them (128 loads) and a product and two choices a step of the
// substitution, a launch took 8.4 us, n = 3501; now 5.4 (forward) and 6.0.

// One half-wave's copy of the diagonal block [k0, k0 + nb): lane off + r holds
// v[j] = A[(k0 + j) n + k0 + r], which is L[r][j] for j < r (the factor's
// transposed copy in the upper triangle) and L[j][r] for j > r, and its diagonal
// entry.  diag_ready clears the entries a solve does not use and takes the
// diagonal's reciprocal, so that a step of the solve is a product, two lane reads
// and an FMA, without a choice in the chain.  (Rows scaled by the reciprocal
// beforehand save the product of the chain, and round every entry of L once
// more: badly scaled 16 x 16 systems came out with twice the error.)
struct DiagBlock {
  double v[kNB];
  double rdii;
};

__device__ __forceinline__ void diag_load(const double* __restrict__ A, int n, int k0, int r, DiagBlock& d) {
  const int nb = min(kNB, n - k0);
  const bool in = r >= 0 && r < nb;
#pragma unroll
  for (int j = 0; j < kNB; ++j) d.v[j] = (in && j < nb) ? A[(int64_t)(k0 + j) * n + k0 + r] : 0.0;
  d.rdii = in ? A[(int64_t)(k0 + r) * n + k0 + r] : 1.0;
}

// kLower: keeps v[j] for j < r; else for j > r
template <bool kLower>
__device__ __forceinline__ void diag_ready(DiagBlock& d, int r) {
  d.rdii = 1.0 / d.rdii;
#pragma unroll
  for (int j = 0; j < kNB; ++j) d.v[j] = (kLower ? j < r : j > r) ? d.v[j] : 0.0;
}

// substitution with the diagonal block held by lanes off .. off + 31 (rows and
// columns past the matrix are zero): lane off + r holds the right-hand side of
// row r on entry and x_r on return; every other lane is left as it is
template <bool kLower>
__device__ __forceinline__ double diag_substitute(const DiagBlock& d, int off, double b) {
  const bool mine = ((int)(threadIdx.x & 63) & ~(kNB - 1)) == off;
  double xi = b;
#pragma unroll
  for (int q = 0; q < kNB; ++q) {
    const int j = kLower ? q : kNB - 1 - q;
    xi = fma(-d.v[j], lane_bcast(xi * d.rdii, off + j), xi);
  }
  return mine ? xi * d.rdii : b;
}

template <bool kLower>
__global__ __launch_bounds__(64) void diag_solve_kernel(const double* __restrict__ A, int n, int k0,
                                                        double* __restrict__ x) {
  DiagBlock d;
  const int lane = threadIdx.x, nb = min(kNB, n - k0);
  diag_load(A, n, k0, lane, d);
  diag_ready<kLower>(d, lane);
  const double b = lane < nb ? x[k0 + lane] : 0.0;
  const double xi = diag_substitute<kLower>(d, 0, b);
  if (lane < nb) x[k0 + lane] = xi;
}

// Forward step.  On entry blocks 0..b of x are final and every later entry
// holds b_i minus the terms of blocks 0..b-2.  The launch takes the terms of
// blocks b-1 (when b > 0) and b out of rows (b+1) kNB .. n-1.  Wave 0 of
// workgroup 0 holds blocks b+1 (lanes 0-31) and b+2 (lanes 32-63): it solves
// block b+1, takes block b+1's terms out of block b+2 and solves block b+2.
// Blocks b-1 and b are full, since rows follow them.
__global__ __launch_bounds__(256) void trsv_lower_pair_kernel(const double* __restrict__ A, int n, int b,
                                                              double* __restrict__ x) {
  __shared__ double xs[2 * kNB], vs[2 * kNB];
  const int nblk = (n + kNB - 1) / kNB;
  const int first = b > 0 ? b - 1 : b;
  const int c0 = first * kNB, nblocks = b - first + 1;
  const int t = threadIdx.x;
  const bool lead = blockIdx.x == 0 && t < 64;
  const int b1 = b + 1, b2 = b + 2;
  const bool has2 = b2 < nblk;
  // this thread's row: 256 a workgroup from b1 kNB - 64 on; the lead's lanes hold the
  // second wave's rows
  const int i = b1 * kNB + (lead ? t : (int)blockIdx.x * 256 + t - 64);
  const bool row = i < n;
  double v = 0.0;
  DiagBlock d;
  double l21[kNB];  // lanes 32-63: L[i][b1 kNB + u], row i in block b2
  if (lead) {
    const bool second = t >= kNB;
    diag_load(A, n, second ? b2 * kNB : b1 * kNB, (second && !has2) ? -1 : (t & (kNB - 1)), d);
#pragma unroll
    for (int u = 0; u < kNB; ++u) l21[u] = (second && row) ? A[(int64_t)(b1 * kNB + u) * n + i] : 0.0;
    diag_ready<true>(d, t & (kNB - 1));
    __syncthreads();
  } else {
    double c[2][kNB];
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int u = 0; u < kNB; ++u)
        c[k][u] = (row && k < nblocks) ? A[(int64_t)(c0 + k * kNB + u) * n + i] : 0.0;
    v = row ? x[i] : 0.0;
    const int e = t - 192;  // the last wave brings the solved entries
    if (e >= 0 && e < nblocks * kNB) xs[e] = x[c0 + e];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (k < nblocks) {
        double s = 0.0;
#pragma unroll
        for (int u = 0; u < kNB; ++u) s += c[k][u] * xs[k * kNB + u];
        v -= s;
      }
    }
    if (blockIdx.x == 0 && t < 128) vs[t - 64] = v;
    else if (row) x[i] = v;
  }
  __syncthreads();
  if (!lead) return;
  v = vs[t];
  v = diag_substitute<true>(d, 0, v);  // lanes 32-63 keep their right-hand sides
  if (has2) {
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < kNB; ++u) s += l21[u] * lane_bcast(v, u);
    if (t >= kNB) v -= s;
    v = diag_substitute<true>(d, kNB, v);
  }
  if (row) x[i] = v;
}

// Backward step.  On entry blocks b..nblk-1 of x are final and every earlier
// entry holds its value minus the terms of blocks b+2 and later.  The launch
// takes the terms of blocks b+1 (when it exists; it may be the partial last
// block) and b, in that order, out of rows 0 .. b kNB - 1.  Wave 0 of
// workgroup 0 holds blocks b-1 (lanes 0-31) and b-2 (lanes 32-63) in row
// order; the other threads take rows (b-2) kNB - 1 downwards.  The wave
// solves block b-1, takes its terms out of block b-2 and solves block b-2.
__global__ __launch_bounds__(256) void trsv_upper_pair_kernel(const double* __restrict__ A, int n, int b,
                                                              double* __restrict__ x) {
  __shared__ double xs[2 * kNB], vs[2 * kNB];
  const int nblk = (n + kNB - 1) / kNB;
  const bool hi = b + 1 < nblk;
  const int kh = (b + 1) * kNB, nbh = hi ? min(kNB, n - kh) : 0;
  const int kb = b * kNB, nbb = min(kNB, n - kb);
  const int t = threadIdx.x;
  const bool lead = blockIdx.x == 0 && t < 64;
  const int g = lead ? t : (int)blockIdx.x * 256 + t - 64;
  const int b1 = b - 1, b2 = b - 2;
  const bool has2 = b2 >= 0;
  const int i = g < kNB ? b1 * kNB + g : (g < 2 * kNB ? b2 * kNB + g - kNB : b2 * kNB + 2 * kNB - 1 - g);
  const bool row = i >= 0;
  double v = 0.0;
  DiagBlock d;
  double l12[kNB];  // lanes 32-63: L[b1 kNB + u][i], row i in block b2
  if (lead) {
    const bool second = t >= kNB;
    diag_load(A, n, second ? b2 * kNB : b1 * kNB, (second && !has2) ? -1 : (t & (kNB - 1)), d);
#pragma unroll
    for (int u = 0; u < kNB; ++u) l12[u] = (second && row) ? A[(int64_t)(b1 * kNB + u) * n + i] : 0.0;
    diag_ready<false>(d, t & (kNB - 1));
    __syncthreads();
  } else {
    double c[2][kNB];
#pragma unroll
    for (int u = 0; u < kNB; ++u) c[0][u] = (row && u < nbh) ? A[(int64_t)(kh + u) * n + i] : 0.0;
#pragma unroll
    for (int u = 0; u < kNB; ++u) c[1][u] = (row && u < nbb) ? A[(int64_t)(kb + u) * n + i] : 0.0;
    v = row ? x[i] : 0.0;
    const int e = t - 192;  // the last wave brings the solved entries
    if (e >= 0) xs[e] = e < kNB ? (e < nbh ? x[kh + e] : 0.0) : (e - kNB < nbb ? x[kb + e - kNB] : 0.0);
    __syncthreads();
    if (hi) {
      double s = 0.0;
#pragma unroll
      for (int u = 0; u < kNB; ++u)
        if (u < nbh) s += c[0][u] * xs[u];
      v -= s;
    }
    {
      double s = 0.0;
#pragma unroll
      for (int u = 0; u < kNB; ++u)
        if (u < nbb) s += c[1][u] * xs[kNB + u];
      v -= s;
    }
    if (blockIdx.x == 0 && t < 128) vs[t - 64] = v;
    else if (row) x[i] = v;
  }
  __syncthreads();
  if (!lead) return;
  v = vs[t];
  v = diag_substitute<false>(d, 0, v);  // lanes 32-63 keep their right-hand sides
  if (has2) {
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < kNB; ++u) s += l12[u] * lane_bcast(v, u);
    if (t >= kNB) v -= s;
    v = diag_substitute<false>(d, kNB, v);
  }
  if (row) x[i] = v;
}

__global__ void clear_status_kernel(int32_t* status) {
  if (threadIdx.x == 0) status[0] = 0;
}

__global__ void copy_kernel(const double* __restrict__ a, int n, double* __restrict__ b) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) b[i] = a[i];
}

int check_group(const apx_group* g) {
  if (!g || !g->win || !g->pix_off || !g->col0 || !g->tile_ptr || !g->tile_src || (g->npair > 0 && !g->pair))
    return set_error(APX_E_INVALID, "group: null array");
  if (g->nx < 1 || g->ny < 1 || g->nsrc < 1 || g->np < 1)
    return set_error(APX_E_INVALID, "group: empty image or no sources");
  if (g->ntx != (g->nx + kTW - 1) / kTW || g->nty != (g->ny + kTH - 1) / kTH)
    return set_error(APX_E_INVALID, "group: tile grid does not match the image");
  if (g->sky_col >= g->np) return set_error(APX_E_INVALID, "group: sky column out of range");
  return APX_OK;
}

int grid_for(int64_t n) { return (int)std::min<int64_t>((n + 255) / 256, 4096); }

}  // namespace

int group_image(const apx_group* g, const float* src, double sky, float* out, hipStream_t stream) {
  if (int rc = check_group(g)) return rc;
  if (!src || !out) return set_error(APX_E_INVALID, "group_image: null pointer");
  hipLaunchKernelGGL(group_image_kernel, dim3((unsigned)(g->ntx * g->nty)), dim3(256), 0, stream, *g, src,
                     sky, out);
  return check_launch("group_image");
}

static int64_t group_part_bytes(const apx_group* g) {
  const int64_t npix = (int64_t)g->nx * g->ny;
  const int S = max_pieces(*g, g->npair);
  return 8 * std::max(npix, S == 1 ? 0 : (int64_t)g->npair * S * APX_BATCH_NP * APX_BATCH_NP);
}

int64_t group_workspace_bytes(const apx_group* g) {
  if (!g) return 0;
  // [u of group_rpp, or the pair partials | image partials | source partials]
  return group_part_bytes(g) + 8 * 2 * 4096 + 8 * 2 * APX_BATCH_NP * (int64_t)g->nsrc * max_pieces(*g, g->nsrc) + 256;
}

int group_normal(const apx_group* g, const float* J, const float* model, const float* data,
                 const float* weight, const uint8_t* mask, double sky_dcol, double* H, double* grad,
                 void* ws, int64_t ws_bytes, hipStream_t stream) {
  if (int rc = check_group(g)) return rc;
  if (!J || !model || !data || !H || !grad || !ws) return set_error(APX_E_INVALID, "group_normal: null pointer");
  if (ws_bytes < group_workspace_bytes(g)) return set_error(APX_E_INVALID, "group_normal: workspace too small");
  const int64_t np2 = (int64_t)g->np * g->np;
  hipLaunchKernelGGL(fill_kernel, dim3(grid_for(np2)), dim3(256), 0, stream, H, np2, 0.0);
  hipLaunchKernelGGL(fill_kernel, dim3(grid_for(g->np)), dim3(256), 0, stream, grad, (int64_t)g->np, 0.0);
  double* part = reinterpret_cast<double*>(static_cast<char*>(ws) + group_part_bytes(g));
  double* spart = part + 2 * 4096;
  if (g->npair > 0) {
    const int S = max_pieces(*g, g->npair);
    double* pp = static_cast<double*>(ws);
    auto* kernel = S == 1 ? &group_pair_kernel<true> : &group_pair_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)g->npair * S), dim3(256), 0, stream, *g, J, weight, mask, S, pp, H);
    if (S > 1)
      hipLaunchKernelGGL(group_pair_final_kernel, dim3((unsigned)g->npair), dim3(64), 0, stream, *g, S,
                         (const double*)pp, H);
  }
  const int S = max_pieces(*g, g->nsrc);
  auto* kernel = S == 1 ? &group_source_kernel<true> : &group_source_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)g->nsrc * S), dim3(256), 0, stream, *g, J, model, data, weight, mask, S, spart,
                     sky_dcol, H, grad);
  if (S > 1)
    hipLaunchKernelGGL(group_source_final_kernel, dim3((unsigned)((2 * APX_BATCH_NP * g->nsrc + 255) / 256)), dim3(256),
                       0, stream, *g, S, sky_dcol, (const double*)spart, H, grad);
  if (g->sky_col >= 0) {
    const int64_t npix = (int64_t)g->nx * g->ny;
    const int nb = std::min(grid_for(npix), 512);
    hipLaunchKernelGGL(group_image_sums_kernel, dim3(nb), dim3(256), 0, stream, npix, 0, model, data, weight,
                       mask, (const double*)nullptr, part);
    hipLaunchKernelGGL(group_sky_final_kernel, dim3(1), dim3(256), 0, stream, nb, 0, g->np, g->sky_col, sky_dcol,
                       part, H, grad);
  }
  return check_launch("group_normal");
}

int group_rpp(const apx_group* g, const float* J, const float* m0, const float* m1, const float* weight,
              const uint8_t* mask, const double* h, double d, double sky_dcol, double* out, void* ws,
              int64_t ws_bytes, hipStream_t stream) {
  if (int rc = check_group(g)) return rc;
  if (!J || !m0 || !m1 || !h || !out || !ws) return set_error(APX_E_INVALID, "group_rpp: null pointer");
  if (ws_bytes < group_workspace_bytes(g)) return set_error(APX_E_INVALID, "group_rpp: workspace too small");
  const int64_t npix = (int64_t)g->nx * g->ny;
  double* u = static_cast<double*>(ws);
  double* part = reinterpret_cast<double*>(static_cast<char*>(ws) + group_part_bytes(g));
  double* spart = part + 2 * 4096;
  hipLaunchKernelGGL(group_rpp_weights_kernel, dim3((unsigned)(g->ntx * g->nty)), dim3(256), 0, stream, *g, J,
                     m0, m1, weight, mask, h, d, sky_dcol, u);
  const int S = max_pieces(*g, g->nsrc);
  hipLaunchKernelGGL(group_jtv_kernel, dim3((unsigned)g->nsrc * S), dim3(256), 0, stream, *g, J, (const double*)u,
                     S, spart, out);
  if (S > 1)
    hipLaunchKernelGGL(group_jtv_final_kernel, dim3((unsigned)((APX_BATCH_NP * g->nsrc + 255) / 256)), dim3(256), 0,
                       stream, *g, S, (const double*)spart, out);
  if (g->sky_col >= 0) {
    const int nb = std::min(grid_for(npix), 512);
    hipLaunchKernelGGL(group_image_sums_kernel, dim3(nb), dim3(256), 0, stream, npix, 1, (const float*)nullptr,
                       (const float*)nullptr, (const float*)nullptr, (const uint8_t*)nullptr, (const double*)u,
                       part);
    hipLaunchKernelGGL(group_sky_final_kernel, dim3(1), dim3(256), 0, stream, nb, 1, g->np, g->sky_col, sky_dcol,
                       part, (double*)nullptr, out);
  }
  return check_launch("group_rpp");
}

int dense_damped_factor(int32_t n, const double* H, double L, double* A, int32_t* status, hipStream_t stream) {
  if (!H || !A || !status) return set_error(APX_E_INVALID, "dense_factor: null pointer");
  if (n < 1) return set_error(APX_E_INVALID, "dense_factor: n < 1");
  const int64_t nn = (int64_t)n * n;
  hipLaunchKernelGGL(damp_kernel, dim3(grid_for(nn)), dim3(256), 0, stream, H, n, L, A);
  hipLaunchKernelGGL(clear_status_kernel, dim3(1), dim3(64), 0, stream, status);
  hipLaunchKernelGGL(envelope_kernel, dim3((unsigned)((n + kNB - 1) / kNB), (unsigned)((n + kEnvCols - 1) / kEnvCols)),
                     dim3(256), 0, stream, A, n);
  for (int k0 = 0; k0 < n; k0 += kNB) {
    const int nb = std::min(kNB, n - k0);
    const int rest = n - k0 - nb, T = k0 > 0 ? (rest + kUT - 1) / kUT : 0, tiles = T * (T + 1) / 2;
    const int rows = std::max(1, (rest + kNB - 1) / kNB);
    const dim3 grid((unsigned)(rows + std::min(tiles, 1024)));
    if (nb == kNB) hipLaunchKernelGGL(panel_kernel<true>, grid, dim3(256), 0, stream, A, n, k0, rows, tiles, status);
    else hipLaunchKernelGGL(panel_kernel<false>, grid, dim3(256), 0, stream, A, n, k0, rows, tiles, status);
  }
  hipLaunchKernelGGL(diag_writeback_kernel, dim3((unsigned)((n + kNB - 1) / kNB)), dim3(128), 0, stream, A, n);
  return check_launch("dense_factor");
}

int dense_cholesky_solve(int32_t n, const double* A, const double* b, double* x, hipStream_t stream) {
  if (!A || !b || !x) return set_error(APX_E_INVALID, "dense_solve: null pointer");
  if (n < 1) return set_error(APX_E_INVALID, "dense_solve: n < 1");
  hipLaunchKernelGGL(copy_kernel, dim3(grid_for(n)), dim3(256), 0, stream, b, n, x);
  const int nblk = (n + kNB - 1) / kNB;
  // forward: block 0's diagonal solve, then two blocks a launch
  hipLaunchKernelGGL(diag_solve_kernel<true>, dim3(1), dim3(64), 0, stream, A, n, 0, x);
  for (int blk = 0; blk + 1 < nblk; blk += 2) {
    const int rest = n - (blk + 1) * kNB;
    hipLaunchKernelGGL(trsv_lower_pair_kernel, dim3((unsigned)((rest + 64 + 255) / 256)), dim3(256), 0, stream, A, n,
                       blk, x);
  }
  // backward: the last block's diagonal solve, then two blocks a launch
  hipLaunchKernelGGL(diag_solve_kernel<false>, dim3(1), dim3(64), 0, stream, A, n, (nblk - 1) * kNB, x);
  for (int blk = nblk - 1; blk >= 1; blk -= 2)
    hipLaunchKernelGGL(trsv_upper_pair_kernel, dim3((unsigned)((blk * kNB + 64 + 255) / 256)), dim3(256), 0, stream, A,
                       n, blk, x);
  return check_launch("dense_solve");
}

}  // namespace apx
