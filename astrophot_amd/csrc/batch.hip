// Batched independent fits on gfx950: thousands of cutouts, one Sersic each,
// fitted by the reference's Levenberg-Marquardt entirely on the device.
//
// Every fit keeps its LM state in device memory (GalState) and advances in
// lock-step "ticks".  A tick is a fixed launch sequence over device-built work
// lists (so it can be captured in a HIP graph):
//   Jacobian stage (fits starting a step):   render value + 5 partial planes,
//       convolve with K, dK/dcx, dK/dcy -> model0 and J (parameter-major, 7 x npix),
//       J^T W J, J^T W (Y - m0), chi2(m0)                 (fit/lm.py:256-260)
//   lm_begin: step bookkeeping                              (lm.py:261-267)
//   lm_solve_h: damped float64 solve, probe point x + 0.1 h and trial point
//       x + h (the reference's x + h + a * acceleration, acceleration 0)
//                                                           (lm.py:269-277, 289)
//   probe stage: value render at x + 0.1 h, then rpp; beside it, on a second
//       stream, the trial stage: value render at x + h, then chi2
//   lm_solve_a + lm_decide (one kernel): rpp and chi2 from the two renders'
//       tile sums, a = -A(L)^-1 rpp / 2                     (lm.py:281-286)
//   lm_decide: the accept / reject / damping logic of one sub-step, and at the
//       end of a step the fit()-level update and convergence tests
//                                                 (lm.py:293-357, 461-485)
// A fit that finishes stops appearing in the work lists.  Renders use the same
// per-pixel device code as the single-component path (render_common.h,
// conv_common.h), so a batched fit evaluates exactly what the plain path does.
#include <hip/hip_runtime.h>

#include <cmath>

#include "capi_internal.h"
#include "conv_common.h"
#include "profile.h"
#include "render_common.h"

namespace apx {

namespace {

constexpr int NP = APX_BATCH_NP;
constexpr int kChunk = 256;
constexpr int kPersist = 2048;
constexpr int kNChan = 6;  // value + q, PA, n, Re, Ie partials
// Ie enters the Sersic profile only as the amplitude 10**Ie (sersic_model.py:
// 61-91), so d model / d Ie = ln(10) model: the Jacobian-stage convolutions
// skip the Ie plane and write its column from the value (times d Ie / d rep).
constexpr int kConvChan = kNChan - 1;
constexpr int kTR = 16;      // output rows of a batch tile (64 x kTR pixels)
// separable-convolution tap vectors are zero-padded to a multiple of 4 taps
__host__ __device__ inline int sp_k4(int k) { return (k + 3) & ~3; }
constexpr int kMfmaMax = kMfmaWide;  // widest kernel the MFMA convolution takes (67, up to 70 KiB LDS)

enum : int32_t { PH_INIT = 0, PH_NEEDJ = 1, PH_SUB = 2, PH_DONE = 3 };
enum : int32_t { ST_JAC = 0, ST_PROBE = 1, ST_TRIAL = 2, ST_ALL = 3, ST_ALL_JAC = 4 };
enum : int32_t { DIR_NONE = 0, DIR_BETTER = 1, DIR_WORSE = 2 };
enum : int32_t { S_RUN = 0, S_SUCCESS = 1, S_IMMOBILE = 2, S_NOSTEP = 3, S_MAXITER = 4, S_SKIPPED = 5 };

struct GalState {
  double x[8], ev[8];
  double L, init_chi2;
  double hist[10];
  double res_chi2, res_x[8];
  double best_dx[8], best_chi2, best_L;
  double scary_dx[8], scary_chi2, scary_L;
  double H[NP * NP], g[NP], h[8], a[8], ha[8], rpp[8];
  double chi2_m0, chi2, ndf;
  double fb[8];  // fallback start (representation), armed when fb_state == 1
  double ev2[8];  // the trial point x + h of the current sub-step
  int32_t nhist, iter, scary_valid, nostep, direction, sub, phase, status;
  int32_t fb_state, iter_total;  // fallback: 0 none, 1 armed, 2 ran; iterations of earlier runs
};

struct GalEval {
  Prof<float> pf;
  Prof<double> pd;
  double thr;
  double dvdr[NP];
  double sx, sy;  // sub-pixel shift of the PSF (model_object.py:320-325)
  int32_t nxw, nyw, ci, cj, bx, by;
};

struct Scratch {
  int32_t* cnt;       // [0] fits, [1] chunks, [2] tiles, [3] level-2 pixels,
                      // [4] selection redos, [5] level-2 redos
  int32_t* gal_list;  // ngal
  int2* chunk_list;   // nchunk
  int2* tile_list;    // ntile
  int32_t* gal_cnt;   // ngal: pixels each fit sends to the level-2 quadrature
  int32_t* deep;      // nwork: per-fit segments (at work_off) of those pixels
  int2* dq;           // nwork: the same pixels as one list of (fit, pixel)
  int2* rq;           // nwork: the redo list in the same form
  int32_t* gal_rcnt;  // ngal: pixels each fit sends to a float64 redo pass
  int32_t* redo;      // nwork: per-fit segments of those pixels
  float* mid;         // nwork: midpoint samples
  double* part;       // ntile * kPart: per-tile partial sums of the reductions
  GalEval* ev;        // ngal
};

constexpr int kPart = 64;  // doubles per tile partial (49 H + 7 g + 1 chi2 fit the largest)

__host__ __device__ inline int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }

// The scratch holds two copies of the work lists: the second, with its own
// plane-0 and tap buffers, serves the LM tick's trial render, which runs
// beside the probe render on a second stream.
struct TrialBranch {
  Scratch s;
  float* planes;  // nwork: the value plane
  float* taps;    // ntap
};

__host__ inline int64_t scratch_layout(const apx_batch& b, Scratch* s, TrialBranch* tb = nullptr) {
  char* p = static_cast<char*>(b.scratch);
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    char* q = p ? p + off : nullptr;
    off += align256(bytes);
    return q;
  };
  for (int copy = 0; copy < 2; ++copy) {
  Scratch t;
  t.cnt = reinterpret_cast<int32_t*>(take(256));
  t.gal_list = reinterpret_cast<int32_t*>(take(4 * (int64_t)b.ngal));
  t.chunk_list = reinterpret_cast<int2*>(take(8 * b.nchunk));
  t.tile_list = reinterpret_cast<int2*>(take(8 * b.ntile));
  t.gal_cnt = reinterpret_cast<int32_t*>(take(4 * (int64_t)b.ngal));
  t.deep = reinterpret_cast<int32_t*>(take(4 * b.nwork));
  t.dq = reinterpret_cast<int2*>(take(8 * b.nwork));
  t.rq = reinterpret_cast<int2*>(take(8 * b.nwork));
  t.gal_rcnt = reinterpret_cast<int32_t*>(take(4 * (int64_t)b.ngal));
  t.redo = reinterpret_cast<int32_t*>(take(4 * b.nwork));
  t.mid = reinterpret_cast<float*>(take(4 * b.nwork));
  t.part = reinterpret_cast<double*>(take(8 * kPart * b.ntile));
  t.ev = reinterpret_cast<GalEval*>(take((int64_t)sizeof(GalEval) * b.ngal));
  if (copy == 0 && s) *s = t;
  if (copy == 1 && tb) tb->s = t;
  }
  float* planes2 = reinterpret_cast<float*>(take(4 * b.nwork));
  float* taps2 = reinterpret_cast<float*>(take(4 * b.ntap));
  if (tb) {
    tb->planes = planes2;
    tb->taps = taps2;
  }
  return off;
}

__host__ inline Scratch carve(const apx_batch& b) {
  Scratch s;
  scratch_layout(b, &s);
  return s;
}

__host__ int64_t scratch_bytes(const apx_batch& b) {
  apx_batch c = b;
  c.scratch = nullptr;
  return scratch_layout(c, nullptr);
}

__device__ __forceinline__ GalState* st_of(const apx_batch& b, int g) {
  return reinterpret_cast<GalState*>(b.state) + g;
}

// ---------------------------------------------------------------------------
// work lists
__global__ void reset_kernel(int32_t* cnt) {
  if (threadIdx.x < 8) cnt[threadIdx.x] = 0;
}

// ---------------------------------------------------------------------------
// parameter maps (utils/conversions/optimization.py:17-54) for
// [cx, cy, q (0,1), PA cyclic (0,pi), n (0.36,8), Re (0,inf), Ie]
__device__ inline void rep_to_values(const double* r, double* v, double* dvdr) {
  v[0] = r[0];
  v[1] = r[1];
  v[2] = (atan(r[2]) + kPi / 2) * 1.0 / kPi;
  v[3] = r[3] - kPi * floor(r[3] / kPi);
  v[4] = (atan(r[4]) + kPi / 2) * (8.0 - 0.36) / kPi + 0.36;
  v[5] = (r[5] + sqrt(r[5] * r[5] + 4.0)) * 0.5;
  v[6] = r[6];
  dvdr[0] = dvdr[1] = dvdr[3] = dvdr[6] = 1.0;
  dvdr[2] = 1.0 / (kPi * (r[2] * r[2] + 1.0));
  dvdr[4] = (8.0 - 0.36) / (kPi * (r[4] * r[4] + 1.0));
  dvdr[5] = 0.5 + 0.5 * r[5] / sqrt(r[5] * r[5] + 4.0);
}

// Render constants of fit g at its parameters (rep_override row g when given), in
// parts that different waves take: the geometry, the profile in float64, the
// profile in float32, and the threshold with the parameter derivatives.
enum : int { EVAL_GEOMETRY = 0, EVAL_PROFD = 1, EVAL_PROFF = 2, EVAL_FLUX = 3 };

__device__ __forceinline__ void eval_fit(const apx_batch& b, const Scratch& s, int g, const double* rep_override, int stage,
                                         int part) {
  const apx_batch_galaxy G = b.gal[g];
  const double* rep = rep_override ? rep_override + (int64_t)g * NP
                                   : (stage == ST_TRIAL ? st_of(b, g)->ev2 : st_of(b, g)->ev);
  double v[NP], dvdr[NP];
  rep_to_values(rep, v, dvdr);
  const int bx = (G.pw + 1) / 2, by = (G.ph + 1) / 2;  // psf_image.py:71-93
  const int nxw = G.nx + 2 * bx, nyw = G.ny + 2 * by;
  const double det = b.P[0] * b.P[3] - b.P[1] * b.P[2];
  const double prm[3] = {v[4], v[5], v[6]};
  const double area = fabs(det);
  GalEval* e = s.ev + g;
  if (part == EVAL_GEOMETRY) {
    const double Pi[4] = {b.P[3] / det, -b.P[1] / det, -b.P[2] / det, b.P[0] / det};
    const double dx = v[0] - G.origin[0], dy = v[1] - G.origin[1];
    const double pcx = Pi[0] * dx + Pi[1] * dy + (-0.5 + bx);
    const double pcy = Pi[2] * dx + Pi[3] * dy + (-0.5 + by);
    const double ci = rint(pcx), cj = rint(pcy);  // ties to even
    e->sx = pcx - ci;
    e->sy = pcy - cj;
    e->nxw = nxw;
    e->nyw = nyw;
    e->ci = (int)ci;
    e->cj = (int)cj;
    e->bx = bx;
    e->by = by;
  } else if (part == EVAL_PROFD) {
    e->pd = make_prof<double>(APX_SERSIC, b.P, 0.0, 0.0, area, b.softening, v[2], v[3], prm);
  } else if (part == EVAL_PROFF) {
    e->pf = make_prof<float>(APX_SERSIC, b.P, 0.0, 0.0, area, b.softening, v[2], v[3], prm);
  } else {
    const double bn = sersic_b(v[4]);
    const double flux = 2.0 * kPi * pow(10.0, v[6]) * v[5] * v[5] * v[2] * v[4] * exp(bn) *
                        pow(bn, -2.0 * v[4]) * exp(lgamma(2.0 * v[4]));  // functions.py:168-190
    e->thr = b.tolerance * flux / (G.ref_npix > 0 ? (double)G.ref_npix : (double)nxw * nyw);
    for (int q = 0; q < NP; ++q) e->dvdr[q] = dvdr[q];
  }
}

// the exclusive prefix of n over the wave plus a base reserved on `counter`
// for the wave's total (one atomic a wave; every lane of the wave calls it)
__device__ __forceinline__ int wave_reserve(int n, int32_t* counter, int lane) {
  int x = n;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  const int tot = __shfl(x, 63, 64);
  int base = 0;
  if (lane == 63 && tot > 0) base = atomicAdd(counter, tot);
  return __shfl(base, 63, 64) + x - n;
}

// Work lists of the fits active in `stage`: the fit, its render chunks and its
// output tiles are appended (each fit's chunks and tiles contiguous and in order),
// its per-fit counts cleared, and its render constants evaluated.  Bound by one
// fit's chain of float64 functions, so a workgroup takes 64 fits and its four
// waves a part of their constants each; the first also writes the lists, the wave
// together one fit after another (a thread a fit took 700 stores in series for a
// 420 x 420 window): 256 uneven fits 33 -> 17 us, 125 windows of up to 420^2 48 -> 20.
__global__ __launch_bounds__(256) void build_kernel(apx_batch b, Scratch s, int stage, const double* rep_override) {
  const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
  const int g = blockIdx.x * 64 + lane;
  bool active = false;
  int nch = 0, ntl = 0;
  if (g < b.ngal) {
    if (part == 0) {
      s.gal_cnt[g] = 0;
      s.gal_rcnt[g] = 0;
    }
    const GalState* st = st_of(b, g);
    const int ph = st->phase;
    // the probe point's rpp only enters the step through the acceleration
    // term, which lm.py:283-286 zeroes for L <= 1e-4: such fits skip the probe
    active = stage == ST_ALL || stage == ST_ALL_JAC ||
             (stage == ST_JAC     ? (ph == PH_INIT || ph == PH_NEEDJ)
              : stage == ST_PROBE ? (ph == PH_SUB && st->L > 1e-4)
                                  : ph == PH_SUB);
    if (active) {
      const apx_batch_galaxy G = b.gal[g];
      const int bx = (G.pw + 1) / 2, by = (G.ph + 1) / 2;
      nch = ((G.nx + 2 * bx) * (G.ny + 2 * by) + kChunk - 1) / kChunk;
      ntl = ((G.nx + 63) / 64) * ((G.ny + kTR - 1) / kTR);
    }
  }
  if (part == 0) {
    const int slot = wave_reserve(active ? 1 : 0, &s.cnt[0], lane);
    const int cb = wave_reserve(nch, &s.cnt[1], lane);
    const int tb = wave_reserve(ntl, &s.cnt[2], lane);
    if (active) s.gal_list[slot] = g;
    for (uint64_t m = __ballot(active); m; m &= m - 1) {
      const int l = __ffsll((unsigned long long)m) - 1, fit = blockIdx.x * 64 + l;
      const int nc = __builtin_amdgcn_readlane(nch, l), c0 = __builtin_amdgcn_readlane(cb, l);
      const int nt = __builtin_amdgcn_readlane(ntl, l), t0 = __builtin_amdgcn_readlane(tb, l);
      for (int c = lane; c < nc; c += 64) s.chunk_list[c0 + c] = make_int2(fit, c);
      for (int t = lane; t < nt; t += 64) s.tile_list[t0 + t] = make_int2(fit, t);
    }
  }
  if (active) eval_fit(b, s, g, rep_override, stage, part);
}

// 1-D linear interpolation of the zero-padded factor f (n values, padded to
// n + 2) at r - s, with the clamped corners of bilinear(); d = d value / d s
__device__ __forceinline__ void lin1d(const float* f, int n, int r, double s, double& val, double& d) {
  const double x = (double)r - s;
  const int xf = (int)floor(x);
  const int x0 = min(max(xf, 0), n), x1 = min(max(xf + 1, 1), n + 1);
  const double f0 = (x0 >= 1 && x0 <= n) ? (double)f[x0 - 1] : 0.0;
  const double f1 = (x1 >= 1 && x1 <= n) ? (double)f[x1 - 1] : 0.0;
  val = f0 * ((double)x1 - x) + f1 * (x - (double)x0);
  d = -(f1 - f0);
}

// Separable kernels of a rank-one PSF P = u v^T.  bilinear() interpolates the
// padded PSF with corners clamped per axis, so the shifted PSF is U V^T with U
// (V) the 1-D interpolation of u (v) at the row (column) shift, and with
// K = U V^T / (sum U sum V) (_model_methods.py:187-207, 243):
//   K = uh vh^T,  dK/ds_x = uh vh'^T,  dK/ds_y = uh' vh^T,
//   uh = U / sum U,  uh' = dU / sum U - U sum dU / (sum U)^2  (likewise v).
// Axis w = 0 writes uh and uh', w = 1 vh and vh' (one wave), flipped for correlation, at
// taps + tap_off as [uh (kh4) | vh (kw4) | uh' (kh4) | vh' (kw4)], each padded
// with zeros from kh (kw) to kh4 (kw4), the length rounded up to 4.
__device__ void prepare_separable_axis(const apx_batch& b, const apx_batch_galaxy& G, int w, double sx, double sy,
                                       int lane) {
  const int H4 = sp_k4(G.ph + 2), W4 = sp_k4(G.pw + 2);
  const int n = w == 0 ? G.ph : G.pw, N2 = n + 2, N4 = sp_k4(N2);
  const float* f = b.psf_sep + G.sep_off + (w == 0 ? 0 : G.ph);
  const double sh = w == 0 ? sy : sx;
  double S = 0.0, Sd = 0.0;
  for (int r = lane; r < N2; r += 64) {
    double v, d;
    lin1d(f, n, r, sh, v, d);
    S += v;
    Sd += d;
  }
  S = wave_sum(S);
  Sd = wave_sum(Sd);
  const double iS = 1.0 / S;
  float* kt = b.taps + G.tap_off;
  float* o = kt + (w == 0 ? 0 : H4);
  float* od = kt + H4 + W4 + (w == 0 ? 0 : H4);
  for (int r = lane; r < N2; r += 64) {
    double v, d;
    lin1d(f, n, r, sh, v, d);
    o[N2 - 1 - r] = (float)(v * iS);
    od[N2 - 1 - r] = (float)(d * iS - v * Sd * iS * iS);
  }
  for (int r = N2 + lane; r < N4; r += 64) o[r] = od[r] = 0.0f;
}

// per fit (one wave each, rows then columns): the separable taps
__global__ __launch_bounds__(256) void prepare_sep_kernel(apx_batch b, Scratch s) {
  const int lane = threadIdx.x & 63;
  for (int k = blockIdx.x * 4 + (int)(threadIdx.x >> 6); k < s.cnt[0]; k += gridDim.x * 4) {
    const int g = s.gal_list[k];
    const apx_batch_galaxy G = b.gal[g];
    const double sx = s.ev[g].sx, sy = s.ev[g].sy;
    prepare_separable_axis(b, G, 0, sx, sy, lane);
    prepare_separable_axis(b, G, 1, sx, sy, lane);
  }
}

// Per fit (one workgroup each): shifted PSF taps in the conv layout, from the
// padded PSF in LDS.  Each tap is sampled once for the value kernel and its two
// centre derivatives (125 scene sources, 67 x 67: 53 -> 21 us).
__global__ __launch_bounds__(256) void prepare_kernel(apx_batch b, Scratch s, int stage) {
  extern __shared__ float padded[];
  __shared__ double red[4][3];
  const int nk = (stage == ST_JAC || stage == ST_ALL_JAC) ? 3 : 1;
  const double det = b.P[0] * b.P[3] - b.P[1] * b.P[2];
  const double Pi[4] = {b.P[3] / det, -b.P[1] / det, -b.P[2] / det, b.P[0] / det};
  for (int k = blockIdx.x; k < s.cnt[0]; k += gridDim.x) {
    const int g = s.gal_list[k];
    const apx_batch_galaxy G = b.gal[g];
    const double sx = s.ev[g].sx, sy = s.ev[g].sy;
    // shifted, normalised PSF (and its centre derivatives), flipped, in the
    // KT[k][b][u] = Kf[u - 7][b] layout of conv_common.h
    const int H2 = G.ph + 2, W2 = G.pw + 2, n = H2 * W2, kts = fast_kts(H2);
    float* kt = b.taps + G.tap_off;
    pad_psf(b.psf + G.psf_off, G.ph, G.pw, padded);
    __syncthreads();
    double sum[3] = {0.0, 0.0, 0.0};
    for (int e = threadIdx.x; e < n; e += 256) {
      double val, ddx, ddy;
      bilinear_lds(padded, G.ph, G.pw, e / W2, e % W2, sx, sy, val, ddx, ddy);
      sum[0] += val;
      sum[1] += ddx;
      sum[2] += ddy;
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      sum[q] = wave_sum(sum[q]);
      if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][q] = sum[q];
    }
    __syncthreads();
    const double S = red[0][0] + red[1][0] + red[2][0] + red[3][0];
    const double Sx = red[0][1] + red[1][1] + red[2][1] + red[3][1];
    const double Sy = red[0][2] + red[1][2] + red[2][2] + red[3][2];
    const double iS = 1.0 / S;
    const int plane = W2 * kts;
    for (int e = threadIdx.x; e < plane; e += 256) {
      const int u = e % kts, col = e / kts;
      const int a = u - (kRYF - 1);  // flipped-kernel row
      float out[3] = {0.0f, 0.0f, 0.0f};
      if (a >= 0 && a < H2) {
        const int r = H2 - 1 - a, c = W2 - 1 - col;  // unflipped sample
        double val, ddx, ddy;
        bilinear_lds(padded, G.ph, G.pw, r, c, sx, sy, val, ddx, ddy);
        out[0] = (float)(val * iS);
        if (nk > 1) {
          const double Kx = ddx * iS - val * Sx * iS * iS, Ky = ddy * iS - val * Sy * iS * iS;
          out[1] = (float)(Kx * Pi[0] + Ky * Pi[2]);
          out[2] = (float)(Kx * Pi[1] + Ky * Pi[3]);
        }
      }
      for (int q = 0; q < nk; ++q) kt[q * plane + e] = out[q];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// render stages
//
// Pixel selection and adaptive quadrature (utils/operations.py:150-247, driven
// by models/_model_methods.py:82-184).  Samples are evaluated in float32 and
// summed in float64; every threshold decision whose float32 value lies within
// kBandRel of the threshold is taken again from float64 samples, so the set of
// refined pixels and sub-pixels is the one float64 arithmetic gives.
constexpr double kBandRel = 1e-4;

// Gauss-Legendre table of order n and the sub-gridding g
// Every galaxy of a batch is a Sersic profile (sersic_model.py:41-91,
// parametric_profiles.py:7-24).  Its float32 samples use the raw v_log_f32 /
// v_exp_f32 / v_rsq_f32 units in base 2, and the value needs no square root:
//   log2(R/Re) = log2(R^2)/2 + log2(1/Re),   (R/Re)^(1/n) = 2^(log2(R/Re)/n),
//   I = scale amp 2^(-b log2(e) ((R/Re)^(1/n) - 1)),
// with R^2 = X'^2 + Y'^2 + softening^2 after the rotation and the 1/q stretch
// (the same quantities as eval_profile, which the float64 decisions keep).
template <bool GRAD>
__device__ __forceinline__ float sersic_f(const Prof<float>& p, float X, float Y, float scale, float* g) {
  const float Xr = p.c * X - p.s * Y;
  const float Yr = (p.s * X + p.c * Y) * p.invq;
  const float R2 = Xr * Xr + Yr * Yr + p.soft2;
  const float l2 = 0.5f * __builtin_amdgcn_logf(R2) + p.l2s;
  const float pw = __builtin_amdgcn_exp2f(l2 * p.inva);
  const float I = p.amp * scale * __builtin_amdgcn_exp2f(p.nbl2e * (pw - 1.0f));
  if (GRAD) {
    const float invR = __builtin_amdgcn_rsqf(R2);
    const float lx = l2 * 0.693147180559945309f;  // ln(R/Re)
    const float t = I * p.b * pw * p.inva;
    const float dIdR = -t * invR;
    const float dRdX = (p.c * Xr + p.s * Yr * p.invq) * invR;
    const float dRdY = (-p.s * Xr + p.c * Yr * p.invq) * invR;
    g[APX_P_CX] = -dIdR * dRdX;  // X = coordinate - centre
    g[APX_P_CY] = -dIdR * dRdY;
    g[APX_P_Q] = -dIdR * Yr * Yr * p.invq * invR;
    g[APX_P_PA] = dIdR * Xr * Yr * p.qm * invR;
    g[APX_P_A] = I * (-p.db * (pw - 1.0f) + p.b * pw * lx * p.inva * p.inva);
    g[APX_P_B] = t * p.inv_s;
    g[APX_P_C] = I * (float)kLn10;
  }
  return I;
}

// sersic_f's value with every multiply-add written out.  Which of two products
// the compiler folds into an addition depends on the code around it, and with it
// the sample's last bit; the level-3 pass keeps this one whatever its shape.
__device__ __forceinline__ float sersic_value_f(const Prof<float>& p, float X, float Y, float scale) {
  const float Xr = fmaf(p.c, X, -(p.s * Y));
  const float Yr = fmaf(p.s, X, p.c * Y) * p.invq;
  const float R2 = fmaf(Xr, Xr, Yr * Yr) + p.soft2;
  const float l2 = fmaf(0.5f, __builtin_amdgcn_logf(R2), p.l2s);
  const float pw = __builtin_amdgcn_exp2f(l2 * p.inva);
  return p.amp * scale * __builtin_amdgcn_exp2f(p.nbl2e * (pw - 1.0f));
}

struct QuadTab {
  int n, nn, g, gg, max_depth;
  float node[APX_MAX_QUAD_LEVEL];
  float w2[APX_MAX_QUAD_LEVEL * APX_MAX_QUAD_LEVEL];  // w_a w_b / 4, node k = (k % n, k / n)
  float lw[9];     // n = 3: log2 w2[k]
  float inv_w4;    // n = 3: 1 / w2[4] (the centre node)
  double noded[APX_MAX_QUAD_LEVEL];
  double w2d[APX_MAX_QUAD_LEVEL * APX_MAX_QUAD_LEVEL];
};

// n x n Gauss-Legendre sample of the square of half-width h (in pixel-matrix
// units) centred on (X, Y) (operations.py:123-147); `centre` is the middle node
// QN: the quadrature level when known at compile time (0: t.n)
template <bool GRAD, int QN = 0>
__device__ __forceinline__ float quad_f(const Prof<float>& p, const QuadTab& t, float X, float Y,
                                        float h, float scale, float* g, float& centre) {
  float res = 0.0f, gl[APX_NSLOT];
  if (GRAD) {
#pragma unroll
    for (int q = 0; q < APX_NSLOT; ++q) g[q] = 0.0f;
  }
  const float h00 = h * p.P00, h01 = h * p.P01, h10 = h * p.P10, h11 = h * p.P11;
  const int n = QN ? QN : t.n, nn = n * n;
#pragma unroll
  for (int k = 0; k < nn; ++k) {
    const float u = t.node[k % n], v = t.node[k / n], w = t.w2[k];
    const float val = sersic_f<GRAD>(p, X + h00 * u + h01 * v, Y + h10 * u + h11 * v, scale, gl);
    res = fmaf(w, val, res);
    if (k == nn / 2) centre = val;
    if (GRAD) {
#pragma unroll
      for (int q = 0; q < APX_NSLOT; ++q) g[q] = fmaf(w, gl[q], g[q]);
    }
  }
  return res;
}

__device__ __forceinline__ double quad_d(const Prof<double>& p, const QuadTab& t, double X,
                                         double Y, double h, double scale, double& centre) {
  double res = 0.0;
  const double h00 = h * p.P00, h01 = h * p.P01, h10 = h * p.P10, h11 = h * p.P11;
  for (int k = 0; k < t.nn; ++k) {
    const double u = t.noded[k % t.n], v = t.noded[k / t.n];
    const double val = eval_profile<double, false>(p, X + h00 * u + h01 * v,
                                                   Y + h10 * u + h11 * v, scale, nullptr);
    res += t.w2d[k] * val;
    if (k == t.nn / 2) centre = val;
  }
  return res;
}

// rotation by theta = -(PA - pi/2) and the 1/q stretch of sersic_f
__device__ __forceinline__ void rot(const Prof<float>& p, float x, float y, float& xr, float& yr) {
  xr = fmaf(p.c, x, -p.s * y);
  yr = fmaf(p.s, x, p.c * y) * p.invq;
}

// Value-only 3 x 3 Gauss-Legendre sample of a Sersic in the rotated,
// stretched frame: (xr, yr) is the rotated sample centre, (ax, ay) and
// (bx, by) the rotated node steps along the two pixel axes; each node's weight
// and the sampling scale sit in its exponent offset (Kc corner, Ke edge, K0
// centre: log2(amp scale w) - nbl2e), so w I = exp2(nbl2e pw + K).  Returns
// the weighted sum (quad_f's value) and sets cen to the centre node's w I.
__device__ __forceinline__ float gl3_rot(const Prof<float>& pf, float xr, float yr, float ax, float ay, float bx,
                                         float by, float Kc, float Ke, float K0, float& cen) {
  const float k1 = 0.5f * pf.inva, k0 = pf.l2s * pf.inva;
  float acc = 0.0f;
#pragma unroll
  for (int vv = -1; vv <= 1; ++vv) {
    const float rx = xr + (float)vv * bx, ry = yr + (float)vv * by;
#pragma unroll
    for (int uu = -1; uu <= 1; ++uu) {
      const float X = rx + (float)uu * ax, Y = ry + (float)uu * ay;
      const float R2 = fmaf(X, X, fmaf(Y, Y, pf.soft2));
      const float pw = __builtin_amdgcn_exp2f(fmaf(__builtin_amdgcn_logf(R2), k1, k0));
      const float K = (uu == 0 && vv == 0) ? K0 : ((uu == 0 || vv == 0) ? Ke : Kc);
      const float I = __builtin_amdgcn_exp2f(fmaf(pf.nbl2e, pw, K));
      acc += I;
      if (uu == 0 && vv == 0) cen = I;
    }
  }
  return acc;
}

// Value and parameter partials (slots APX_P_*, as quad_f<true, 3>) of the 3 x 3
// Gauss-Legendre sample in the rotated, stretched frame of gl3_rot.  With
// w I = exp2(nbl2e pw + K) at a node (pw = (R / Re)^(1/n), K = log2(amp scale
// w) - nbl2e) sersic_f's partials are, per node,
//   cx, cy: (b/n) (w I pw / R^2) (c X + s Y / q, -s X + c Y / q)
//   q: (b/n) (w I pw / R^2) Y^2 / q      PA: -(b/n) (q - 1/q) (w I pw / R^2) X Y
//   n: -db (w I pw - w I) + (b / n^2) ln2 w I pw log2(R / Re)
//   Re: (b/n) w I pw / Re                Ie: ln10 w I
// (X, Y rotated and stretched), so only seven node sums are kept and the
// constants are applied once.  `centre` is the middle node's I, as quad_f's.
__device__ __forceinline__ float quad3_grad(const Prof<float>& pf, const QuadTab& t, float X, float Y, float h,
                                            float l2scale, float* g, float& centre) {
  float xr, yr, ax, ay, bx, by;
  rot(pf, X, Y, xr, yr);
  const float hn = h * t.node[2];
  rot(pf, hn * pf.P00, hn * pf.P10, ax, ay);
  rot(pf, hn * pf.P01, hn * pf.P11, bx, by);
  const float base = pf.l2amp - pf.nbl2e + l2scale;
  const float Kc = base + t.lw[0], Ke = base + t.lw[1], K0 = base + t.lw[4];
  float sI = 0.0f, sIp = 0.0f, sA = 0.0f, sB = 0.0f, sAY = 0.0f, sBY = 0.0f, sL = 0.0f, cen = 0.0f;
#pragma unroll
  for (int vv = -1; vv <= 1; ++vv) {
    const float rx = xr + (float)vv * bx, ry = yr + (float)vv * by;
#pragma unroll
    for (int uu = -1; uu <= 1; ++uu) {
      const float Xn = rx + (float)uu * ax, Yn = ry + (float)uu * ay;
      const float R2 = fmaf(Xn, Xn, fmaf(Yn, Yn, pf.soft2));
      const float l2 = fmaf(__builtin_amdgcn_logf(R2), 0.5f, pf.l2s);  // log2(R / Re)
      const float pw = __builtin_amdgcn_exp2f(l2 * pf.inva);
      const float K = (uu == 0 && vv == 0) ? K0 : ((uu == 0 || vv == 0) ? Ke : Kc);
      const float I = __builtin_amdgcn_exp2f(fmaf(pf.nbl2e, pw, K));
      const float Ip = I * pw;
      const float r = Ip * __builtin_amdgcn_rcpf(R2);
      const float A = r * Xn, B = r * Yn;
      sI += I;
      sIp += Ip;
      sA += A;
      sB += B;
      sAY = fmaf(A, Yn, sAY);
      sBY = fmaf(B, Yn, sBY);
      sL = fmaf(Ip, l2, sL);
      if (uu == 0 && vv == 0) cen = I;
    }
  }
  const float bn = pf.b * pf.inva, bq = bn * pf.invq;
  g[APX_P_CX] = bn * pf.c * sA + bq * pf.s * sB;
  g[APX_P_CY] = bq * pf.c * sB - bn * pf.s * sA;
  g[APX_P_Q] = bq * sBY;
  g[APX_P_PA] = -bn * pf.qm * sAY;
  g[APX_P_A] = pf.db * (sI - sIp) + bn * pf.inva * 0.693147180559945309f * sL;
  g[APX_P_B] = bn * pf.inv_s * sIp;
  g[APX_P_C] = (float)kLn10 * sI;
  centre = cen * t.inv_w4;
  return sI;
}

// quad_f<false, 3> (value only, quad_level 3) through gl3_rot: the 3 x 3
// sample of half-width h and area scale 2^l2scale centred on plane offset (X, Y)
__device__ __forceinline__ float quad3_value(const Prof<float>& pf, const QuadTab& t, float X, float Y, float h,
                                             float l2scale, float& centre) {
  float xr, yr, ax, ay, bx, by;
  rot(pf, X, Y, xr, yr);
  const float hn = h * t.node[2];
  rot(pf, hn * pf.P00, hn * pf.P10, ax, ay);
  rot(pf, hn * pf.P01, hn * pf.P11, bx, by);
  const float base = pf.l2amp - pf.nbl2e + l2scale;
  float cen = 0.0f;
  const float r = gl3_rot(pf, xr, yr, ax, ay, bx, by, base + t.lw[0], base + t.lw[1], base + t.lw[4], cen);
  centre = cen * t.inv_w4;
  return r;
}

// |res - centre| > thr, decided in float64 when float32 is too close to call
__device__ __forceinline__ int band_test(float res, float centre, double thr) {
  const double D = fabs((double)res - (double)centre);
  const double band = kBandRel * (fabs((double)res) + fabs((double)centre)) + 1e-7 * thr;
  if (D > thr + band) return 1;
  if (D < thr - band) return 0;
  return -1;
}

// The chunk list and the per-fit records arrive again as read-only,
// non-aliasing arguments: the compiler then reads them with scalar loads, whose
// wait counter is separate from the vector memory counter.  Read through the
// structs' pointers they are vector loads, and the wait for them at the top of
// each chunk also waits for the previous chunk's plane stores to complete.

// midpoint samples of every working pixel (and their parameter partials)
template <bool GRAD>
__global__ __launch_bounds__(kChunk) void init_kernel(apx_batch b, Scratch s,
                                                      const int2* __restrict__ chunks,
                                                      const apx_batch_galaxy* __restrict__ gal,
                                                      const GalEval* __restrict__ ev) {
  // a contiguous run of chunks per workgroup: a fit's chunks are listed
  // together, so its record is read again only when the fit changes
  // (fit g, chunk c) entries list a fit's chunks c = 0 .. nch - 1 in order, so
  // the next entry is (g, c + 1) until the fit's last chunk: the list is read
  // only where a fit begins
  const int n = s.cnt[1], per = (n + (int)gridDim.x - 1) / (int)gridDim.x;
  const int k0 = blockIdx.x * per, k1 = min(n, k0 + per);
  int64_t work_off = 0;
  GalEval E;
  int2 e = make_int2(-1, 0);
  int nch = 0;
  for (int k = k0; k < k1; ++k) {
    if (e.x >= 0 && e.y + 1 < nch) {
      ++e.y;
    } else {
      e = chunks[k];
      work_off = gal[e.x].work_off;
      E = ev[e.x];
      nch = (E.nxw * E.nyw + kChunk - 1) / kChunk;
    }
    const int pix = e.y * kChunk + threadIdx.x;
    if (pix >= E.nxw * E.nyw) continue;
    float X, Y, gr[APX_NSLOT];
    pixel_xy(E.pf, E.ci, E.cj, pix % E.nxw, pix / E.nxw, X, Y);
    const float val = sersic_f<GRAD>(E.pf, X, Y, 1.0f, gr);
    s.mid[work_off + pix] = val;
    if (GRAD) {
      // planes 1..5: q, PA, n, Re, Ie in representation units
      float* pl = b.planes + work_off + pix;
#pragma unroll
      for (int c = 1; c < kNChan; ++c) pl[c * b.nwork] = gr[c + 1] * (float)E.dvdr[c + 1];
    }
  }
}

// Outcome of one pixel's selection and level-1 test.  Instantiated with F64
// false a test too close to call in float32 gives PX_UNDECIDED and writes
// nothing; the pixel then goes to its fit's redo list and is taken again by
// the F64 instantiation, whose float64 path keeps the register use of the
// common float32 kernels low.
enum : int { PX_DONE = 0, PX_DEEPER = 1, PX_UNDECIDED = 2 };

// curvature selection (_model_methods.py:87-97, 155-166) of working pixel
// `pix` and, if selected, its level-1 quadrature (operations.py:210-228)
template <bool GRAD, bool F64, int QN>
__device__ __forceinline__ int select_pixel(const apx_batch& b, const Scratch& s,
                                            const apx_batch_galaxy& G, const GalEval& E,
                                            const QuadTab& t, int pix) {
  const int i = pix % E.nxw, j = pix / E.nxw;
  const int ii = min(max(i, 1), E.nxw - 2), jj = min(max(j, 1), E.nyw - 2);
  const float* v = s.mid + G.work_off + (int64_t)jj * E.nxw + ii;
  const float l = v[-1], r = v[1], u = v[-E.nxw], d = v[E.nxw], m = v[0];
  const float metric = fabsf(l + r + u + d - 4.0f * m);
  const float scale = fabsf(l) + fabsf(r) + fabsf(u) + fabsf(d) + 4.0f * fabsf(m);
  const double band = 1.6e-5 * (double)scale + 2.0e-7 * E.thr;
  bool sel = false;
  if ((double)metric > E.thr + band) {
    sel = true;
  } else if ((double)metric >= E.thr - band) {  // float64 decision
    if (!F64) return PX_UNDECIDED;
    double X, Y;
    auto at = [&](int a, int c) {
      pixel_xy(E.pd, E.ci, E.cj, a, c, X, Y);
      return eval_profile<double, false>(E.pd, X, Y, 1.0, nullptr);
    };
    const double mc = at(ii, jj);
    const double curv = at(ii - 1, jj) + at(ii + 1, jj) + at(ii, jj - 1) + at(ii, jj + 1) - 4.0 * mc;
    const double mid = (i == ii && j == jj) ? mc : at(i, j);
    sel = fabs(mid - (mid + curv)) > E.thr;
  }
  float* pl = b.planes + G.work_off + pix;
  if (!sel) {
    pl[0] = s.mid[G.work_off + pix];
    return PX_DONE;
  }
  float X0, Y0, gs[APX_NSLOT], centre = 0.0f;
  pixel_xy(E.pf, E.ci, E.cj, i, j, X0, Y0);
  const float r1 = QN == 3 ? (GRAD ? quad3_grad(E.pf, t, X0, Y0, 0.5f, 0.0f, gs, centre)
                                  : quad3_value(E.pf, t, X0, Y0, 0.5f, 0.0f, centre))
                           : quad_f<GRAD, QN>(E.pf, t, X0, Y0, 0.5f, 1.0f, gs, centre);
  if (t.max_depth > 1) {
    const int dec = band_test(r1, centre, E.thr);
    bool deeper = dec == 1;
    if (dec < 0) {
      if (!F64) return PX_UNDECIDED;
      double X, Y, cd = 0.0;
      pixel_xy(E.pd, E.ci, E.cj, i, j, X, Y);
      const double rd = quad_d(E.pd, t, X, Y, 0.5, 1.0, cd);
      deeper = fabs(rd - cd) > E.thr;
    }
    if (deeper) return PX_DEEPER;
  }
  pl[0] = r1;
  if (GRAD) {
#pragma unroll
    for (int c = 1; c < kNChan; ++c) pl[c * b.nwork] = gs[c + 1] * (float)E.dvdr[c + 1];
  }
  return PX_DONE;
}

// appends `value` for every lane with `flag` to a segment whose length is
// `*counter`: one atomic per wave (all lanes share the counter)
__device__ __forceinline__ void wave_append(bool flag, int32_t* counter, int32_t* seg, int value,
                                            int lane) {
  const uint64_t ballot = __ballot(flag);
  if (!ballot) return;
  int base = 0;
  if (lane == 0) base = atomicAdd(counter, (int)__popcll(ballot));
  base = __shfl(base, 0, 64);
  if (flag) {
    const uint64_t below = ballot & ((lane == 0) ? 0ull : (~0ull >> (64 - lane)));
    seg[base + (int)__popcll(below)] = value;
  }
}

// float32 selection of every listed chunk, one lane per pixel
template <bool GRAD, int QN>
__global__ __launch_bounds__(256) void select_kernel(apx_batch b, Scratch s, QuadTab t,
                                                    const int2* __restrict__ chunks,
                                                    const apx_batch_galaxy* __restrict__ gal,
                                                    const GalEval* __restrict__ ev) {
  const int lane = threadIdx.x & 63;
  // contiguous chunk runs, as in init_kernel
  const int n = s.cnt[1], per = (n + (int)gridDim.x - 1) / (int)gridDim.x;
  const int k0 = blockIdx.x * per, k1 = min(n, k0 + per);
  apx_batch_galaxy G;
  GalEval E;
  int2 e = make_int2(-1, 0);
  int nch = 0;
  for (int k = k0; k < k1; ++k) {
    if (e.x >= 0 && e.y + 1 < nch) {  // the fit's next chunk (see init_kernel)
      ++e.y;
    } else {
      e = chunks[k];
      G = gal[e.x];
      E = ev[e.x];
      nch = (E.nxw * E.nyw + kChunk - 1) / kChunk;
    }
    const int pix = e.y * kChunk + threadIdx.x;
    const int res = pix < E.nxw * E.nyw ? select_pixel<GRAD, false, QN>(b, s, G, E, t, pix) : PX_DONE;
    wave_append(res == PX_DEEPER, &s.gal_cnt[e.x], s.deep + G.work_off, pix, lane);
    wave_append(res == PX_UNDECIDED, &s.gal_rcnt[e.x], s.redo + G.work_off, pix, lane);
  }
}

// The per-fit segments of pixels (a count and a run at work_off each) as one list
// of (fit, pixel), so that the passes over it take any fit's pixels evenly: a
// workgroup takes `fits` of the listed fits (at most kPackFits) and one place in
// the list (one atomic on its length).  The order of the workgroups' runs in the
// list does not matter: every pixel is taken by itself.  One launch a list in
// place of two for a scan and a compaction, with three lists a stage:
// 56 -> 38 launches a tick (4,096 fits to convergence, with the level-3 pass by
// waves below: 117.5 -> 102.4 ms).
// `clear`: the counts start from zero again.
constexpr int kPackFits = 8;

__global__ __launch_bounds__(256) void pack_kernel(apx_batch b, Scratch s, int fits, int32_t* __restrict__ cnt,
                                                   const int32_t* __restrict__ seg, int2* __restrict__ out,
                                                   int32_t* len, int clear) {
  __shared__ int pre[kPackFits + 1], fit[kPackFits], base;
  __shared__ int64_t off[kPackFits];
  for (int first = blockIdx.x * fits; first < s.cnt[0]; first += gridDim.x * fits) {
    __syncthreads();  // the previous run is read
    if (threadIdx.x < kPackFits) {
      const int i = first + (int)threadIdx.x;
      int n = 0, g = 0;
      if ((int)threadIdx.x < fits && i < s.cnt[0]) {
        g = s.gal_list[i];
        n = cnt[g];
        if (clear) cnt[g] = 0;
      }
      fit[threadIdx.x] = g;
      off[threadIdx.x] = b.gal[g].work_off;
      int x = n;
#pragma unroll
      for (int o = 1; o < kPackFits; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if ((int)threadIdx.x >= o) x += y;
      }
      pre[threadIdx.x + 1] = x;
      if (threadIdx.x == 0) pre[0] = 0;
      if (threadIdx.x == kPackFits - 1 && x > 0) base = atomicAdd(len, x);
    }
    __syncthreads();
    const int total = pre[kPackFits];
    for (int e = threadIdx.x; e < total; e += 256) {
      int f = 0;
#pragma unroll
      for (int o = kPackFits / 2; o > 0; o >>= 1)
        if (e >= pre[f + o]) f += o;
      out[base + e] = make_int2(fit[f], seg[off[f] + (e - pre[f])]);
    }
  }
}

// select_pixel<GRAD, true, 3> by a team of 16 lanes (every lane of the wave calls
// it; `active` is the same in a team's lanes): the float64 samples of a decision
// go to a lane each, 5 or 6 for the curvature and 9 for the level-1 test
template <bool GRAD>
__device__ __forceinline__ void select_team(const apx_batch& b, const Scratch& s, const QuadTab& t, bool active, int g,
                                            int pix) {
  const int tl = threadIdx.x & 15;
  const apx_batch_galaxy G = b.gal[g];
  const GalEval& E = s.ev[g];
  const int nxw = E.nxw, i = pix % nxw, j = pix / nxw;
  const int ii = min(max(i, 1), nxw - 2), jj = min(max(j, 1), E.nyw - 2);
  const float* v = s.mid + G.work_off + (int64_t)jj * nxw + ii;
  const float l = v[-1], r = v[1], u = v[-nxw], d = v[nxw], m = v[0];
  const float metric = fabsf(l + r + u + d - 4.0f * m);
  const float scale = fabsf(l) + fabsf(r) + fabsf(u) + fabsf(d) + 4.0f * fabsf(m);
  const double band = 1.6e-5 * (double)scale + 2.0e-7 * E.thr;
  bool sel = (double)metric > E.thr + band;
  const bool close = active && !sel && (double)metric >= E.thr - band;
  double X, Y, val = 0.0;
  if (close && tl < 6) {  // the centre, its left, right, upper and lower neighbours, the pixel
    const int a = tl == 1 ? ii - 1 : tl == 2 ? ii + 1 : tl == 5 ? i : ii;
    const int c = tl == 3 ? jj - 1 : tl == 4 ? jj + 1 : tl == 5 ? j : jj;
    pixel_xy(E.pd, E.ci, E.cj, a, c, X, Y);
    val = eval_profile<double, false>(E.pd, X, Y, 1.0, nullptr);
  }
  double at[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) at[q] = __shfl(val, q, 16);
  if (close) {
    const double curv = at[1] + at[2] + at[3] + at[4] - 4.0 * at[0];
    const double mid = at[5];
    sel = fabs(mid - (mid + curv)) > E.thr;
  }
  float* pl = b.planes + G.work_off + pix;
  float X0, Y0, gs[APX_NSLOT], centre = 0.0f;
  pixel_xy(E.pf, E.ci, E.cj, i, j, X0, Y0);
  const float r1 = GRAD ? quad3_grad(E.pf, t, X0, Y0, 0.5f, 0.0f, gs, centre)
                        : quad3_value(E.pf, t, X0, Y0, 0.5f, 0.0f, centre);
  const int dec = t.max_depth > 1 ? band_test(r1, centre, E.thr) : 0;
  const bool test = active && sel && dec < 0;
  val = 0.0;
  if (test && tl < 9) {
    pixel_xy(E.pd, E.ci, E.cj, i, j, X, Y);
    const double un = t.noded[tl % 3], vn = t.noded[tl / 3];
    const double h00 = 0.5 * E.pd.P00, h01 = 0.5 * E.pd.P01, h10 = 0.5 * E.pd.P10, h11 = 0.5 * E.pd.P11;
    val = eval_profile<double, false>(E.pd, X + h00 * un + h01 * vn, Y + h10 * un + h11 * vn, 1.0, nullptr);
  }
  double rd = 0.0, cd = 0.0;
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const double x = __shfl(val, q, 16);
    rd += t.w2d[q] * x;
    if (q == 4) cd = x;
  }
  const bool deeper = test ? fabs(rd - cd) > E.thr : dec == 1;
  if (!active || tl != 0) return;
  if (!sel) {
    pl[0] = s.mid[G.work_off + pix];
  } else if (deeper) {
    s.deep[G.work_off + atomicAdd(&s.gal_cnt[g], 1)] = pix;
  } else {
    pl[0] = r1;
    if (GRAD) {
#pragma unroll
      for (int c = 1; c < kNChan; ++c) pl[c * b.nwork] = gs[c + 1] * (float)E.dvdr[c + 1];
    }
  }
}

// The pixels select_kernel left undecided, with float64 decisions: a lane each,
// or 16 lanes each where the list is short enough that every team of the launch
// has one at most.  One lane takes up to 15 float64 samples one after another
// (11 -> 6 us with about 100 fits left); on a long list (125 scene sources, 0.3 ms)
// the lanes are all busy.
template <bool GRAD, int QN>
__global__ __launch_bounds__(256) void select_redo_kernel(apx_batch b, Scratch s, QuadTab t) {
  const int total = s.cnt[4];
  if (QN == 3 && total <= (int)gridDim.x * 16) {
    const int k = blockIdx.x * 16 + (int)(threadIdx.x >> 4);
    if ((k & ~3) >= total) return;  // none of the wave's four teams has a pixel
    const int2 q = s.rq[min(k, total - 1)];
    select_team<GRAD>(b, s, t, k < total, q.x, q.y);
    return;
  }
  for (int k = blockIdx.x * 256 + threadIdx.x; k < total; k += gridDim.x * 256) {
    const int2 q = s.rq[k];
    const int g = q.x, pix = q.y;
    const apx_batch_galaxy G = b.gal[g];
    if (select_pixel<GRAD, true, QN>(b, s, G, s.ev[g], t, pix) == PX_DEEPER)
      s.deep[G.work_off + atomicAdd(&s.gal_cnt[g], 1)] = pix;
  }
}

// A lane's level-3 samples of one flagged sub-pixel at (xs, ys), summed in float32
template <bool GRAD, int GS, int ITS>
__device__ __forceinline__ void level3_lane(const Prof<float>& pf, float xs, float ys, const float (&l3x)[ITS],
                                            const float (&l3y)[ITS], const float (&l3w)[ITS], int gl, int nq, float sc3,
                                            float (&fs)[1 + APX_NSLOT]) {
#pragma unroll
  for (int q = 0; q <= APX_NSLOT; ++q) fs[q] = 0.0f;
#pragma unroll
  for (int it = 0; it < ITS; ++it) {
    if (gl + GS * it < nq) {
      float gv[APX_NSLOT];
      const float val = sersic_f<GRAD>(pf, xs + l3x[it], ys + l3y[it], sc3, gv);
      fs[0] = fmaf(l3w[it], val, fs[0]);
      if (GRAD) {
#pragma unroll
        for (int q = 0; q < APX_NSLOT; ++q) fs[1 + q] = fmaf(l3w[it], gv[q], fs[1 + q]);
      }
    }
  }
}

// levels 2 and 3 of the quadrature (operations.py:229-247): a group of GS
// lanes per listed pixel, one lane per level-2 sub-pixel; each sub-pixel the
// level-2 test flags is then integrated by the whole group.  F64 false: the
// deep list, and a pixel with an undecided sub-pixel test goes to the redo
// list unwritten; F64 true: the redo list, float64 decisions.
// QN, QG: quadrature level and gridding when known at compile time (0: from
// t).  With both known, each lane's level-3 sample offsets (plane units) and
// weights are computed once per launch.
//
// A short list (at most two pixels a resident workgroup, kWideMax) is taken a
// workgroup a pixel: its 8 groups of 32 lanes evaluate level 2 alike and take the
// flagged sub-pixels in turn, and thread (channel, lane) adds that lane's level-2
// value and sub-pixel sums in the order the one group adds them, so the bits do
// not change.  One group walks up to 25 sub-pixels of 8 samples a lane one after
// another, and a lane up to 9 float64 samples of an undecided one, which sets the
// time of a launch with few fits left (about 100 of 4,096: Jacobian pass 30 -> 21
// us, its float64 pass 28 -> 12, the value pass's 19 -> 10).
// A long list keeps a group a pixel, which evaluates level 2 once.  The two cross
// between 2,000 and 10,000 pixels, by how many sub-pixels are flagged: renders of
// 3,100 refined pixels of small cutouts 57 us so and 61 wide, of 3,000 of larger
// windows 77 and 76 (Jacobians 61 and 65, 98 and 84), of 12,000 75 and 91.
constexpr int kWideMax = 2048;
template <bool GRAD, int GS, bool F64, int QN, int QG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void integrate_kernel(apx_batch b, Scratch s,
                                                                                                QuadTab t) {
  constexpr int NG = 64 / GS;
  constexpr bool FIXED = QN > 0 && QG > 0;
  constexpr int ITS = FIXED ? (QN * QN * QG * QG + GS - 1) / GS : 1;
  const int lane = threadIdx.x & 63, gl = lane % GS, grp = lane / GS;
  const int wave = blockIdx.x * 4 + (threadIdx.x >> 6), nwaves = gridDim.x * 4;
  const int total = F64 ? s.cnt[5] : s.cnt[3];
  const int qn = QN ? QN : t.n, qnn = qn * qn;
  const int g_ = QG ? QG : t.g, gg = g_ * g_, nq = gg * qnn;
  const float ig = 1.0f / (float)g_;
  const float l2ig2 = 2.0f * __builtin_amdgcn_logf(ig);  // log2 of the level-2 scale ig^2
  const float sub0 = -(float)(g_ - 1) / (2.0f * (float)g_), subd = ig;
  const float h3 = 0.5f * ig * ig;
  float l3x[ITS], l3y[ITS], l3w[ITS];
  if (FIXED) {
    const float P00 = (float)b.P[0], P01 = (float)b.P[1], P10 = (float)b.P[2], P11 = (float)b.P[3];
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
      const int e = gl + GS * it;
      l3x[it] = l3y[it] = l3w[it] = 0.0f;
      if (e < nq) {
        const int tt = e / qnn, kk = e % qnn;
        const float a = (sub0 + subd * (float)(tt % g_)) * ig, c = (sub0 + subd * (float)(tt / g_)) * ig;
        const float u = a + h3 * t.node[kk % qn], v = c + h3 * t.node[kk / qn];
        l3x[it] = P00 * u + P01 * v;
        l3y[it] = P10 * u + P11 * v;
        l3w[it] = t.w2[kk];
      }
    }
  }
  const uint64_t gmask = GS == 64 ? ~0ull : (((1ull << GS) - 1ull) << (grp * GS));
  int nsub3 = 0;  // level-3 sub-pixels this wave integrates (work counter, wave-uniform)
  constexpr bool CAN_WIDE = FIXED && GS == 32;
  constexpr int NV = GRAD ? 1 + APX_NSLOT : 1;
  __shared__ double sample[CAN_WIDE && F64 ? QG * QG : 1][9];  // wide: an undecided sub-pixel's float64 samples
  __shared__ float subsum[CAN_WIDE ? QG * QG : 1][NV][32];  // wide: a lane's sum of a flagged sub-pixel
  const bool wide = CAN_WIDE && total <= min(kWideMax, 2 * (int)gridDim.x);
  const int team = threadIdx.x / GS;  // wide: group of the workgroup, and channel it adds up
  for (int k0 = wide ? (int)blockIdx.x : wave * NG; k0 < total; k0 += wide ? (int)gridDim.x : nwaves * NG) {
    const int k = wide ? k0 : k0 + grp;
    const bool active = k < total;
    int gal = 0, pix = 0;
    if (active) {
      const int2 q = F64 ? s.rq[k] : s.dq[k];
      gal = q.x;
      pix = q.y;
    }
    const GalEval* E = s.ev + gal;  // fit 0's constants for an idle group: read, never used
    const Prof<float> pf = E->pf;
    const int nxw = active ? E->nxw : 1, ci = E->ci, cj = E->cj;
    const int pi = pix % nxw, pj = pix / nxw;
    float X0, Y0;
    pixel_xy(pf, ci, cj, pi, pj, X0, Y0);
    double acc[1 + APX_NSLOT];
#pragma unroll
    for (int q = 0; q <= APX_NSLOT; ++q) acc[q] = 0.0;
    // level 2
    int dec = 0;
    float x2 = 0.0f, y2 = 0.0f, r2 = 0.0f, gs[APX_NSLOT];
    if (active && gl < gg) {
      const float a = sub0 + subd * (float)(gl % g_), c = sub0 + subd * (float)(gl / g_);
      x2 = X0 + pf.P00 * a + pf.P01 * c;
      y2 = Y0 + pf.P10 * a + pf.P11 * c;
      float c2 = 0.0f;
      r2 = (GRAD && QN == 3) ? quad3_grad(pf, t, x2, y2, 0.5f * ig, l2ig2, gs, c2)
                             : quad_f<GRAD, QN>(pf, t, x2, y2, 0.5f * ig, ig * ig, gs, c2);
      if (t.max_depth > 2) {
        const double thr2 = E->thr * (double)gg;
        dec = band_test(r2, c2, thr2);
        if (F64 && dec < 0 && !wide) {
          const double igd = 1.0 / (double)g_, sub0d = -(double)(g_ - 1) / (2.0 * g_);
          const double ad = sub0d + igd * (gl % g_), bd = sub0d + igd * (gl / g_);
          const Prof<double>& pd = E->pd;
          double X, Y, cd = 0.0;
          pixel_xy(pd, ci, cj, pi, pj, X, Y);
          const double rd = quad_d(pd, t, X + pd.P00 * ad + pd.P01 * bd, Y + pd.P10 * ad + pd.P11 * bd,
                                   0.5 * igd, igd * igd, cd);
          dec = fabs(rd - cd) > thr2 ? 1 : 0;
        }
      }
    }
    if (F64 && wide) {
      // the undecided sub-pixels' float64 samples, one a thread (25 x 9 at most),
      // then each sub-pixel's sum in quad_d's order
      const uint64_t und = (__ballot(dec < 0) & gmask) >> (grp * GS);
      const int nu = (int)__popcll(und);
      if (nu > 0) {
        const int f = (int)threadIdx.x / 9, kk = (int)threadIdx.x % 9;
        if (f < nu) {
          uint64_t m = und;
          for (int i = 0; i < f; ++i) m &= m - 1ull;
          const int sp = __ffsll((unsigned long long)m) - 1;
          const double igd = 1.0 / (double)g_, sub0d = -(double)(g_ - 1) / (2.0 * g_);
          const double ad = sub0d + igd * (sp % g_), bd = sub0d + igd * (sp / g_), h = 0.5 * igd;
          const Prof<double>& pd = E->pd;
          double X, Y;
          pixel_xy(pd, ci, cj, pi, pj, X, Y);
          const double u = t.noded[kk % 3], v = t.noded[kk / 3];
          sample[f][kk] = eval_profile<double, false>(pd, X + pd.P00 * ad + pd.P01 * bd + h * pd.P00 * u + h * pd.P01 * v,
                                                      Y + pd.P10 * ad + pd.P11 * bd + h * pd.P10 * u + h * pd.P11 * v,
                                                      igd * igd, nullptr);
        }
        __syncthreads();
        if (dec < 0) {
          const int f2 = (int)__popcll(und & ((1ull << gl) - 1ull));
          double rd = 0.0;
#pragma unroll
          for (int q = 0; q < 9; ++q) rd += t.w2d[q] * sample[f2][q];
          dec = fabs(rd - sample[f2][4]) > E->thr * (double)gg ? 1 : 0;
        }
      }
    }
    const bool undecided = !F64 && (__ballot(dec < 0) & gmask) != 0ull;
    const bool deeper = dec == 1 && !undecided;
    if (active && gl < gg && dec == 0 && !undecided) {
      acc[0] = (double)r2;
      if (GRAD) {
#pragma unroll
        for (int q = 0; q < APX_NSLOT; ++q) acc[1 + q] = (double)gs[q];
      }
    }
    // level 3: the group integrates each flagged sub-pixel in turn
    uint64_t todo = (__ballot(deeper) & gmask) >> (GS == 64 ? 0 : grp * GS);
    const float sc3 = ig * ig * ig * ig;
    if (wide) {
      const int nf = (int)__popcll(todo);
      nsub3 += (threadIdx.x >> 6) == 0 ? nf : 0;
      // sub-pixel f, f + 8, ... of the flagged ones
      for (int f0 = 0; f0 < nf; f0 += 256 / GS) {
        uint64_t m = todo;
        const int f = f0 + team;
        for (int i = 0; i < f; ++i) m &= m - 1ull;
        const int sp = m ? __ffsll((unsigned long long)m) - 1 : 0;
        const float xs = __shfl(x2, grp * GS + sp, 64), ys = __shfl(y2, grp * GS + sp, 64);
        if (f < nf) {
          float fs[1 + APX_NSLOT];
          level3_lane<GRAD, GS, ITS>(pf, xs, ys, l3x, l3y, l3w, gl, nq, sc3, fs);
#pragma unroll
          for (int q = 0; q < NV; ++q) subsum[f][q][gl] = fs[q];
        }
      }
      __syncthreads();
      if (team < NV) {
        float first = r2;  // this channel's level-2 value
        if (GRAD) {
#pragma unroll
          for (int q = 0; q < APX_NSLOT; ++q) first = team == 1 + q ? gs[q] : first;
        }
        double a = (gl < gg && dec == 0 && !undecided) ? (double)first : 0.0;
        for (int f = 0; f < nf; ++f) a += (double)subsum[f][team][gl];
        a = half_sum(a);
        if (gl == 0) {
          const int64_t wo = b.gal[gal].work_off;
          if (undecided) {
            if (team == 0) s.redo[wo + atomicAdd(&s.gal_rcnt[gal], 1)] = pix;
          } else {
            // slots 2 .. 6 (channels 3 .. 7) go to planes 1 .. 5
            float* pl = b.planes + wo + pix;
            if (team == 0) pl[0] = (float)a;
            else if (team >= 3 && team - 2 < kNChan) pl[(team - 2) * b.nwork] = (float)(a * E->dvdr[team - 1]);
          }
        }
      }
      __syncthreads();
      continue;
    }
    nsub3 += (int)__popcll(__ballot(deeper));
    while (__ballot(todo != 0ull)) {
      int sp = -1;
      if (todo) {
        sp = __ffsll((unsigned long long)todo) - 1;
        todo &= todo - 1ull;
      }
      const int src = grp * GS + (sp < 0 ? 0 : sp);
      const float xs = __shfl(x2, src, 64), ys = __shfl(y2, src, 64);
      if (sp >= 0) {
        if (FIXED) {
          // this lane's at most ITS samples of the sub-pixel, summed in float32,
          // then into the float64 accumulators
          float fs[1 + APX_NSLOT];
          level3_lane<GRAD, GS, ITS>(pf, xs, ys, l3x, l3y, l3w, gl, nq, sc3, fs);
          acc[0] += (double)fs[0];
          if (GRAD) {
#pragma unroll
            for (int q = 0; q < APX_NSLOT; ++q) acc[1 + q] += (double)fs[1 + q];
          }
        } else {
          for (int e = gl; e < nq; e += GS) {
            const int tt = e / qnn, kk = e % qnn;
            const float a = (sub0 + subd * (float)(tt % g_)) * ig, c = (sub0 + subd * (float)(tt / g_)) * ig;
            const float u = a + h3 * t.node[kk % qn], v = c + h3 * t.node[kk / qn];
            float gv[APX_NSLOT];
            const float val = sersic_f<GRAD>(pf, xs + pf.P00 * u + pf.P01 * v, ys + pf.P10 * u + pf.P11 * v,
                                              sc3, gv);
            const double w = (double)t.w2[kk];
            acc[0] += w * (double)val;
            if (GRAD) {
#pragma unroll
              for (int q = 0; q < APX_NSLOT; ++q) acc[1 + q] += w * (double)gv[q];
            }
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q <= APX_NSLOT; ++q) {
      if (!GRAD && q > 0) break;
      acc[q] = GS == 64 ? wave_sum(acc[q]) : half_sum(acc[q]);
    }
    if (active && gl == 0) {
      const int64_t wo = b.gal[gal].work_off;
      if (undecided) {
        s.redo[wo + atomicAdd(&s.gal_rcnt[gal], 1)] = pix;
      } else {
        float* pl = b.planes + wo + pix;
        pl[0] = (float)acc[0];
        if (GRAD) {
#pragma unroll
          for (int c = 1; c < kNChan; ++c) pl[c * b.nwork] = (float)(acc[1 + c + 1] * E->dvdr[c + 1]);
        }
      }
    }
  }
  if (lane == 0 && nsub3 > 0) atomicAdd(&s.cnt[F64 ? 7 : 6], nsub3);
}

// ---------------------------------------------------------------------------
// The float32 level-2/3 pass for the default quadrature (quad_level 3,
// gridding 5) with one lane per level-2 sub-pixel: a workgroup takes 10
// refined pixels at a time (250 of its 256 lanes; a 32-lane group per pixel
// keeps only 25 busy).  Each lane integrates its sub-pixel with the 3 x 3
// Gauss-Legendre rule; the sub-pixels the level-2 test flags are collected in
// workgroup order and integrated a wave each (225 level-3 samples); the 25
// sub-pixel sums of a pixel are added in float64 in sub-pixel order.  Same decisions and outputs as
// integrate_kernel<..., F64 = false, 3, 5>; a pixel with an undecided test goes
// to the redo list unwritten.
//
// Value-only level 2 evaluates in the rotated, stretched frame: the nodes of
// a sub-pixel sit at R(x_s) +- A, +- B (A, B: the rotated node steps along the
// two pixel axes) and each node's weight and the sampling scale fold into the
// exponent, w I = exp2(nbl2e pw + log2(amp scale w) - nbl2e).
constexpr int kWgPix = 10;  // refined pixels a workgroup takes at once
constexpr int kWgSub = 25;  // level-2 sub-pixels a pixel (gridding 5)


template <bool GRAD>
__global__ __launch_bounds__(256) void integrate_wg_kernel(apx_batch b, Scratch s, QuadTab t) {
  constexpr int NV = GRAD ? 1 + APX_NSLOT : 1;
  __shared__ double sums[NV][256];     // per-lane sub-pixel totals (level 2 or 3)
  __shared__ int flagged[256];         // slots whose sub-pixel goes to level 3, in slot order
  __shared__ int wcnt[4], undec[kWgPix], nflag;
  __shared__ float fx[256], fy[256];   // level-2 sub-pixel centres (plane offsets)
  __shared__ int fgal[kWgPix];
  const int slot = threadIdx.x, lane = slot & 63, w = slot >> 6;
  const int px = slot / kWgSub, sub = slot - kWgSub * px;
  const int total = s.cnt[3];
  constexpr float ig = 0.2f, sub0 = -0.4f, subd = 0.2f;
  // level-2 node steps in plane units: (g3 h) P e_i with h = ig / 2 and g3 = sqrt(3/5)
  const float P00 = (float)b.P[0], P01 = (float)b.P[1], P10 = (float)b.P[2], P11 = (float)b.P[3];
  const float hn = 0.5f * ig * t.node[2];  // node 2 = +sqrt(3/5)
  // log2 of the level-2 scale ig^2 times the corner, edge and centre weights
  const float l2sc = 2.0f * __builtin_amdgcn_logf(ig);
  const float lwc = l2sc + t.lw[0], lwe = l2sc + t.lw[1], lw0 = l2sc + t.lw[4];
  // level-3 samples of this lane, 64 rd + lane (225 in all): sub-sub-pixel tt, node kk
  float l3x[4], l3y[4], l3w[4];
#pragma unroll
  for (int rd = 0; rd < 4; ++rd) {
    const int e = 64 * rd + lane;
    l3x[rd] = l3y[rd] = l3w[rd] = 0.0f;
    if (e >= 225) continue;
    const int tt = e / 9, kk = e % 9;
    const float h3 = 0.5f * ig * ig;
    // written out: the last round's tt / 5 is a constant, and the compiler would fold it differently
    const float nu = h3 * t.node[kk % 3], nv = h3 * t.node[kk / 3];
    const float u = fmaf(ig, fmaf(subd, (float)(tt % 5), sub0), nu), v = fmaf(ig, fmaf(subd, (float)(tt / 5), sub0), nv);
    l3x[rd] = fmaf(P00, u, P01 * v);
    l3y[rd] = fmaf(P10, u, P11 * v);
    l3w[rd] = t.w2[kk];
  }
  const float sc3 = ig * ig * ig * ig;
  int nsub3 = 0;
  // pixels a workgroup takes at once: fewer than kWgPix where the list is short,
  // so that it spreads over the CUs
  const int np = max(1, min(kWgPix, (total + (int)gridDim.x - 1) / (int)gridDim.x));
  for (int k0 = blockIdx.x * np; k0 < total; k0 += gridDim.x * np) {
    const int k = k0 + px;
    const bool active = px < np && k < total;
    int gal = 0, pix = 0;
    if (active) {
      const int2 q = s.dq[k];
      gal = q.x;
      pix = q.y;
    }
    const GalEval* E = s.ev + gal;
    const Prof<float> pf = E->pf;
    const int nxw = active ? E->nxw : 1;
    float X0, Y0;
    pixel_xy(pf, E->ci, E->cj, pix % nxw, pix / nxw, X0, Y0);
    const float x2 = X0 + pf.P00 * (sub0 + subd * (float)(sub % 5)) + pf.P01 * (sub0 + subd * (float)(sub / 5));
    const float y2 = Y0 + pf.P10 * (sub0 + subd * (float)(sub % 5)) + pf.P11 * (sub0 + subd * (float)(sub / 5));
    int dec = 0;
    float r2 = 0.0f, gs[APX_NSLOT];
    if (active) {
      float c2 = 0.0f;
      if (GRAD) {
        r2 = quad3_grad(pf, t, x2, y2, 0.5f * ig, l2sc, gs, c2);
      } else {
        // rotated frame: sub-pixel centre and the node steps along the pixel axes
        float xr, yr, ax, ay, bx, by;
        rot(pf, x2, y2, xr, yr);
        rot(pf, hn * pf.P00, hn * pf.P10, ax, ay);
        rot(pf, hn * pf.P01, hn * pf.P11, bx, by);
        const float base = pf.l2amp - pf.nbl2e;
        float cen = 0.0f;
        r2 = gl3_rot(pf, xr, yr, ax, ay, bx, by, base + lwc, base + lwe, base + lw0, cen);
        c2 = cen * t.inv_w4;
      }
      if (t.max_depth > 2) dec = band_test(r2, c2, E->thr * 25.0);
    }
    // flag list (slot order) and undecided pixels
    if (slot < kWgPix) undec[slot] = 0;
    const uint64_t bal = __ballot(dec == 1);
    if (lane == 0) wcnt[w] = (int)__popcll(bal);
    __syncthreads();
    if (dec < 0) undec[px] = 1;
    if (dec == 1) {
      int off = 0;
      for (int i = 0; i < w; ++i) off += wcnt[i];
      flagged[off + (int)__popcll(bal & ((lane == 0) ? 0ull : (~0ull >> (64 - lane))))] = slot;
      fx[slot] = x2;
      fy[slot] = y2;
    }
    if (sub == 0 && active) fgal[px] = gal;
    if (slot == 0) nflag = wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
    // level-2 contribution of this sub-pixel
    sums[0][slot] = (active && dec == 0) ? (double)r2 : 0.0;
    if (GRAD) {
#pragma unroll
      for (int q = 0; q < APX_NSLOT; ++q) sums[1 + q][slot] = (active && dec == 0) ? (double)gs[q] : 0.0;
    }
    __syncthreads();
    const int nf = nflag;
    nsub3 += nf;
    // level 3: a wave a flagged sub-pixel, its 225 samples as 4 rounds of 64 lanes,
    // each round summed over the wave.  (The whole workgroup on one sub-pixel after
    // another took two barriers and an LDS round trip each; here the flagged
    // sub-pixels of ten pixels run four abreast.)
    for (int f = w; f < nf; f += 4) {
      const int fs = flagged[f];
      const GalEval* F = s.ev + fgal[fs / kWgSub];
      const Prof<float> pg = F->pf;
      const float cx = fx[fs], cy = fy[fs];
      double tot[NV];
#pragma unroll
      for (int rd = 0; rd < 4; ++rd) {
        float v[NV];
#pragma unroll
        for (int q = 0; q < NV; ++q) v[q] = 0.0f;
        if (rd < 3 || lane < 225 - 192) {
          float gv[APX_NSLOT];
          const float X = cx + l3x[rd], Y = cy + l3y[rd];
          const float val = GRAD ? sersic_f<true>(pg, X, Y, sc3, gv) : sersic_value_f(pg, X, Y, sc3);
          {
            // the weighted sample is rounded before the sum over the wave (not
            // folded into its first addition), whether the round is full or not
#pragma clang fp contract(off)
            v[0] = l3w[rd] * val;
            if (GRAD) {
#pragma unroll
              for (int q = 0; q < APX_NSLOT; ++q) v[1 + q] = l3w[rd] * gv[q];
            }
          }
        }
#pragma unroll
        for (int q = 0; q < NV; ++q) {
          const double r = (double)wave_sum(v[q]);
          tot[q] = rd == 0 ? r : tot[q] + r;
        }
      }
      if (lane == 0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) sums[q][fs] = tot[q];
      }
    }
    __syncthreads();
    // per pixel and channel: the 25 sub-pixel totals in order
    if (slot < np * NV) {
      const int p = slot / NV, q = slot % NV;
      const int kk = k0 + p;
      if (kk < total && !undec[p]) {
        double acc = 0.0;
        for (int j = 0; j < kWgSub; ++j) acc += sums[q][kWgSub * p + j];
        const int2 e = s.dq[kk];
        const int64_t wo = b.gal[e.x].work_off;
        if (q == 0) {
          b.planes[wo + e.y] = (float)acc;
        } else if (q >= 3 && q - 2 < kNChan) {
          // partial slot q - 1 goes to plane q - 2 (slots 2..6 -> planes 1..5)
          b.planes[(int64_t)(q - 2) * b.nwork + wo + e.y] = (float)(acc * s.ev[e.x].dvdr[q - 1]);
        }
      } else if (kk < total && q == 0) {
        const int2 e = s.dq[kk];
        const int64_t wo = b.gal[e.x].work_off;
        s.redo[wo + atomicAdd(&s.gal_rcnt[e.x], 1)] = e.y;
      }
    }
    __syncthreads();
  }
  if (slot == 0 && nsub3 > 0) atomicAdd(&s.cnt[6], nsub3);
}

// ---------------------------------------------------------------------------
// convolution of every listed tile, with the per-fit reductions of the stage
// folded into the epilogue as per-tile partial sums:
//   EPI_OUT     value -> out
//   EPI_NORMAL  value -> out (model0), centre derivatives -> J cols 0, 1,
//               partial planes -> J cols 2..6; normal_kernel then forms
//               J^T W J, J^T W (Y - m0), chi2(m0) per tile  (lm.py:256-260)
//   EPI_RPP     J^T (2 / d) (W (m(x + d h) - m0) / d - W J h), d = 0.1
//                                                           (lm.py:276-280)
//   EPI_CHI2    sum W (Y - m)^2 of the tile                 (lm.py:290-292)
enum : int { EPI_OUT = 0, EPI_NORMAL = 1, EPI_RPP = 2, EPI_CHI2 = 3 };


// dynamic LDS of conv_kernel: the staged input tile, reused for the
// cross-wave reduction of one kernel's outputs at a time
__host__ __device__ inline int conv_stage_floats(int kmax) {
  const int tile = 8 * fast_nt(kmax) * (64 + kmax - 1);
  const int red = 4 * kRYF * 64;
  return tile > red ? tile : red;
}
__host__ inline size_t conv_lds_bytes(int kmax) { return sizeof(float) * (size_t)conv_stage_floats(kmax); }
constexpr size_t kConvStaticLds = sizeof(double) * 4 * 8;
// MFMA passes a tile: 3 kernels of the value plane and the partial planes, or the value alone
__host__ __device__ constexpr int mfma_passes(bool jac) { return jac ? kConvChan + 2 : 1; }

// The probe (rpp) and trial (chi2) epilogues of one output pixel, summed into
// rd[] in float64 (lm.py:276-292)
template <int MODE>
__device__ __forceinline__ void epilogue_pixel(const apx_batch& b, const GalState* st, int64_t p,
                                               float m, double* rd) {
  if (MODE == EPI_RPP) {
    constexpr double d = 0.1;
    float jr[NP];
    double jh = 0.0;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      jr[i] = b.jac[(int64_t)i * b.npix + p];
      jh += (double)jr[i] * st->h[i];
    }
    const double wt = (double)b.weight[p];
    const double v = (2.0 / d) * (wt * ((double)m - (double)b.model0[p]) / d - wt * jh);
#pragma unroll
    for (int i = 0; i < NP; ++i) rd[i] += (double)jr[i] * v;
  } else if (MODE == EPI_CHI2) {
    const double dd = (double)b.data[p] - (double)m;
    rd[0] += (double)b.weight[p] * dd * dd;
  }
}

// The probe and trial epilogues of 4 consecutive output pixels p0 .. p0 + 3
// of one row (valid[k]: pixel k exists), with the same arithmetic as
// epilogue_pixel, pixel by pixel in order.  h is the fit's step, read once a
// tile.  When all 4 exist and the rows they are read from are 16-byte
// aligned (`vec`), each input is one 4-wide load.
template <int MODE>
__device__ __forceinline__ void epilogue_quad(const apx_batch& b, const double* h, int64_t p0, const bool* valid,
                                              bool vec, const float* m, double* rd) {
  // the inputs: the 7 J columns, the model at x and the weight (probe), or the
  // data and the weight (trial), all requested before any is used
  constexpr int NA = MODE == EPI_RPP ? NP + 2 : 2;
  const float* src[NA];
  if (MODE == EPI_RPP) {
#pragma unroll
    for (int i = 0; i < NP; ++i) src[i] = b.jac + (int64_t)i * b.npix + p0;
    src[NP] = b.model0 + p0;
    src[NP + 1] = b.weight + p0;
  } else {
    src[0] = b.data + p0;
    src[1] = b.weight + p0;
  }
  float a[NA][4];
  if (vec) {
    float4 q[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) q[i] = *reinterpret_cast<const float4*>(src[i]);
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      a[i][0] = q[i].x;
      a[i][1] = q[i].y;
      a[i][2] = q[i].z;
      a[i][3] = q[i].w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) a[i][k] = valid[k] ? src[i][k] : 0.0f;
  }
  if (MODE == EPI_RPP) {
    constexpr double d = 0.1;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (!valid[k]) continue;
      double jh = 0.0;
#pragma unroll
      for (int i = 0; i < NP; ++i) jh += (double)a[i][k] * h[i];
      const double w = (double)a[NP + 1][k];
      const double v = (2.0 / d) * (w * ((double)m[k] - (double)a[NP][k]) / d - w * jh);
#pragma unroll
      for (int i = 0; i < NP; ++i) rd[i] += (double)a[i][k] * v;
    }
  } else if (MODE == EPI_CHI2) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (!valid[k]) continue;
      const double dd = (double)a[0][k] - (double)m[k];
      rd[0] += (double)a[1][k] * dd * dd;
    }
  }
}

// block sum of rd[0..W) into the tile's partial sums
template <int W>
__device__ __forceinline__ void tile_partial(double (&redd)[4][8], const double* rd, double* part,
                                             int lane, int w) {
#pragma unroll
  for (int i = 0; i < W; ++i) {
    const double v = wave_sum(rd[i]);
    if (lane == 0) redd[w][i] = v;
  }
  __syncthreads();
  if (threadIdx.x < W) {
    const int i = threadIdx.x;
    part[i] = redd[0][i] + redd[1][i] + redd[2][i] + redd[3][i];
  }
  __syncthreads();
}

// Tile entry of this workgroup in the round of tile entries starting at
// `base` (count c), or -1.  Workgroups go to the 8 XCDs round robin; with a
// grid that is a multiple of 8 the round's entries are cut into 8 contiguous
// runs, one per XCD, so the tiles of one cutout, which re-read each other's
// halo rows, run on one XCD at about the same time and find those rows in its
// L2, while a short list still spreads over every XCD.
__device__ __forceinline__ int xcd_tile(int base, int c) {
  const int nb = (int)gridDim.x, b = (int)blockIdx.x;
  const int m = min(nb, c - base);
  if (nb & 7) return b < m ? base + b : -1;
  const int q = (m + 7) >> 3, slot = b >> 3, x = b & 7;
  const int k = x * q + slot;
  return (slot < q && k < m) ? base + k : -1;
}

// VALU convolution (kernels wider than kMfmaMax): the 64 x kTR tile in two
// halves of kRYF rows; after the cross-wave reduction each wave owns output
// rows w and w + 4 of a half (lane = column) for every kernel and channel
template <int MODE>
__global__ __launch_bounds__(256) void conv_kernel(apx_batch b, Scratch s, float* out) {
  extern __shared__ float smem[];
  __shared__ double redd[4][8];  // kConvStaticLds
  constexpr bool JAC = MODE == EPI_NORMAL;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wu = __builtin_amdgcn_readfirstlane(w);
  constexpr int NKmax = JAC ? 3 : 1;
  constexpr int nchan = JAC ? kConvChan : 1;
  constexpr int W = MODE == EPI_RPP ? NP : 1;
  for (int base = 0; base < s.cnt[2]; base += gridDim.x) {
    const int k = xcd_tile(base, s.cnt[2]);
    if (k < 0) continue;
    const int2 e = s.tile_list[k];
    const int g = __builtin_amdgcn_readfirstlane(e.x);
    const apx_batch_galaxy G = b.gal[g];
    const GalState* st = st_of(b, g);
    const float ie_scale = JAC ? (float)(kLn10 * s.ev[g].dvdr[NP - 1]) : 0.0f;
    const int nxw = G.nx + G.pw + 1, nyw = G.ny + G.ph + 1;  // cutout + 2 * border
    const int ntx = (G.nx + 63) / 64;
    const int ox0 = (e.y % ntx) * 64;
    const int kh = G.ph + 2, kw = G.pw + 2;
    const int nT = fast_nt(kh), kts = fast_kts(kh), rows = 8 * nT, LW = 64 + kw - 1;
    const int64_t tile = G.tile_off + e.y;
    // output (ox, oy) sits at working (bx + ox, by + oy); taps span +-(k-1)/2 = border
    const float* kt = b.taps + G.tap_off;
    const int ox = ox0 + lane;
    double rd[W];
#pragma unroll
    for (int i = 0; i < W; ++i) rd[i] = 0.0;
    for (int half = 0; half < kTR / kRYF; ++half) {
      const int oy0 = (e.y / ntx) * kTR + half * kRYF;
      bool valid[2];
      int64_t pp[2];
#pragma unroll
      for (int sl = 0; sl < 2; ++sl) {
        const int oy = oy0 + w + 4 * sl;
        valid[sl] = ox < G.nx && oy < G.ny;
        pp[sl] = G.pix_off + (int64_t)oy * G.nx + ox;
      }
      for (int c = 0; c < nchan; ++c) {
        const float* plane = b.planes + (int64_t)c * b.nwork + G.work_off;
        __syncthreads();
        for (int q = threadIdx.x; q < rows * LW; q += 256) {
          const int gy = oy0 + q / LW, gx = ox0 + q % LW;
          smem[q] = (gy < nyw && gx < nxw) ? plane[(int64_t)gy * nxw + gx] : 0.0f;
        }
        __syncthreads();
        const int nk = (JAC && c == 0) ? 3 : 1;
        float acc[NKmax][kRYF];
#pragma unroll
        for (int kk = 0; kk < NKmax; ++kk)
#pragma unroll
          for (int r = 0; r < kRYF; ++r) acc[kk][r] = 0.0f;
        conv_accumulate<NKmax>(smem, LW, lane, wu, nT, kw, kts, nk, kt, acc);
#pragma unroll
        for (int kk = 0; kk < NKmax; ++kk) {
          if (kk >= nk) break;
          __syncthreads();
#pragma unroll
          for (int r = 0; r < kRYF; ++r) smem[(w * kRYF + r) * 64 + lane] = acc[kk][r];
          __syncthreads();
          const int col = c == 0 ? kk - 1 : c + 1;  // J column, -1 for the value
#pragma unroll
          for (int sl = 0; sl < 2; ++sl) {
            const int r = w + 4 * sl;
            float sum = 0.0f;
#pragma unroll
            for (int ww = 0; ww < 4; ++ww) sum += smem[(ww * kRYF + r) * 64 + lane];
            if (!valid[sl]) continue;
            if (JAC) {
              if (col < 0) {
                out[pp[sl]] = sum;
                b.jac[(int64_t)(NP - 1) * b.npix + pp[sl]] = ie_scale * sum;
              } else {
                b.jac[(int64_t)col * b.npix + pp[sl]] = sum;
              }
            } else if (MODE == EPI_OUT) {
              out[pp[sl]] = sum;
            } else {
              epilogue_pixel<MODE>(b, st, pp[sl], sum, rd);
            }
          }
        }
      }
    }
    if (MODE == EPI_RPP || MODE == EPI_CHI2) tile_partial<W>(redd, rd, s.part + tile * kPart, lane, w);
  }
}

// ---------------------------------------------------------------------------
// MFMA convolution (kernels up to kMfmaMax): the Toeplitz formulation of
// conv_common.h (mfma_columns), one 16 x 16 output block per wave of the
// 64 x kTR tile.  A work item is one (tile, plane, kernel) pass: its LDS is one
// staged plane and one tap table, so at least two workgroups share a CU and one
// loads while the other multiplies.  Both arrive by stage_rows.  Bound by the
// FP32 matrix pipe.  With a tile's 7 passes in one workgroup (three tap tables:
// one workgroup a CU for 67-px kernels) and rows copied through registers one
// wait at a time, 125 sources on 1024 x 1024 took 5.83 ms; 2.78 ms so.
template <int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void conv_mfma_kernel(apx_batch b, Scratch s, float* out) {
  extern __shared__ float smem[];
  __shared__ double redd[4][8];  // kConvStaticLds
  constexpr bool JAC = MODE == EPI_NORMAL;
  constexpr int W = MODE == EPI_RPP ? NP : 1;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lm = lane & 15, lk = lane >> 4;
  const int total = s.cnt[2] * mfma_passes(JAC);
  for (int base = 0; base < total; base += gridDim.x) {
    const int item = xcd_tile(base, total);
    if (item < 0) continue;
    // passes 0 .. 2: the value plane with K, dK/dcx, dK/dcy; 3 ..: a partial plane with K
    const int pass = item % mfma_passes(JAC), c = pass < 3 ? 0 : pass - 2, kk = pass < 3 ? pass : 0;
    const int2 e = s.tile_list[item / mfma_passes(JAC)];
    const int g = __builtin_amdgcn_readfirstlane(e.x);
    const apx_batch_galaxy G = b.gal[g];
    const GalState* st = st_of(b, g);
    const int nxw = G.nx + G.pw + 1, nyw = G.ny + G.ph + 1;  // cutout + 2 * border
    const int ntx = (G.nx + 63) / 64;
    const int ox0 = (e.y % ntx) * 64, oy0 = (e.y / ntx) * kTR;
    const int kh = G.ph + 2, kw = G.pw + 2;
    const int nks = mf_nks(kh), DD = mf_dd(kh), kts = fast_kts(kh);
    const int rows = mf_rows(kh), cols = 64 + kw - 1;
    float* tin = smem;             // rows x kMfLW
    float* tab = smem + rows * kMfLW; // [kx][dd]
    __syncthreads();  // the previous item's readers are done with LDS
    stage_rows(b.planes + (int64_t)c * b.nwork + G.work_off, nxw, nxw, nyw, ox0, oy0, rows, cols, tin, kMfLW);
    // tap-table row kx: dd -> Kf[dd - 15][kx] = KT[kk][kx][dd - 8], zero outside KT's row
    stage_rows(b.taps + G.tap_off + (int64_t)kk * kw * kts, kts, kts, kw, -8, 0, kw, DD, tab, DD);
    if (threadIdx.x < 16) tab[kw * DD + threadIdx.x] = 0.0f;  // the last column's trailing zeros
    // this lane's 4 output pixels: x = 16 w + 4 lk + i, row lm
    const int oy = oy0 + lm;
    bool valid[4];
    int64_t pp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ox = ox0 + 16 * w + 4 * lk + i;
      valid[i] = ox < G.nx && oy < G.ny;
      pp[i] = G.pix_off + (int64_t)oy * G.nx + ox;
    }
    double rd[W];
#pragma unroll
    for (int i = 0; i < W; ++i) rd[i] = 0.0;
    __builtin_amdgcn_s_waitcnt(0);  // this wave's rows have landed in LDS
    __syncthreads();
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    if (ox0 + 16 * w < G.nx)  // a wave past the cutout's right edge has no output
      acc = mfma_block(nks, tin + lk * kMfLW + 16 * w + lm, tab + lk - lm + 15, kw, DD);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (!valid[i]) continue;
      if (JAC) {
        const int col = c == 0 ? kk - 1 : c + 1;  // J column, -1 for the value
        if (col < 0) {
          out[pp[i]] = acc[i];
          b.jac[(int64_t)(NP - 1) * b.npix + pp[i]] = (float)(kLn10 * s.ev[g].dvdr[NP - 1]) * acc[i];
        } else {
          b.jac[(int64_t)col * b.npix + pp[i]] = acc[i];
        }
      } else if (MODE == EPI_OUT) {
        out[pp[i]] = acc[i];
      } else {
        epilogue_pixel<MODE>(b, st, pp[i], acc[i], rd);
      }
    }
    if (MODE == EPI_RPP || MODE == EPI_CHI2) tile_partial<W>(redd, rd, s.part + (G.tile_off + e.y) * kPart, lane, w);
  }
}

// ---------------------------------------------------------------------------
// Separable convolution (conv_impl 3, every PSF rank one; prepare_separable):
// per plane of the 64 x kTR tile, a column pass
//   hu[t][u] = sum_a uh_f[a] in[t + a][u]      (u over the 64 + kw - 1 staged columns)
// and a row pass  out[t][x] = sum_b vh_f[b] hu[t][x + b],  2 (kh + kw) flops an
// output instead of 2 kh kw.  In the Jacobian stage the value plane also takes
// the column pass with uh' (hu2) and gives, with C_x = hu * vh' and
// C_y = hu2 * vh, the centre columns P^-1-mixed as the MFMA taps are:
//   dm/dcx = P^-1[0][0] C_x + P^-1[1][0] C_y,  dm/dcy = P^-1[0][1] C_x + P^-1[1][1] C_y.
// The tap vectors are padded with zeros to kh4 = kh rounded up to 4 (kw4
// likewise), so both passes run whole 4-tap steps; a zero tap adds exactly 0.
// Layout and overlap:
//  * the staged input is row-major with a compile-time pitch SP (96 or 128
//    floats), so the column pass's LDS reads take immediate offsets; rows go
//    from HBM straight into LDS (buffer loads with the lds modifier, no
//    registers), and return 0 past the end of the plane;
//  * the next (tile, plane)'s rows are requested as soon as the column pass
//    has read the current ones, so they arrive during the row pass, the
//    stores and the next item's set-up;
//  * a column-pass item (row group rg, column u) slides a 4-row window down
//    column u; the taps come through the scalar cache (one SGPR operand an FMA);
//  * hu is row-major with pitch hp = 1 mod 4; thread (ty, x4) of the row pass
//    owns the 4 consecutive outputs 4 x4 .. 4 x4 + 3 of row ty and slides a
//    4-wide window along the row (lanes 4 x4 + (ty hp mod 4) meet distinct banks).
// Staged columns past the plane's width hold the next row's values (or 0 past
// the plane's end): they reach only outputs past the cutout's width.
typedef const __attribute__((address_space(4))) float* ctaps;

constexpr int kSepMax = 61;  // widest kernel the separable convolution takes (LDS)
__host__ __device__ inline int sp_pitch(int cols) { return cols + ((1 - cols) & 3); }  // >= cols, 1 mod 4
// staged-row pitch for kernels up to kmax columns: 64 + kw4 - 1 columns fit
__host__ inline int sp_stage_pitch(int kmax) { return 63 + sp_k4(kmax) <= 96 ? 96 : 128; }
__host__ inline size_t sep_lds_bytes(int kmax, bool jac) {
  const int k4 = sp_k4(kmax), rows = kTR + k4 - 1, cols = 64 + k4 - 1;
  return sizeof(float) * ((size_t)rows * sp_stage_pitch(kmax) + (jac ? 2 : 1) * (size_t)kTR * sp_pitch(cols));
}

// One tile entry of the separable convolution.
struct SepTile {
  int g, nxw, nyw, ox0, oy0, kh4, kw4, rows, cols;
  int64_t work_off, pix_off, tile;
  int nx, ny;
  int64_t tap_off;
};

__device__ __forceinline__ SepTile sep_tile(const apx_batch& b, const Scratch& s, int k) {
  const int2 e = s.tile_list[k];
  SepTile T;
  T.g = __builtin_amdgcn_readfirstlane(e.x);
  const apx_batch_galaxy G = b.gal[T.g];
  T.nx = G.nx, T.ny = G.ny;
  T.nxw = G.nx + G.pw + 1, T.nyw = G.ny + G.ph + 1;  // cutout + 2 * border
  const int ntx = (G.nx + 63) / 64;
  T.ox0 = (e.y % ntx) * 64, T.oy0 = (e.y / ntx) * kTR;
  T.kh4 = sp_k4(G.ph + 2), T.kw4 = sp_k4(G.pw + 2);
  T.rows = kTR + T.kh4 - 1, T.cols = 64 + T.kw4 - 1;
  T.work_off = G.work_off, T.pix_off = G.pix_off, T.tile = G.tile_off + e.y;
  T.tap_off = G.tap_off;
  return T;
}

// Request plane c of tile T into tin (rows x SP, row-major): wave w the rows
// w, w + 4, ..., each row one or two 64-lane loads written by the memory
// system straight into LDS.  Completion: vmcnt.
template <int SP>
__device__ __forceinline__ void sep_stage(const apx_batch& b, const SepTile& T, int c, float* tin) {
  const int64_t off0 = (int64_t)T.oy0 * T.nxw + T.ox0;
  // every field of the resource is uniform: read it from lane 0 so that the
  // compiler keeps it in SGPRs (no per-load uniformity loop)
  const uint64_t a = (uint64_t)(b.planes + (int64_t)c * b.nwork + T.work_off + off0);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  const int nrec = __builtin_amdgcn_readfirstlane((int)(((int64_t)T.nyw * T.nxw - off0) * 4));
  const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
      reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), (short)0, nrec, kBufWord3);
  const int lane = threadIdx.x & 63;
  for (int t = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); t < T.rows; t += 4) {
    const int vo = (t * T.nxw + lane) * 4;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_ptr)(tin + t * SP), 4, vo, 0, 0, 0);
    if (lane < SP - 64) __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_ptr)(tin + t * SP + 64), 4, vo + 256, 0, 0, 0);
  }
}

// Column pass of item (rg, u): rows 4 rg .. 4 rg + 3 of hu (and hu2) at column u.
template <bool TWO, int SP>
__device__ __forceinline__ void sconv_column(const float* tin, float* hu, float* hu2, int hp, int rg, int u, int kh4,
                                             ctaps fu, ctaps fdu) {
  const float* col = tin + 4 * rg * SP + u;
  float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f, d0 = 0.0f, d1 = 0.0f, d2 = 0.0f, d3 = 0.0f;
  float r0 = col[0], r1 = col[SP], r2 = col[2 * SP];
  for (int a = 0; a < kh4; a += 4) {
    const float* c = col + a * SP;
    const float r[7] = {r0, r1, r2, c[3 * SP], c[4 * SP], c[5 * SP], c[6 * SP]};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float f = fu[a + q];
      a0 = fmaf(f, r[q], a0);
      a1 = fmaf(f, r[q + 1], a1);
      a2 = fmaf(f, r[q + 2], a2);
      a3 = fmaf(f, r[q + 3], a3);
      if (TWO) {
        const float fd = fdu[a + q];
        d0 = fmaf(fd, r[q], d0);
        d1 = fmaf(fd, r[q + 1], d1);
        d2 = fmaf(fd, r[q + 2], d2);
        d3 = fmaf(fd, r[q + 3], d3);
      }
    }
    r0 = r[4];
    r1 = r[5];
    r2 = r[6];
  }
  float* h = hu + 4 * rg * hp + u;
  h[0] = a0;
  h[hp] = a1;
  h[2 * hp] = a2;
  h[3 * hp] = a3;
  if (TWO) {
    float* h2 = hu2 + 4 * rg * hp + u;
    h2[0] = d0;
    h2[hp] = d1;
    h2[2 * hp] = d2;
    h2[3 * hp] = d3;
  }
}

// Row pass of thread (ty, x4): o[i] = conv(hu, vh) at row ty, column 4 x4 + i;
// with TWO also ox_ = conv(hu, vh') and oy_ = conv(hu2, vh).
template <bool TWO>
__device__ __forceinline__ void sconv_row(const float* hu, const float* hu2, int hp, int kw4, ctaps fv, ctaps fdv,
                                          float* o, float* ox_, float* oy_) {
  const int ty = threadIdx.x >> 4, x4 = threadIdx.x & 15;
  const float* h = hu + ty * hp + 4 * x4;
  const float* h2 = hu2 + ty * hp + 4 * x4;
  float o0 = 0.0f, o1 = 0.0f, o2 = 0.0f, o3 = 0.0f;
  float p0 = 0.0f, p1 = 0.0f, p2 = 0.0f, p3 = 0.0f;  // TWO: conv(hu, vh')
  float q0 = 0.0f, q1 = 0.0f, q2 = 0.0f, q3 = 0.0f;  // TWO: conv(hu2, vh)
  float w0 = h[0], w1 = h[1], w2 = h[2];
  float z0 = TWO ? h2[0] : 0.0f, z1 = TWO ? h2[1] : 0.0f, z2 = TWO ? h2[2] : 0.0f;
  for (int bb = 0; bb < kw4; bb += 4) {
    const float wv[7] = {w0, w1, w2, h[bb + 3], h[bb + 4], h[bb + 5], h[bb + 6]};
    float zv[7];
    if (TWO) {
      zv[0] = z0, zv[1] = z1, zv[2] = z2;
      zv[3] = h2[bb + 3], zv[4] = h2[bb + 4], zv[5] = h2[bb + 5], zv[6] = h2[bb + 6];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float f = fv[bb + q];
      o0 = fmaf(f, wv[q], o0);
      o1 = fmaf(f, wv[q + 1], o1);
      o2 = fmaf(f, wv[q + 2], o2);
      o3 = fmaf(f, wv[q + 3], o3);
      if (TWO) {
        const float fd = fdv[bb + q];
        p0 = fmaf(fd, wv[q], p0);
        p1 = fmaf(fd, wv[q + 1], p1);
        p2 = fmaf(fd, wv[q + 2], p2);
        p3 = fmaf(fd, wv[q + 3], p3);
        q0 = fmaf(f, zv[q], q0);
        q1 = fmaf(f, zv[q + 1], q1);
        q2 = fmaf(f, zv[q + 2], q2);
        q3 = fmaf(f, zv[q + 3], q3);
      }
    }
    w0 = wv[4], w1 = wv[5], w2 = wv[6];
    if (TWO) z0 = zv[4], z1 = zv[5], z2 = zv[6];
  }
  o[0] = o0, o[1] = o1, o[2] = o2, o[3] = o3;
  if (TWO) {
    ox_[0] = p0, ox_[1] = p1, ox_[2] = p2, ox_[3] = p3;
    oy_[0] = q0, oy_[1] = q1, oy_[2] = q2, oy_[3] = q3;
  }
}

// Work items are (tile, plane) pairs in order: the tiles of this workgroup
// (xcd_tile rounds), each with its NPL planes.
template <int MODE, int SP>
__global__ __launch_bounds__(256) void sconv_kernel(apx_batch b, Scratch s, float* out) {
  extern __shared__ float smem[];
  __shared__ double redd[4][8];  // kConvStaticLds
  constexpr bool JAC = MODE == EPI_NORMAL;
  constexpr int NPL = JAC ? kConvChan : 1;
  constexpr int W = MODE == EPI_RPP ? NP : 1;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int ty = threadIdx.x >> 4, x4 = threadIdx.x & 15;
  const double det = b.P[0] * b.P[3] - b.P[1] * b.P[2];
  const float pi00 = (float)(b.P[3] / det), pi01 = (float)(-b.P[1] / det);
  const float pi10 = (float)(-b.P[2] / det), pi11 = (float)(b.P[0] / det);
  const ctaps taps = (ctaps)b.taps;
  const int cnt = s.cnt[2];
  const bool aligned16 = ((reinterpret_cast<uintptr_t>(b.jac) | reinterpret_cast<uintptr_t>(b.model0) |
                           reinterpret_cast<uintptr_t>(b.weight) | reinterpret_cast<uintptr_t>(b.data)) & 15) == 0;
  // LDS: the staged rows (rows x SP) of any tile of the launch, then hu (and
  // hu2) at a fixed place, so a tile's rows can arrive while the previous
  // tile's row pass still reads hu
  float* tin = smem;
  float* hu = tin + (kTR + sp_k4(b.max_kernel) - 1) * SP;
  // next tile entry of this workgroup from round `base` on (base advances to
  // that entry's round), or -1
  auto next_tile = [&](int& base) {
    for (; base < cnt; base += (int)gridDim.x) {
      const int k = xcd_tile(base, cnt);
      if (k >= 0) return k;
    }
    return -1;
  };
  int base = 0;
  const int k0 = next_tile(base);
  if (k0 < 0) return;
  SepTile T = sep_tile(b, s, k0);
  sep_stage<SP>(b, T, 0, tin);
  while (true) {
    const int hp = sp_pitch(T.cols);
    float* hu2 = hu + kTR * hp;  // kTR x hp (Jacobian stage, value plane)
    const ctaps fu = taps + T.tap_off;  // uh | vh | uh' | vh', each zero-padded to kh4 or kw4
    const ctaps fv = fu + T.kh4, fdu = fv + T.kw4, fdv = fdu + T.kh4;
    const GalState* st = st_of(b, T.g);
    const float ie_scale = JAC ? (float)(kLn10 * s.ev[T.g].dvdr[NP - 1]) : 0.0f;
    double hst[NP];  // the fit's step (probe epilogue), read once a tile
#pragma unroll
    for (int i = 0; i < NP; ++i) hst[i] = MODE == EPI_RPP ? st->h[i] : 0.0;
    // column-pass items of this thread, packed as rg * 256 + u (-1: none)
    int it0 = -1, it1 = -1;
    {
      const int i0 = (int)threadIdx.x, i1 = i0 + 256;
      if (i0 < 4 * T.cols) it0 = (i0 / T.cols) * 256 + i0 % T.cols;
      if (i1 < 4 * T.cols) it1 = (i1 / T.cols) * 256 + i1 % T.cols;
    }
    const int oy = T.oy0 + ty;
    bool valid[4];
    int64_t pp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ox = T.ox0 + 4 * x4 + i;
      valid[i] = ox < T.nx && oy < T.ny;
      pp[i] = T.pix_off + (int64_t)oy * T.nx + ox;
    }
    // the epilogue's 4-wide loads: every input row starts at pp[0] (in each J
    // column at a multiple of npix more) on a 16-byte boundary
    const bool vec4 = aligned16 && valid[3] && ((pp[0] | b.npix) & 3) == 0;
    double rd[W];
#pragma unroll
    for (int i = 0; i < W; ++i) rd[i] = 0.0;
    // the next tile entry, requested when this tile's last column pass is done
    int kn = -1;
    SepTile Tn;
#pragma unroll
    for (int c = 0; c < NPL; ++c) {
      const bool two = JAC && c == 0;
      __builtin_amdgcn_s_waitcnt(0);  // this wave's rows have landed in LDS
      __syncthreads();                // every wave's rows; the last row pass is done with hu
      if (two) {
        if (it0 >= 0) sconv_column<true, SP>(tin, hu, hu2, hp, it0 >> 8, it0 & 255, T.kh4, fu, fdu);
        if (it1 >= 0) sconv_column<true, SP>(tin, hu, hu2, hp, it1 >> 8, it1 & 255, T.kh4, fu, fdu);
      } else {
        if (it0 >= 0) sconv_column<false, SP>(tin, hu, hu2, hp, it0 >> 8, it0 & 255, T.kh4, fu, fdu);
        if (it1 >= 0) sconv_column<false, SP>(tin, hu, hu2, hp, it1 >> 8, it1 & 255, T.kh4, fu, fdu);
      }
      __syncthreads();  // tin is free, hu is complete
      if (c + 1 < NPL) {
        sep_stage<SP>(b, T, c + 1, tin);
      } else {
        base += (int)gridDim.x;
        kn = next_tile(base);
        if (kn >= 0) {
          Tn = sep_tile(b, s, kn);
          sep_stage<SP>(b, Tn, 0, tin);
        }
      }
      float o[4], ox_[4], oy_[4];
      if (two) {
        // value plane: K, dK/dcx (from vh'), dK/dcy (from uh')
        sconv_row<true>(hu, hu2, hp, T.kw4, fv, fdv, o, ox_, oy_);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (!valid[i]) continue;
          out[pp[i]] = o[i];
          b.jac[(int64_t)(NP - 1) * b.npix + pp[i]] = ie_scale * o[i];
          b.jac[pp[i]] = pi00 * ox_[i] + pi10 * oy_[i];
          b.jac[b.npix + pp[i]] = pi01 * ox_[i] + pi11 * oy_[i];
        }
      } else {
        sconv_row<false>(hu, hu2, hp, T.kw4, fv, fdv, o, ox_, oy_);
        if (MODE == EPI_RPP || MODE == EPI_CHI2) {
          epilogue_quad<MODE>(b, hst, pp[0], valid, vec4, o, rd);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (!valid[i]) continue;
            if (JAC) b.jac[(int64_t)(c + 1) * b.npix + pp[i]] = o[i];
            else out[pp[i]] = o[i];
          }
        }
      }
    }
    if (MODE == EPI_RPP || MODE == EPI_CHI2) tile_partial<W>(redd, rd, s.part + T.tile * kPart, lane, w);
    if (kn < 0) break;
    T = Tn;
  }
  __builtin_amdgcn_s_waitcnt(0);
}

// per tile: J^T W J (MFMA 16x16x4 f32, 4 pixels per step, 16 kTR pixels per
// wave), J^T W (Y - m0) and chi2(m0), into the tile's partial sums
__global__ __launch_bounds__(256) void normal_kernel(apx_batch b, Scratch s) {
  __shared__ double redH[4][256];
  __shared__ double redg[4][16];
  __shared__ double redc[4];
  __shared__ float sJ[4][NP][64];  // one tile row of J columns, per wave
  __shared__ float sW[4][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int r16 = lane & 15, kq = lane >> 4;
  for (int k = blockIdx.x; k < s.cnt[2]; k += gridDim.x) {
    const int2 e = s.tile_list[k];
    const apx_batch_galaxy G = b.gal[e.x];
    const int ntx = (G.nx + 63) / 64;
    const int ox0 = (e.y % ntx) * 64, oy0 = (e.y / ntx) * kTR;
    v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
    float gl[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) gl[i] = 0.0f;
    double cacc = 0.0;
    // wave wv takes tile rows 4 wv .. 4 wv + 3: each row is read coalesced
    // (one pixel a lane), staged in LDS, and fed to the MFMA 4 pixels a step
    for (int r = 0; r < kTR / 4; ++r) {
      const int px = ox0 + lane, py = oy0 + wv * (kTR / 4) + r;
      float wt = 0.0f, res = 0.0f, jv[NP];
#pragma unroll
      for (int i = 0; i < NP; ++i) jv[i] = 0.0f;
      if (px < G.nx && py < G.ny) {
        const int64_t p = G.pix_off + (int64_t)py * G.nx + px;
        const float m = b.model0[p], y = b.data[p];
        wt = b.weight[p];
        res = y - m;
#pragma unroll
        for (int i = 0; i < NP; ++i) jv[i] = b.jac[(int64_t)i * b.npix + p];
        const double dd = (double)y - (double)m;
        cacc += (double)wt * dd * dd;
      }
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        sJ[wv][i][lane] = jv[i];
        gl[i] = fmaf(jv[i] * wt, res, gl[i]);
      }
      sW[wv][lane] = wt;
      __syncthreads();
      // pixels 4 stp + kq of the row, in the order of the row
      for (int stp = 0; stp < 16; ++stp) {
        const int q = stp * 4 + kq;
        const float a = r16 < NP ? sJ[wv][r16][q] : 0.0f;
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, sW[wv][q] * a, acc, 0, 0, 0);
      }
      __syncthreads();  // the row's LDS is rewritten by the next row
    }
    // D[4 kq + i][r16] = acc[i]
#pragma unroll
    for (int i = 0; i < 4; ++i) redH[wv][(4 * kq + i) * 16 + r16] = (double)acc[i];
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const double gd = wave_sum((double)gl[i]);
      if (lane == 0) redg[wv][i] = gd;
    }
    cacc = wave_sum(cacc);
    if (lane == 0) redc[wv] = cacc;
    __syncthreads();
    double* part = s.part + (G.tile_off + e.y) * kPart;  // H row-major, g, chi2
    const int t = threadIdx.x;
    if (t < NP * NP) {
      const int idx = (t / NP) * 16 + t % NP;
      part[t] = redH[0][idx] + redH[1][idx] + redH[2][idx] + redH[3][idx];
    } else if (t < NP * NP + NP) {
      const int i = t - NP * NP;
      part[t] = redg[0][i] + redg[1][i] + redg[2][i] + redg[3][i];
    } else if (t == NP * NP + NP) {
      part[t] = redc[0] + redc[1] + redc[2] + redc[3];
    }
    __syncthreads();
  }
}

// per-fit sums of the tile partials (fixed order), into the LM state
__global__ __launch_bounds__(256) void tile_reduce_kernel(apx_batch b, Scratch s, int mode) {
  const int e = threadIdx.x & 63;
  const int W = mode == EPI_NORMAL ? NP * NP + NP + 1 : (mode == EPI_RPP ? NP : 1);
  for (int k = blockIdx.x * 4 + (int)(threadIdx.x >> 6); k < s.cnt[0]; k += gridDim.x * 4) {
    const int g = s.gal_list[k];
    const apx_batch_galaxy G = b.gal[g];
    const int ntl = ((G.nx + 63) / 64) * ((G.ny + kTR - 1) / kTR);
    if (e >= W) continue;
    // tiles t = r, r + 4, r + 8, ... into a[r], then the four in order
    const double* p = s.part + G.tile_off * kPart + e;
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    for (int t0 = 0; t0 < ntl; t0 += 4) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (t0 + r < ntl) a[r] += p[(int64_t)(t0 + r) * kPart];
    }
    const double v = a[0] + a[1] + a[2] + a[3];
    GalState* st = st_of(b, g);
    if (mode == EPI_NORMAL) {
      if (e < NP * NP) st->H[e] = v;
      else if (e < NP * NP + NP) st->g[e - NP * NP] = v;
      else st->chi2_m0 = v;
    } else if (mode == EPI_RPP) {
      st->rpp[e] = v;
    } else {
      st->chi2 = v / st->ndf;
    }
  }
}

// ---------------------------------------------------------------------------
// LM control, one thread per fit (fit/lm.py)
__device__ inline void Lup(GalState* st) { st->L = fmin(1e9, st->L * 11.0); }
__device__ inline void Ldn(GalState* st) { st->L = fmax(1e-9, st->L / 9.0); }

// h = A(L)^-1 rhs, A_ii = H_ii + L (1 + H_ii), A_ij = H_ij / (1 + L) (lm.py:359-371):
// float64 Cholesky, Gaussian elimination with partial pivoting if a pivot fails
// (every loop has a fixed trip count and every index is known at compile time,
// so A, C and y stay in registers; the pivot row is found and swapped by
// comparison with each candidate row instead of by an index)
__device__ void damped_solve(const double* H, const double* rhs, double L, double* out) {
  double A[NP][NP], y[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
#pragma unroll
    for (int j = 0; j < NP; ++j) A[i][j] = (i == j) ? H[i * NP + j] + L * (1.0 + H[i * NP + j]) : H[i * NP + j] / (1.0 + L);
    y[i] = rhs[i];
  }
  bool ok = true;
  double C[NP][NP];
#pragma unroll
  for (int j = 0; j < NP; ++j) {
    if (!ok) continue;
    double d = A[j][j];
#pragma unroll
    for (int k = 0; k < j; ++k) d -= C[j][k] * C[j][k];
    if (!(d > 0.0) || !isfinite(d)) {
      ok = false;
      continue;
    }
    C[j][j] = sqrt(d);
#pragma unroll
    for (int i = j + 1; i < NP; ++i) {
      double t = A[i][j];
#pragma unroll
      for (int k = 0; k < j; ++k) t -= C[i][k] * C[j][k];
      C[i][j] = t / C[j][j];
    }
  }
  if (ok) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      double t = y[i];
#pragma unroll
      for (int k = 0; k < i; ++k) t -= C[i][k] * y[k];
      y[i] = t / C[i][i];
    }
#pragma unroll
    for (int i = NP - 1; i >= 0; --i) {
      double t = y[i];
#pragma unroll
      for (int k = i + 1; k < NP; ++k) t -= C[k][i] * y[k];
      y[i] = t / C[i][i];
    }
  } else {
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      // the first row (from k) of largest |A[i][k]|
      int pr = k;
      double big = fabs(A[k][k]);
#pragma unroll
      for (int i = k + 1; i < NP; ++i) {
        const double v = fabs(A[i][k]);
        if (v > big) {
          big = v;
          pr = i;
        }
      }
#pragma unroll
      for (int i = k + 1; i < NP; ++i) {
        if (pr != i) continue;
#pragma unroll
        for (int j = 0; j < NP; ++j) {
          const double t = A[k][j];
          A[k][j] = A[i][j];
          A[i][j] = t;
        }
        const double t = y[k];
        y[k] = y[i];
        y[i] = t;
      }
#pragma unroll
      for (int i = k + 1; i < NP; ++i) {
        const double f = A[i][k] / A[k][k];
#pragma unroll
        for (int j = k; j < NP; ++j) A[i][j] -= f * A[k][j];
        y[i] -= f * y[k];
      }
    }
#pragma unroll
    for (int i = NP - 1; i >= 0; --i) {
      double t = y[i];
#pragma unroll
      for (int j = i + 1; j < NP; ++j) t -= A[i][j] * y[j];
      y[i] = t / A[i][i];
    }
  }
#pragma unroll
  for (int i = 0; i < NP; ++i) out[i] = y[i];
}

__device__ inline double hist_back(const GalState* st, int k) {  // loss_history[-k]
  return st->hist[(st->nhist - k) % 10];
}

__device__ inline void push_hist(GalState* st, double c) {
  st->hist[st->nhist % 10] = c;
  st->nhist += 1;
  if (isfinite(c) && (!isfinite(st->res_chi2) || c < st->res_chi2)) {  // base.py:104-117 argmin
    st->res_chi2 = c;
    for (int i = 0; i < NP; ++i) st->res_x[i] = st->x[i];
  }
}

// a fresh LM run from x0 (lm.py:155-234 state); a non-finite start is not run
__device__ void begin_run(const apx_batch& b, GalState* st, const double* x0) {
  bool finite = true;
  for (int i = 0; i < 8; ++i) {
    const double v = i < NP ? x0[i] : 0.0;
    st->x[i] = st->ev[i] = v;
    finite = finite && isfinite(v);
  }
  st->L = b.L0;
  st->nhist = 0;
  st->iter = 0;
  st->res_chi2 = INFINITY;
  for (int i = 0; i < NP; ++i) st->res_x[i] = st->x[i];
  st->phase = finite ? PH_INIT : PH_DONE;
  st->status = finite ? S_RUN : S_SKIPPED;
}

__global__ void start_kernel(apx_batch b, const double* rep0, const double* fallback) {
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= b.ngal) return;
  GalState* st = st_of(b, g);
  const apx_batch_galaxy G = b.gal[g];
  st->ndf = fmax(1.0, (double)G.nx * G.ny - NP);
  st->iter_total = 0;
  st->fb_state = 0;
  if (fallback) {
    bool finite = true;
    for (int i = 0; i < 8; ++i) {
      st->fb[i] = i < NP ? fallback[(int64_t)g * NP + i] : 0.0;
      finite = finite && isfinite(st->fb[i]);
    }
    st->fb_state = finite ? 1 : 0;
  }
  double x0[NP];
  for (int i = 0; i < NP; ++i) x0[i] = rep0[(int64_t)g * NP + i];
  begin_run(b, st, x0);
}

// the end of a run: a run that failed (no improving step, or max_iter) with
// an armed fallback starts again from the fallback, once; else the fit is done
__device__ void end_run(const apx_batch& b, GalState* st, int32_t status) {
  if ((status == S_NOSTEP || status == S_MAXITER) && st->fb_state == 1) {
    st->fb_state = 2;
    st->iter_total += st->iter;
    double x0[NP];
    for (int i = 0; i < NP; ++i) x0[i] = st->fb[i];
    begin_run(b, st, x0);
    return;
  }
  st->status = status;
  st->phase = PH_DONE;
}

// The LM kernels that precede a render stage in a tick also clear that
// stage's work counters (cnt[0..7]), in place of a launch of their own.
__device__ __forceinline__ void clear_counters(int32_t* cnt) {
  if (blockIdx.x == 0 && threadIdx.x < 8) cnt[threadIdx.x] = 0;
}

__global__ void stage_eval_kernel(apx_batch b, int32_t* cnt) {  // Jacobian stage evaluates at x
  clear_counters(cnt);
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= b.ngal) return;
  GalState* st = st_of(b, g);
  if (st->phase == PH_INIT || st->phase == PH_NEEDJ)
    for (int i = 0; i < NP; ++i) st->ev[i] = st->x[i];
}

__device__ void lm_begin(GalState* st) {
  if (st->phase != PH_INIT && st->phase != PH_NEEDJ) return;
  if (st->phase == PH_INIT) push_hist(st, st->chi2_m0 / st->ndf);  // lm.py:444-448
  st->init_chi2 = hist_back(st, 1);
  for (int i = 0; i < NP; ++i) st->best_dx[i] = 0.0;
  st->best_chi2 = st->init_chi2;
  st->best_L = st->L;
  st->scary_valid = 0;
  st->scary_chi2 = st->init_chi2;
  st->scary_L = st->L;
  st->direction = DIR_NONE;
  st->nostep = 1;
  st->sub = 0;
  st->phase = PH_SUB;
}

__device__ void lm_solve_h(GalState* st) {
  if (st->phase != PH_SUB) return;
  if (st->sub > 5 && st->L < 1e-3) st->L = 1.0;  // lm.py:270-271
  damped_solve(st->H, st->g, st->L, st->h);
  for (int i = 0; i < NP; ++i) {
    st->ev[i] = st->x[i] + 0.1 * st->h[i];  // probe point
    st->ev2[i] = st->x[i] + st->h[i];       // trial point: x + h + a * acceleration, acceleration = 0
  }
}

// step bookkeeping of the fits that have their Jacobian (lm_begin), then the
// damped solve of every fit in a sub-step
__global__ __launch_bounds__(256) void lm_begin_solve_h_kernel(apx_batch b, int32_t* cnt, int32_t* cnt2) {
  clear_counters(cnt);
  clear_counters(cnt2);
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= b.ngal) return;
  GalState* st = st_of(b, g);
  lm_begin(st);
  lm_solve_h(st);
}

__device__ void lm_solve_a(GalState* st) {
  if (st->phase != PH_SUB) return;
  if (st->L > 1e-4) {  // lm.py:283-286
    double t[NP];
    damped_solve(st->H, st->rpp, st->L, t);
    for (int i = 0; i < NP; ++i) st->a[i] = -t[i] / 2.0;
  } else {
    for (int i = 0; i < NP; ++i) st->a[i] = 0.0;
  }
  for (int i = 0; i < NP; ++i) st->ha[i] = st->h[i] + st->a[i] * 0.0;  // acceleration = 0
}

__device__ void finish_step(const apx_batch& b, GalState* st) {
  const double* dx;
  double chi2, L;
  if (st->nostep) {
    if (!st->scary_valid) {  // OptimizeStop (lm.py:348-355, 455-459)
      end_run(b, st, S_NOSTEP);
      return;
    }
    dx = st->scary_dx;
    chi2 = st->scary_chi2;
    L = st->scary_L;
  } else {
    dx = st->best_dx;
    chi2 = st->best_chi2;
    L = st->best_L;
  }
  st->L = L;  // lm.py:461-467
  for (int i = 0; i < NP; ++i) st->x[i] += dx[i];
  push_hist(st, chi2);
  Ldn(st);
  st->iter += 1;
  const int n = st->nhist;
  int32_t status = S_RUN;
  if (n >= 3 && (hist_back(st, 3) - hist_back(st, 1)) / hist_back(st, 1) < b.relative_tolerance &&
      st->L < 0.1) {
    status = S_SUCCESS;
  } else if (n > 10 &&
             (hist_back(st, 10) - hist_back(st, 1)) / hist_back(st, 1) < b.relative_tolerance) {
    status = S_IMMOBILE;
  } else if (st->iter >= b.max_iter) {
    status = S_MAXITER;
  }
  if (status == S_RUN) st->phase = PH_NEEDJ;
  else end_run(b, st, status);
}

__device__ void lm_decide(const apx_batch& b, GalState* st) {  // lm.py:293-346
  if (st->phase != PH_SUB) return;
  // The trial is rendered at x + h beside the probe; the reference's trial
  // point x + h + a * 0 (lm.py:289) differs from it only when a is not finite,
  // and there it renders at NaN, whose chi^2 is NaN.
  bool afin = true;
  for (int i = 0; i < NP; ++i) afin = afin && isfinite(st->a[i]);
  const double chi2 = afin ? st->chi2 : NAN;
  bool brk = false;
  if (!isfinite(chi2)) {
    Lup(st);
    if (st->direction == DIR_BETTER) brk = true;
    else st->direction = DIR_WORSE;
  } else {
    if (chi2 <= st->scary_chi2) {
      for (int i = 0; i < NP; ++i) st->scary_dx[i] = st->ha[i];
      st->scary_chi2 = chi2;
      st->scary_L = st->L;
      st->scary_valid = 1;
    }
    double na = 0.0, nh = 0.0;
    for (int i = 0; i < NP; ++i) {
      na += st->a[i] * st->a[i];
      nh += st->h[i] * st->h[i];
    }
    if (sqrt(na) / sqrt(nh) > 1.0) {  // curvature_limit
      Lup(st);
      if (st->direction == DIR_BETTER) brk = true;
      else st->direction = DIR_WORSE;
    } else {
      if (chi2 < st->best_chi2) {
        for (int i = 0; i < NP; ++i) st->best_dx[i] = st->ha[i];
        st->best_chi2 = chi2;
        st->best_L = st->L;
        st->nostep = 0;
        Ldn(st);
        if (st->L <= 1e-8 || st->direction == DIR_WORSE) brk = true;
        else st->direction = DIR_BETTER;
      } else if (chi2 > st->best_chi2 &&
                 (st->direction == DIR_NONE || st->direction == DIR_WORSE)) {
        Lup(st);
        if (st->L == 1e9) brk = true;
        else st->direction = DIR_WORSE;
      } else {
        brk = true;
      }
      if (!brk && (st->best_chi2 - st->init_chi2) / st->init_chi2 < -0.1) brk = true;
    }
  }
  st->sub += 1;
  if (brk || st->sub >= 10) finish_step(b, st);
}

// per fit: the sum over tiles t = r, r + 4, ... of partial e, then of the four
// in order (the order of tile_reduce_kernel)
__device__ __forceinline__ double fit_tile_sum(const double* part, int64_t tile_off, int ntl, int e) {
  double a[4] = {0.0, 0.0, 0.0, 0.0};
  for (int t0 = 0; t0 < ntl; t0 += 4) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (t0 + r < ntl) a[r] += part[(tile_off + t0 + r) * kPart + e];
  }
  return a[0] + a[1] + a[2] + a[3];
}

// The end of a sub-step, one thread per fit: rpp from the probe's tile sums
// (fits with L > 1e-4, those the probe rendered) and chi2 from the trial's,
// then a (lm_solve_a) and the decision (lm_decide)
__global__ __launch_bounds__(256) void lm_solve_a_decide_kernel(apx_batch b, Scratch sp, Scratch sq) {
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= b.ngal) return;
  GalState* st = st_of(b, g);
  if (st->phase != PH_SUB) return;
  const apx_batch_galaxy G = b.gal[g];
  const int ntl = ((G.nx + 63) / 64) * ((G.ny + kTR - 1) / kTR);
  if (st->L > 1e-4)
    for (int e = 0; e < NP; ++e) st->rpp[e] = fit_tile_sum(sp.part, G.tile_off, ntl, e);
  st->chi2 = fit_tile_sum(sq.part, G.tile_off, ntl, 0) / st->ndf;
  lm_solve_a(st);
  lm_decide(b, st);
}

__global__ void results_kernel(apx_batch b, double* rep, double* chi2, int32_t* status,
                               int32_t* iters, int32_t* fallback, int32_t* done) {
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= b.ngal) return;
  const GalState* st = st_of(b, g);
  for (int i = 0; i < NP; ++i) rep[(int64_t)g * NP + i] = st->nhist > 0 ? st->res_x[i] : st->x[i];
  if (chi2) chi2[g] = st->res_chi2;
  if (status) status[g] = st->status;
  if (iters) iters[g] = st->iter_total + st->iter;
  if (fallback) fallback[g] = st->fb_state == 2;
  if (done && st->phase == PH_DONE) atomicAdd(done, 1);
}

__global__ void zero_int_kernel(int32_t* p) { p[0] = 0; }

// Gauss-Legendre table on [-1, 1] by Newton iteration on P_n (the table
// scipy.special.roots_legendre returns, operations.py:110)
void gauss_legendre(int n, double* node, double* weight) {
  for (int i = 0; i < n; ++i) {
    double x = cos(kPi * (i + 0.75) / (n + 0.5));
    double dp = 1.0;
    for (int it = 0; it < 100; ++it) {
      double p0 = 1.0, p1 = x;
      for (int k = 2; k <= n; ++k) {
        const double p2 = ((2.0 * k - 1.0) * x * p1 - (k - 1.0) * p0) / k;
        p0 = p1;
        p1 = p2;
      }
      const double pn = n == 1 ? x : p1, pm = n == 1 ? 1.0 : p0;
      dp = n * (x * pn - pm) / (x * x - 1.0);
      const double dx = pn / dp;
      x -= dx;
      if (fabs(dx) < 1e-16) break;
    }
    node[n - 1 - i] = x;
    weight[n - 1 - i] = 2.0 / ((1.0 - x * x) * dp * dp);
  }
}

QuadTab quad_table(const apx_batch& b) {
  QuadTab t = {};
  t.n = b.quad_level;
  t.nn = t.n * t.n;
  t.g = b.gridding;
  t.gg = t.g * t.g;
  t.max_depth = b.max_depth;
  double node[APX_MAX_QUAD_LEVEL], weight[APX_MAX_QUAD_LEVEL];
  gauss_legendre(t.n, node, weight);
  for (int i = 0; i < t.n; ++i) {
    t.noded[i] = node[i];
    t.node[i] = (float)node[i];
  }
  for (int k = 0; k < t.nn; ++k) {
    t.w2d[k] = weight[k % t.n] * weight[k / t.n] * 0.25;
    t.w2[k] = (float)t.w2d[k];
  }
  for (int k = 0; k < 9; ++k) t.lw[k] = t.n == 3 ? (float)std::log2(t.w2d[k]) : 0.0f;
  t.inv_w4 = t.n == 3 ? (float)(1.0 / t.w2d[4]) : 0.0f;
  return t;
}

// The packed list of the segments `seg` with counts `cnt`.  Few fits go a workgroup
// each, since few are often large (125 windows of 100^2 to 420^2: renders 285 us so,
// 303 with 8 fits a workgroup); many fits share them (48^2 cutouts: 4,096 fits 596 us
// with a workgroup each, 421 with 8; 512 fits 134 and 125).
inline void pack_list(const apx_batch& b, const Scratch& s, int32_t* cnt, const int32_t* seg, int2* out, int32_t* len,
                      int clear, hipStream_t stream) {
  const int fits = std::max(1, std::min(kPackFits, b.ngal / 512));
  hipLaunchKernelGGL(pack_kernel, dim3(std::min((b.ngal + fits - 1) / fits, 8192)), dim3(256), 0, stream, b, s, fits,
                     cnt, seg, out, len, clear);
}

// the lane grouping of a stage's level-2/3 pass: the Jacobian stage takes
// quad_group, value-only renders quad_group_value when it is set
inline int stage_group(const apx_batch& b, bool jac) {
  return (!jac && b.quad_group_value != 0) ? b.quad_group_value : b.quad_group;
}

template <int GS, int QN, int QG>
void launch_integrate(const apx_batch& b, const Scratch& s, const QuadTab& t, bool jac,
                      hipStream_t stream, bool float_pass_only = false) {
  const dim3 ig(b.quad_blocks > 0 ? b.quad_blocks : kPersist / 2);
  if (stage_group(b, jac) == 25 && QN == 3 && QG == 5) {
    // one lane per level-2 sub-pixel, 10 pixels a workgroup
    if (jac) hipLaunchKernelGGL(integrate_wg_kernel<true>, ig, dim3(256), 0, stream, b, s, t);
    else hipLaunchKernelGGL(integrate_wg_kernel<false>, ig, dim3(256), 0, stream, b, s, t);
  } else {
    if (jac) hipLaunchKernelGGL((integrate_kernel<true, GS, false, QN, QG>), ig, dim3(256), 0, stream, b, s, t);
    else hipLaunchKernelGGL((integrate_kernel<false, GS, false, QN, QG>), ig, dim3(256), 0, stream, b, s, t);
  }
  if (float_pass_only) return;
  pack_list(b, s, s.gal_rcnt, s.redo, s.rq, s.cnt + 5, 0, stream);
  if (jac) hipLaunchKernelGGL((integrate_kernel<true, GS, true, QN, QG>), ig, dim3(256), 0, stream, b, s, t);
  else hipLaunchKernelGGL((integrate_kernel<false, GS, true, QN, QG>), ig, dim3(256), 0, stream, b, s, t);
}

// the render launches after prepare, for quadrature level QN and gridding QG
// fixed at compile time (the defaults, 3 and 5) or taken from t (0, 0)
template <int QN, int QG>
void render_launches(const apx_batch& b, const Scratch& s, const QuadTab& t, bool jac, int pc,
                     hipStream_t stream) {
  if (jac) {
    hipLaunchKernelGGL(init_kernel<true>, dim3(pc), dim3(kChunk), 0, stream, b, s, s.chunk_list, b.gal, s.ev);
    hipLaunchKernelGGL((select_kernel<true, QN>), dim3(pc), dim3(256), 0, stream, b, s, t, s.chunk_list, b.gal,
                       s.ev);
  } else {
    hipLaunchKernelGGL(init_kernel<false>, dim3(pc), dim3(kChunk), 0, stream, b, s, s.chunk_list, b.gal, s.ev);
    hipLaunchKernelGGL((select_kernel<false, QN>), dim3(pc), dim3(256), 0, stream, b, s, t, s.chunk_list, b.gal,
                       s.ev);
  }
  // float64 redo of undecided selections, then the level-2/3 quadrature of
  // the deep list, then its undecided pixels in float64
  const dim3 ig(b.quad_blocks > 0 ? b.quad_blocks : kPersist / 2);
  pack_list(b, s, s.gal_rcnt, s.redo, s.rq, s.cnt + 4, 1, stream);
  if (jac) hipLaunchKernelGGL((select_redo_kernel<true, QN>), ig, dim3(256), 0, stream, b, s, t);
  else hipLaunchKernelGGL((select_redo_kernel<false, QN>), ig, dim3(256), 0, stream, b, s, t);
  pack_list(b, s, s.gal_cnt, s.deep, s.dq, s.cnt + 3, 0, stream);
  if (t.gg <= 32 && stage_group(b, jac) != 64) launch_integrate<32, QN, QG>(b, s, t, jac, stream);
  else launch_integrate<64, QN, QG>(b, s, t, jac, stream);
}

__global__ void zero_ints_kernel(int32_t* p, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0;
}

// the float32 level-2/3 quadrature pass of the previous render again, on its
// deep list (for timing that kernel alone): the per-fit redo counts it appends
// to start from zero again, and undecided pixels are left as the float64 pass
// wrote them, so the planes do not change
void quad_again(const apx_batch& b, const Scratch& s, bool jac, hipStream_t stream) {
  const QuadTab t = quad_table(b);
  hipLaunchKernelGGL(zero_ints_kernel, dim3((b.ngal + 255) / 256), dim3(256), 0, stream, s.gal_rcnt, b.ngal);
  const bool g32 = t.gg <= 32 && stage_group(b, jac) != 64;
  if (t.n == 3 && t.g == 5) {
    if (g32) launch_integrate<32, 3, 5>(b, s, t, jac, stream, true);
    else launch_integrate<64, 3, 5>(b, s, t, jac, stream, true);
  } else {
    if (g32) launch_integrate<32, 0, 0>(b, s, t, jac, stream, true);
    else launch_integrate<64, 0, 0>(b, s, t, jac, stream, true);
  }
}

// work lists + render planes of the fits active in `stage`; `reset`: clear
// the work counters first (the LM tick's kernels clear them themselves)
void render_part(const apx_batch& b, const Scratch& s, int stage, const double* rep_override,
                 hipStream_t stream, bool reset) {
  const bool jac = stage == ST_JAC || stage == ST_ALL_JAC;
  if (reset) hipLaunchKernelGGL(reset_kernel, dim3(1), dim3(64), 0, stream, s.cnt);
  hipLaunchKernelGGL(build_kernel, dim3((b.ngal + 63) / 64), dim3(256), 0, stream, b, s, stage, rep_override);
  if (b.conv_impl == 3)
    hipLaunchKernelGGL(prepare_sep_kernel, dim3(std::min((b.ngal + 3) / 4, 16384)), dim3(256), 0, stream, b, s);
  else
    hipLaunchKernelGGL(prepare_kernel, dim3(std::min(b.ngal, 1024)), dim3(256),
                       sizeof(float) * b.max_kernel * b.max_kernel, stream, b, s, stage);
  const int pc = (int)std::min<int64_t>(b.nchunk, b.chunk_blocks > 0 ? b.chunk_blocks : 4 * kPersist);
  const QuadTab t = quad_table(b);
  if (t.n == 3 && t.g == 5) render_launches<3, 5>(b, s, t, jac, pc, stream);
  else render_launches<0, 0>(b, s, t, jac, pc, stream);
}

// convolution of the listed tiles (epilogue `mode`), then for the LM stages
// (`reduce`) the per-fit sums of the tile partials
void conv_part(const apx_batch& b, const Scratch& s, int mode, float* out, hipStream_t stream,
               bool reduce) {
  // MFMA convolution unless the caller asks for the VALU one or the PSF is too wide
  const bool sep = b.conv_impl == 3;
  const bool mf = !sep && b.conv_impl != 1 && b.max_kernel <= kMfmaMax;
  const size_t lds = sep  ? sep_lds_bytes(b.max_kernel, mode == EPI_NORMAL)
                     : mf ? mfma_lds_bytes(b.max_kernel)
                          : conv_lds_bytes(b.max_kernel);
  const int64_t items = b.ntile * (mf ? mfma_passes(mode == EPI_NORMAL) : 1);
  const int tc = (int)std::min<int64_t>(items, b.conv_blocks > 0 ? b.conv_blocks : 2 * kPersist);
#define APX_CONV(M)                                                                                \
  do {                                                                                             \
    if (sep) {                                                                                     \
      if (sp_stage_pitch(b.max_kernel) == 96)                                                      \
        hipLaunchKernelGGL((sconv_kernel<M, 96>), dim3(tc), dim3(256), lds, stream, b, s, out);    \
      else                                                                                         \
        hipLaunchKernelGGL((sconv_kernel<M, 128>), dim3(tc), dim3(256), lds, stream, b, s, out);   \
    } else if (mf) {                                                                               \
      if (lds > 65536) /* wide kernels: more than the default 64 KiB of dynamic LDS */             \
        hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_mfma_kernel<M>),                   \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                 \
      hipLaunchKernelGGL(conv_mfma_kernel<M>, dim3(tc), dim3(256), lds, stream, b, s, out);        \
    } else {                                                                                       \
      hipLaunchKernelGGL(conv_kernel<M>, dim3(tc), dim3(256), lds, stream, b, s, out);             \
    }                                                                                              \
  } while (0)
  switch (mode) {
    case EPI_OUT:
      APX_CONV(EPI_OUT);
      return;
    case EPI_NORMAL:
      APX_CONV(EPI_NORMAL);
      if (!reduce) return;
      hipLaunchKernelGGL(normal_kernel, dim3(tc), dim3(256), 0, stream, b, s);
      break;
    case EPI_RPP:
      APX_CONV(EPI_RPP);
      if (!reduce) return;
      break;
    default:
      APX_CONV(EPI_CHI2);
      if (!reduce) return;
      break;
  }
#undef APX_CONV
  hipLaunchKernelGGL(tile_reduce_kernel, dim3(std::min((b.ngal + 3) / 4, 16384)), dim3(256), 0, stream,
                     b, s, mode);
}

// one render stage over the fits active in `stage`; parts: 1 planes, 2 conv
// (`reset`: clear the work counters first; the probe and trial stages, used
// by the LM tick only, leave their per-fit sums to lm_solve_a_decide_kernel)
int run_stage(const apx_batch& b, const Scratch& s, int stage, int mode, const double* rep_override,
              float* out, hipStream_t stream, int parts = 3, bool reset = true) {
  if (parts == 4) {
    quad_again(b, s, stage == ST_JAC || stage == ST_ALL_JAC, stream);
    return check_launch("batch stage");
  }
  if (parts & 1) render_part(b, s, stage, rep_override, stream, reset);
  if (parts & 2) conv_part(b, s, mode, out, stream, stage == ST_JAC);
  return check_launch("batch stage");
}

}  // namespace

int batch_plan(apx_batch_galaxy* gal, int32_t ngal, apx_batch* b) {
  if (!gal || !b || ngal < 1) return set_error(APX_E_INVALID, "batch_plan: bad arguments");
  int64_t pix = 0, psf = 0, work = 0, tap = 0, chunk = 0, tile = 0;
  int kmax = 1;
  for (int g = 0; g < ngal; ++g) {
    apx_batch_galaxy& G = gal[g];
    if (G.nx < 1 || G.ny < 1) return set_error(APX_E_INVALID, "batch_plan: empty cutout");
    if (G.ph < 1 || G.pw < 1 || G.ph % 2 == 0 || G.pw % 2 == 0)
      return set_error(APX_E_INVALID, "batch_plan: psf must have odd shape");
    if (G.ph + 2 > kFastMax || G.pw + 2 > kFastMax)
      return set_error(APX_E_LIMIT, "batch_plan: psf larger than the batched kernel supports");
    const int bx = (G.pw + 1) / 2, by = (G.ph + 1) / 2;
    const int64_t nw = (int64_t)(G.nx + 2 * bx) * (G.ny + 2 * by);
    G.pix_off = pix;
    G.psf_off = psf;
    G.work_off = work;
    G.tap_off = tap;
    G.chunk_off = chunk;
    G.tile_off = tile;
    pix += (int64_t)G.nx * G.ny;
    psf += (int64_t)G.ph * G.pw;
    work += nw;
    tap += 3 * (int64_t)(G.pw + 2) * fast_kts(G.ph + 2);
    chunk += (nw + kChunk - 1) / kChunk;
    tile += (int64_t)((G.nx + 63) / 64) * ((G.ny + kTR - 1) / kTR);
    kmax = std::max(kmax, std::max(G.ph, G.pw) + 2);
  }
  // the VALU convolution is every batch's fallback and must fit 64 KiB; the MFMA
  // one (kmax <= kMfmaMax) takes up to 70 KiB of the 160 KiB a workgroup has
  static_assert(mfma_lds_bytes(kMfmaMax) + kConvStaticLds <= 70 * 1024, "two workgroups a CU");
  if (conv_lds_bytes(kmax) + kConvStaticLds > 65536)
    return set_error(APX_E_LIMIT, "batch_plan: psf too large for the batched Jacobian convolution");
  if (work > (int64_t)INT32_MAX || chunk > (int64_t)INT32_MAX || tile > (int64_t)INT32_MAX)
    return set_error(APX_E_LIMIT, "batch_plan: batch too large");
  b->ngal = ngal;
  b->max_kernel = kmax;
  b->npix = pix;
  b->nwork = work;
  b->nchunk = chunk;
  b->ntile = tile;
  b->ntap = tap;
  return APX_OK;
}

int64_t batch_state_bytes() { return (int64_t)sizeof(GalState); }

int64_t batch_scratch_bytes(const apx_batch* b) { return b ? scratch_bytes(*b) : 0; }

static int check_batch(const apx_batch* b) {
  if (!b || !b->gal || !b->data || !b->weight || !b->psf || !b->model0 || !b->model1 || !b->jac ||
      !b->planes || !b->taps || !b->state || !b->scratch)
    return set_error(APX_E_INVALID, "batch: null buffer");
  if (b->quad_level < 1 || b->quad_level > APX_MAX_QUAD_LEVEL || b->gridding < 1 ||
      b->gridding > APX_MAX_GRIDDING || b->max_depth < 1 || b->max_depth > APX_MAX_DEPTH)
    return set_error(APX_E_LIMIT, "batch: integration settings out of range");
  if (b->max_kernel > kFastMax) return set_error(APX_E_LIMIT, "batch: psf too large");
  if (b->conv_impl < 0 || b->conv_impl > 3 || (b->conv_impl == 2 && b->max_kernel > kMfmaMax))
    return set_error(APX_E_INVALID, "batch: conv_impl must be 0, 1, 2 or 3 (2 needs psf <= 65 px)");
  if (b->conv_impl == 3 &&
      (!b->sep_all || !b->psf_sep || b->max_kernel > kSepMax ||
       sep_lds_bytes(b->max_kernel, true) + kConvStaticLds > 65536))
    return set_error(APX_E_INVALID,
                     "batch: conv_impl 3 needs rank-one factors of every PSF (sep_all, psf_sep) and psf <= 59 px");
  for (const int grp : {b->quad_group, b->quad_group_value}) {
    if (grp != 0 && grp != 25 && grp != 32 && grp != 64)
      return set_error(APX_E_INVALID, "batch: quad_group must be 0, 25, 32 or 64");
    if (grp == 25 && (b->quad_level != 3 || b->gridding != 5))
      return set_error(APX_E_INVALID, "batch: quad_group 25 needs quad_level 3 and gridding 5");
    if (grp == 32 && b->gridding * b->gridding > 32)
      return set_error(APX_E_INVALID, "batch: quad_group 32 needs gridding <= 5");
  }
  if (b->conv_blocks < 0 || b->quad_blocks < 0 || b->chunk_blocks < 0 || b->conv_blocks > (1 << 20) ||
      b->quad_blocks > (1 << 20) || b->chunk_blocks > (1 << 20))
    return set_error(APX_E_INVALID, "batch: launch sizes out of range");
  return APX_OK;
}

int batch_render(const apx_batch* b, const double* rep, float* out, int32_t parts,
                 hipStream_t stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!rep || !out) return set_error(APX_E_INVALID, "batch_render: null pointer");
  if (parts < 1 || parts > 4) return set_error(APX_E_INVALID, "batch_render: parts must be 1, 2, 3 or 4");
  const Scratch s = carve(*b);
  return run_stage(*b, s, ST_ALL, EPI_OUT, rep, out, stream, parts);
}

int batch_jacobian(const apx_batch* b, const double* rep, float* out, int32_t parts,
                   hipStream_t stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!rep || !out) return set_error(APX_E_INVALID, "batch_jacobian: null pointer");
  if (parts < 1 || parts > 4) return set_error(APX_E_INVALID, "batch_jacobian: parts must be 1, 2, 3 or 4");
  const Scratch s = carve(*b);
  return run_stage(*b, s, ST_ALL_JAC, EPI_NORMAL, rep, out, stream, parts);
}

// The second stream of a tick (the trial render) and the events that fork
// it from the caller's stream and join it back, one set per device, made by
// batch_start (never inside a graph capture) and kept until the process ends.
struct TickStreams {
  hipStream_t side = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};
constexpr int kMaxDevices = 64;
TickStreams g_tick[kMaxDevices];

static int tick_streams(TickStreams** out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return set_error(APX_E_HIP, "batch: no current device");
  TickStreams& t = g_tick[dev];
  if (!t.side) {
    if (hipStreamCreateWithFlags(&t.side, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&t.fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&t.join, hipEventDisableTiming) != hipSuccess)
      return set_error(APX_E_HIP, "batch: cannot create the tick's second stream");
  }
  *out = &t;
  return APX_OK;
}

int batch_start(const apx_batch* b, const double* rep0, const double* fallback, hipStream_t stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!rep0) return set_error(APX_E_INVALID, "batch_start: null pointer");
  TickStreams* ts = nullptr;
  if ((rc = tick_streams(&ts))) return rc;
  hipLaunchKernelGGL(start_kernel, dim3((b->ngal + 255) / 256), dim3(256), 0, stream, *b, rep0, fallback);
  return check_launch("batch_start");
}

int batch_tick(const apx_batch* b, hipStream_t stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  const Scratch s = carve(*b);
  const int gb = (b->ngal + 255) / 256;
  // Jacobian stage for fits starting a step: model0, J, J^T W J, J^T W r, chi2(m0)
  TickStreams* ts = nullptr;
  {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices || !g_tick[dev].side)
      return set_error(APX_E_INVALID, "batch_tick: call apx_batch_start on this device first");
    ts = &g_tick[dev];
  }
  TrialBranch tb;
  scratch_layout(*b, nullptr, &tb);
  apx_batch bt = *b;  // the trial render's view: its own planes, taps and lists
  bt.planes = tb.planes;
  bt.taps = tb.taps;
  // (the LM kernels before each stage clear its work counters)
  hipLaunchKernelGGL(stage_eval_kernel, dim3(gb), dim3(256), 0, stream, *b, s.cnt);
  if ((rc = run_stage(*b, s, ST_JAC, EPI_NORMAL, nullptr, b->model0, stream, 3, false))) return rc;
  // step bookkeeping, then one sub-step: the probe point (rpp) on this stream
  // and the trial point x + h (chi2) on the second, then a and the decision
  hipLaunchKernelGGL(lm_begin_solve_h_kernel, dim3(gb), dim3(256), 0, stream, *b, s.cnt, tb.s.cnt);
  if (hipEventRecord(ts->fork, stream) != hipSuccess || hipStreamWaitEvent(ts->side, ts->fork, 0) != hipSuccess)
    return set_error(APX_E_HIP, "batch_tick: cannot fork the trial render");
  if ((rc = run_stage(*b, s, ST_PROBE, EPI_RPP, nullptr, b->model1, stream, 3, false))) return rc;
  if ((rc = run_stage(bt, tb.s, ST_TRIAL, EPI_CHI2, nullptr, b->model1, ts->side, 3, false))) return rc;
  if (hipEventRecord(ts->join, ts->side) != hipSuccess || hipStreamWaitEvent(stream, ts->join, 0) != hipSuccess)
    return set_error(APX_E_HIP, "batch_tick: cannot join the trial render");
  hipLaunchKernelGGL(lm_solve_a_decide_kernel, dim3(gb), dim3(256), 0, stream, *b, s, tb.s);
  return check_launch("batch_tick");
}

__global__ void copy_ints_kernel(const int32_t* src, int32_t* dst, int n) {
  if ((int)threadIdx.x < n) dst[threadIdx.x] = src[threadIdx.x];
}

int batch_counters(const apx_batch* b, int32_t* out, hipStream_t stream) {
  if (!b || !b->scratch || !out) return set_error(APX_E_INVALID, "batch_counters: null pointer");
  const Scratch s = carve(*b);
  hipLaunchKernelGGL(copy_ints_kernel, dim3(1), dim3(64), 0, stream, s.cnt, out, 8);
  return check_launch("batch_counters");
}

int batch_results(const apx_batch* b, double* rep, double* chi2, int32_t* status, int32_t* iters,
                  int32_t* fallback, int32_t* done, hipStream_t stream) {
  if (!b || !b->state || !rep) return set_error(APX_E_INVALID, "batch_results: null pointer");
  if (done) hipLaunchKernelGGL(zero_int_kernel, dim3(1), dim3(1), 0, stream, done);
  hipLaunchKernelGGL(results_kernel, dim3((b->ngal + 255) / 256), dim3(256), 0, stream, *b, rep,
                     chi2, status, iters, fallback, done);
  return check_launch("batch_results");
}

}  // namespace apx
