// Moment-based initial Sersic parameters for every cutout of a batch: the
// device counterpart of the reference's initialise chain, which runs on the
// host with numpy / scipy:
//   centre  iterative light-weighted centre of mass in a window
//           (utils/initialize/center.py:8-52, models/model_object.py:176-233)
//   PA      angular centre of mass of the edge-subtracted light
//           (utils/angle_operations.py:35-56, galaxy_model_object.py:78-96)
//   q       here: PSF-corrected second moments of the pixels above 3 sigma of
//           the edge near the centre (the reference scans isophote amplitudes
//           over q in [0.2, 0.9], galaxy_model_object.py:97-113)
//   n, Re,  a Sersic fit of the binned elliptical radial profile, log10 I(R),
//   Ie      by a grid search over (n, Re) with log10 Ie by least squares (the
//           reference fits the same binned profile with Nelder-Mead,
//           _shared_methods.py:71-164); when fewer than 3 bins have S/N >= 3,
//           the half-light radius and R80 / R20 concentration of the growth
//           curve, inverted through the Sersic growth curve, and Ie from the
//           total flux (utils/conversions/functions.py:168-190)
// One workgroup per cutout.  The edge level is the mean of the border pixels
// and its scatter their standard deviation (the reference takes the median
// and half the 16-84 inter-percentile range).
#include <hip/hip_runtime.h>

#include <cmath>

#include "capi_internal.h"
#include "profile.h"
#include "wave.h"

namespace apx {

namespace {

constexpr int NP = APX_BATCH_NP;
constexpr int kNB = 64;      // growth-curve bins (log-spaced) after the r < kR0 bin
constexpr float kR0 = 0.25f;
constexpr int kNT = 64;      // concentration table size

struct ConcTable {
  float n[kNT];  // Sersic index, increasing
  float c[kNT];  // R80 / R20 of that index, increasing
};

// the workgroup's sums of N values, each its four waves' in order (red: 4 N)
template <typename T, int N>
__device__ __forceinline__ void block_sums(T (&v)[N], T* red) {
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = wave_sum(v[k]);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < N; ++k) red[4 * k + (threadIdx.x >> 6)] = v[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) v[k] = red[4 * k] + red[4 * k + 1] + red[4 * k + 2] + red[4 * k + 3];
}

// Coordinates along and across an angle, and a difference of two squares, with
// every multiply-add written out: which of two products the compiler folds into
// an addition depends on the code around it, and with it the last bit of the
// estimates and the course of the fits that start from them.
__device__ __forceinline__ float along(float c, float s, float X, float Y) { return fmaf(c, X, s * Y); }
__device__ __forceinline__ float across(float c, float s, float X, float Y) { return fmaf(c, Y, -(s * X)); }
__device__ __forceinline__ float diff(float xx, float yy) {
#pragma clang fp contract(off)
  return xx - yy;
}

// column and row of this thread's pixel, and of the one 256 further on
struct PixelWalk {
  int i, j, di, dj, nx;
  __device__ __forceinline__ explicit PixelWalk(int nx_) : nx(nx_) {
    j = (int)threadIdx.x / nx;
    i = (int)threadIdx.x - j * nx;
    dj = 256 / nx;
    di = 256 - dj * nx;
  }
  __device__ __forceinline__ void next() {
    i += di;
    j += dj;
    if (i >= nx) {
      i -= nx;
      ++j;
    }
  }
};

// Bound by vector issue: 20,000 instructions a wave a 64 x 64 cutout, of 12 kB of
// data.  So no pixel is divided into column and row, three passes over the pixels
// take what five did, the bins' exponentials and logarithms and the indices' b_n
// are taken a lane each (one thread took them bin after bin, and each point of
// the (n, Re) grid its own b_n), and a centre window of up to 64 pixels is summed
// by every wave for itself, without a barrier: 8,192 cutouts 784 -> 496 us (600 with
// 98 registers, 4 waves a SIMD, in place of 64 and 8), the same bits.
__global__ __launch_bounds__(256, 8) void moment_init_kernel(apx_batch b, ConcTable T, double* rep) {
  __shared__ float redf[16];
  __shared__ double redd[8];
  __shared__ float hist[kNB + 1], cnt[kNB + 1], yk[kNB + 1], lrk[kNB + 1];
  __shared__ float rhi[kNB + 1];  // upper edges of the bins
  __shared__ unsigned long long hq[kNB + 1];  // fixed-point bin sums (two's complement)
  __shared__ float est[3], bres[4];
  __shared__ int bidx[4], nvalid;
  // the concentration table in LDS (read at run-time indices)
  __shared__ float tn[kNT], tc[kNT], tb[kNT];  // tb: b_n
  if (threadIdx.x < kNT) {
    tn[threadIdx.x] = T.n[threadIdx.x];
    tc[threadIdx.x] = T.c[threadIdx.x];
    tb[threadIdx.x] = (float)sersic_b((double)T.n[threadIdx.x]);
  }
  __syncthreads();
  for (int g = blockIdx.x; g < b.ngal; g += gridDim.x) {
    const apx_batch_galaxy G = b.gal[g];
    const float* im = b.data + G.pix_off;
    const int nx = G.nx, ny = G.ny, n = nx * ny;
    // ---- edge level and scatter
    const int ne = nx > 1 && ny > 1 ? 2 * nx + 2 * (ny - 2) : n;
    double s12[2] = {0.0, 0.0};
    for (int e = threadIdx.x; e < ne; e += 256) {
      int i, j;
      if (ne == n) {
        i = e % nx, j = e / nx;
      } else if (e < nx) {
        i = e, j = 0;
      } else if (e < 2 * nx) {
        i = e - nx, j = ny - 1;
      } else {
        const int k = e - 2 * nx;
        i = (k & 1) ? nx - 1 : 0, j = 1 + (k >> 1);
      }
      const double v = im[(int64_t)j * nx + i];
      s12[0] += v;
      s12[1] += v * v;
    }
    block_sums(s12, redd);
    const double s1 = s12[0], s2 = s12[1];
    const float edge = (float)(s1 / ne);
    const float scatter = (float)sqrt(fmax(s2 / ne - (s1 / ne) * (s1 / ne), 0.0));
    // ---- PSF second moment (per axis), for the moment corrections
    const float* K = b.psf + G.psf_off;
    double k02[2] = {0.0, 0.0};
    for (int e = threadIdx.x; e < G.ph * G.pw; e += 256) {
      const double dx = e % G.pw - (G.pw - 1) / 2, dy = e / G.pw - (G.ph - 1) / 2;
      k02[0] += K[e];
      k02[1] += K[e] * (dx * dx + dy * dy);
    }
    block_sums(k02, redd);
    const float psf2 = (float)(0.5 * k02[1] / fmax(k02[0], 1e-30));  // sigma^2 per axis
    // ---- centre: windowed centre of mass from the cutout centre (row, col)
    int win = max(min(min(nx, ny) / 10, 30), 6);
    win += win % 2;
    const float init_r = 0.5f * (ny - 1), init_c = 0.5f * (nx - 1);  // row, column
    float pr = init_r, pc = init_c;  // pixel indices of the centre, the same in every thread
    const bool one_wave = win * win <= 64;  // every wave sums the whole window
    for (int it = 0; it < 100; ++it) {
      const int r0 = (int)rintf(pr) - win / 2, c0 = (int)rintf(pc) - win / 2;
      if (r0 < 0 || c0 < 0 || r0 + win >= ny || c0 + win >= nx) {  // image edge: keep the start
        pr = init_r;
        pc = init_c;
        break;
      }
      float m[3] = {0.0f, 0.0f, 0.0f};
      for (int e = one_wave ? (int)threadIdx.x & 63 : (int)threadIdx.x; e < win * win; e += 256) {
        const int rr = e / win, cc = e % win;
        const float v = im[(int64_t)(r0 + rr) * nx + c0 + cc];
        m[0] += v;
        m[1] += v * rr;
        m[2] += v * cc;
      }
      if (one_wave) {
#pragma unroll
        for (int k = 0; k < 3; ++k) m[k] = wave_sum(m[k]);
      } else {
        block_sums(m, redf);
      }
      const float nr = r0 + m[1] / m[0], nc = c0 + m[2] / m[0];
      // converged: keep the previous centre, as center.py:45-49 does
      if (!(fabsf(nr - pr) + fabsf(nc - pc) >= 0.1f)) {
        if (!isfinite(nr) || !isfinite(nc)) {
          pr = init_r;
          pc = init_c;
        }
        break;
      }
      pr = nr;
      pc = nc;
    }
    // ---- one pass: PA (angular centre of mass of (data - edge) about the
    // centre), the rms radius of the pixels above 5 sigma (for q), and the sum of
    // |data - edge| (for the growth curve)
    float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // cos, sin, light and r^2 light above 5 sigma
    double sab[1] = {0.0};
    {
      PixelWalk at(nx);
      for (int p = threadIdx.x; p < n; p += 256, at.next()) {
        const float X = at.i - pc, Y = at.j - pr;
        const float w = im[p] - edge;
        const float xx = X * X, yy = Y * Y, r2 = fmaf(X, X, yy);
        float c = w;  // a pixel on the centre: arctan2(0, 0) = 0 (angle_operations.py:52-55)
        if (r2 > 0.0f) {
          const float inv = 1.0f / r2;
          c = w * diff(xx, yy) * inv;                      // cos 2 theta
          ps[1] = fmaf(w * (2.0f * X * Y), inv, ps[1]);  // sin 2 theta
        }
        ps[0] += c;
        if (w > 5.0f * scatter) {
          ps[2] += w;
          ps[3] = fmaf(w, r2, ps[3]);
        }
        sab[0] += fabs((double)w);
      }
    }
    block_sums(ps, redf);
    block_sums(sab, redd);
    const float cs = ps[0], sn = ps[1], c0 = ps[2], c2 = ps[3];
    const double sabs = sab[0];
    float ang = 0.5f * atan2f(sn, cs);  // angle of the light, mod pi
    // ---- q: second moments along / across that angle of the pixels above
    // 3 sigma within 4 core radii (+2 px) of the centre; the core radius is the
    // rms radius of the pixels above 5 sigma.  The radius cut keeps isolated
    // noise pixels far out, whose r^2 lever arm would otherwise round the light.
    const float ca = cosf(ang), sa = sinf(ang);
    const float thr = 3.0f * scatter;
    const float rcore = c0 > 0.0f ? sqrtf(c2 / c0) : 0.125f * (float)min(nx, ny);
    const float rlim2 = (4.0f * rcore + 2.0f) * (4.0f * rcore + 2.0f);
    float ms[3] = {0.0f, 0.0f, 0.0f};
    {
      PixelWalk at(nx);
      for (int p = threadIdx.x; p < n; p += 256, at.next()) {
        const float w = im[p] - edge;
        if (!(w > thr)) continue;
        const float X = at.i - pc, Y = at.j - pr;
        if (fmaf(X, X, Y * Y) > rlim2) continue;
        const float u = along(ca, sa, X, Y), v = across(ca, sa, X, Y);
        ms[0] = fmaf(u, w * u, ms[0]);
        ms[1] = fmaf(v, w * v, ms[1]);
        ms[2] += w;
      }
    }
    block_sums(ms, redf);
    const float mu = ms[0], mv = ms[1], mw = ms[2];
    // half the PSF second moment is removed: the thresholded moments see
    // only the part of the PSF wings above the threshold
    float q = 0.7f;
    if (mw > 0.0f) {
      const float a2 = fmaxf(mu / mw - 0.5f * psf2, 0.25f);
      const float b2 = fmaxf(mv / mw - 0.5f * psf2, 0.04f * a2);
      q = sqrtf(b2 / a2);
    }
    if (q > 1.0f) {  // the light is wider across the angle: swap the axes
      q = 1.0f / q;
      ang += 0.5f * (float)kPi;
    }
    q = fminf(fmaxf(q, 0.2f), 0.95f);
    const float cu = cosf(ang), su = sinf(ang);
    // ---- growth curve in elliptical radius
    const float rmax = 0.5f * sqrtf((float)(nx * nx + ny * ny)) + 1.0f;
    const float lstep = logf(rmax / kR0) / kNB;
    // The bin sums are accumulated in 64-bit fixed point, so that they do not
    // depend on the order of the atomic adds: the scale puts sum |data - edge|
    // below 2^60, and each pixel is rounded to 2^-60 of that sum.
    const bool fin = isfinite(sabs);  // else every bin takes the non-finite sum
    const double fx = sabs > 0.0 && fin ? ldexp(1.0, 60 - ilogb(sabs) - 1) : 1.0;
    for (int k = threadIdx.x; k <= kNB; k += 256) {
      cnt[k] = 0.0f;
      hq[k] = 0ull;
      rhi[k] = kR0 * expf(lstep * k);
    }
    __syncthreads();
    PixelWalk at(nx);
    for (int p = threadIdx.x; p < n; p += 256, at.next()) {
      const float X = at.i - pc, Y = at.j - pr;
      const float u = along(cu, su, X, Y), v = across(cu, su, X, Y) / q;
      const float R = sqrtf(fmaf(u, u, v * v));
      const int k = R < kR0 ? 0 : min(kNB, 1 + (int)(logf(R / kR0) / lstep));
      const float w = im[p] - edge;
      if (fin) atomicAdd(&hq[k], (unsigned long long)(long long)rint((double)w * fx));
      atomicAdd(&cnt[k], 1.0f);  // integer counts, exact in float
    }
    __syncthreads();
    for (int k = threadIdx.x; k <= kNB; k += 256) hist[k] = fin ? (float)((double)(long long)hq[k] / fx) : (float)sabs;
    __syncthreads();
    if (threadIdx.x < 64) {
      // radial profile bins for the fit below: mean surface brightness with
      // S/N >= 3, outside the PSF core when enough such bins remain; lane k - 1
      // looks at bin k and the kept ones close up in order
      const int k = (int)threadIdx.x + 1;
      const float rk = kR0 * expf(lstep * (k - 0.5f));
      const float Ik = hist[k] / cnt[k];
      const bool bright = !(cnt[k] < 4.0f) && Ik > 3.0f * scatter / sqrtf(cnt[k]);
      const float y = log10f(Ik), lr = logf(rk);
      int nv = 0;
      for (int pass = 0; pass < 2 && nv < 4; ++pass) {
        const float rcut = pass == 0 ? 1.5f * sqrtf(psf2) : 0.0f;
        const bool keep = bright && !(rk < rcut);
        const uint64_t bal = __ballot(keep);
        nv = (int)__popcll(bal);
        if (keep) {
          const int at_k = (int)__popcll(bal & ((1ull << threadIdx.x) - 1));
          yk[at_k] = y;
          lrk[at_k] = lr;
        }
      }
      if (threadIdx.x == 0) nvalid = nv;
    } else if (threadIdx.x == 64) {
      float tot = 0.0f;
      for (int k = 0; k <= kNB; ++k) tot += hist[k];
      // radius (upper bin edge, linear within a bin) where the curve first reaches f * tot
      auto radius = [&](float f) {
        float cum = 0.0f, prev_r = 0.0f;
        for (int k = 0; k <= kNB; ++k) {
          const float r_hi = rhi[k];
          const float nc = cum + hist[k];
          if (nc >= f * tot && hist[k] > 0.0f) return prev_r + (r_hi - prev_r) * (f * tot - cum) / hist[k];
          cum = nc;
          prev_r = r_hi;
        }
        return rmax;
      };
      float r20 = radius(0.2f), r50 = radius(0.5f), r80 = radius(0.8f);
      // remove the PSF in quadrature (half-light radius of a Gaussian: 1.1774 sigma)
      const float pw2 = 1.1774f * 1.1774f * psf2;
      const float re = sqrtf(fmaxf(r50 * r50 - pw2, 0.25f));
      const float cc = r80 / fmaxf(r20, 1e-3f);
      float ns = tn[0];
      if (cc >= tc[kNT - 1]) {
        ns = tn[kNT - 1];
      } else if (cc > tc[0]) {
        int k = 0;
        while (k < kNT - 2 && tc[k + 1] < cc) ++k;
        const float t = (cc - tc[k]) / (tc[k + 1] - tc[k]);
        ns = tn[k] + t * (tn[k + 1] - tn[k]);
      }
      ns = fminf(fmaxf(ns, 0.4f), 7.5f);
      // Ie from the total flux when the profile fit below finds nothing
      // (moment_finish_kernel)
      est[0] = re;
      est[1] = ns;
      est[2] = tot;
    }
    __syncthreads();
    // ---- Sersic profile fit of log10 I(R) over an (n, Re) grid, log10 Ie
    // by least squares (the reference fits the same binned profile with
    // Nelder-Mead, _shared_methods.py:126-164)
    constexpr int kNRe = 48;
    const int nv = nvalid;
    float best = INFINITY;
    int bi = -1;
    if (nv >= 3) {
      const float lre0 = logf(0.5f), lre1 = logf(4.0f * rmax);
      for (int c = threadIdx.x; c < kNT * kNRe; c += 256) {
        const float nn = tn[c / kNRe];
        if (nn < 0.4f || nn > 7.5f) continue;
        const float lre = lre0 + (lre1 - lre0) * (float)(c % kNRe) / (kNRe - 1);
        const float bn = tb[c / kNRe], inv = 1.0f / nn;
        float s1 = 0.0f, s2 = 0.0f;
        for (int k = 0; k < nv; ++k) {
          const float m = -bn * (__expf((lrk[k] - lre) * inv) - 1.0f) * 0.43429448f;
          const float d = yk[k] - m;
          s1 += d;
          s2 += d * d;
        }
        const float res = s2 - s1 * s1 / (float)nv;
        if (res < best) {
          best = res;
          bi = c;
        }
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ob = __shfl_xor(best, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (ob < best || (ob == best && oi >= 0 && (bi < 0 || oi < bi))) {
        best = ob;
        bi = oi;
      }
    }
    if ((threadIdx.x & 63) == 0) {
      bres[threadIdx.x >> 6] = best;
      bidx[threadIdx.x >> 6] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      float re = est[0], ns = est[1];
      double ie = est[2];  // the total flux until a profile fit replaces it
      int c = -1;
      float bb = INFINITY;
      for (int w = 0; w < 4; ++w)
        if (bidx[w] >= 0 && (bres[w] < bb || (bres[w] == bb && bidx[w] < c))) {
          bb = bres[w];
          c = bidx[w];
        }
      if (c >= 0) {
        ns = tn[c / kNRe];
        const float lre0 = logf(0.5f), lre1 = logf(4.0f * rmax);
        re = expf(lre0 + (lre1 - lre0) * (float)(c % kNRe) / (kNRe - 1));
        const float bn = tb[c / kNRe], inv = 1.0f / ns;
        float s1 = 0.0f;
        for (int k = 0; k < nv; ++k) s1 += yk[k] + bn * (__expf((lrk[k] - logf(re)) * inv) - 1.0f) * 0.43429448f;
        // log10 of the surface brightness at Re, per unit plane area
        ie = (double)(s1 / (float)nv) - log10(fabs(b.P[0] * b.P[3] - b.P[1] * b.P[2]));
      }
      // the float estimates, for moment_finish_kernel; a negative n marks
      // an Ie still to be taken from the total flux
      double* r = rep + (int64_t)g * NP;
      r[0] = pc;
      r[1] = pr;
      r[2] = q;
      r[3] = ang;
      r[4] = c >= 0 ? ns : -ns;
      r[5] = re;
      r[6] = ie;
    }
    __syncthreads();
  }
}

// per cutout (one thread each): the float64 end of the moment estimate, kept
// out of moment_init_kernel, whose registers it would otherwise set
__global__ __launch_bounds__(256) void moment_finish_kernel(apx_batch b, double* rep) {
  const int g = blockIdx.x * 256 + threadIdx.x;
  if (g >= b.ngal) return;
  const apx_batch_galaxy G = b.gal[g];
  double* r = rep + (int64_t)g * NP;
  const float pc = (float)r[0], pr = (float)r[1], q = (float)r[2], ang = (float)r[3];
  const bool from_flux = r[4] < 0.0;
  const float ns = (float)fabs(r[4]), re = (float)r[5];
  double ie = r[6];
  if (from_flux) {
    // Ie from the total flux (functions.py:168-190)
    const double bn = sersic_b((double)ns);
    const double flux_per_ie = 2.0 * kPi * (double)re * re * q * ns * exp(bn) * pow(bn, -2.0 * ns) *
                               exp(lgamma(2.0 * ns));
    ie = (double)(float)log10(fmax((double)(float)ie, 1e-30) / flux_per_ie);
  }
  // plane coordinates (pixel i at origin + i + 0.5 for the batch's pixel matrix)
  const double px = (double)pc + 0.5, py = (double)pr + 0.5;
  const double cx = G.origin[0] + b.P[0] * px + b.P[1] * py;
  const double cy = G.origin[1] + b.P[2] * px + b.P[3] * py;
  // PA parameter: light angle + north, mod pi (galaxy_model_object.py:94)
  double pa = fmod((double)ang + 0.5 * kPi, kPi);
  if (pa < 0.0) pa += kPi;
  // value -> representation (utils/conversions/optimization.py:6-14)
  r[0] = cx;
  r[1] = cy;
  r[2] = tan((double)q * kPi - 0.5 * kPi);
  r[3] = pa;
  r[4] = tan(((double)ns - 0.36) * kPi / (8.0 - 0.36) - 0.5 * kPi);
  r[5] = (double)re - 1.0 / (double)re;
  r[6] = ie;
}

// ---- host: Sersic growth curve R80 / R20 as a function of n ------------
// regularised lower incomplete gamma P(a, x): series for x < a + 1, else the
// continued fraction of Q (Legendre's), both to 1e-12
double gamma_p(double a, double x) {
  if (x <= 0.0) return 0.0;
  const double lg = lgamma(a);
  if (x < a + 1.0) {
    double term = 1.0 / a, sum = term;
    for (int k = 1; k < 1000; ++k) {
      term *= x / (a + k);
      sum += term;
      if (fabs(term) < fabs(sum) * 1e-13) break;
    }
    return sum * exp(-x + a * log(x) - lg);
  }
  double bb = x + 1.0 - a, c = 1e300, d = 1.0 / bb, h = d;
  for (int k = 1; k < 1000; ++k) {
    const double an = -k * (k - a);
    bb += 2.0;
    d = an * d + bb;
    if (fabs(d) < 1e-300) d = 1e-300;
    c = bb + an / c;
    if (fabs(c) < 1e-300) c = 1e-300;
    d = 1.0 / d;
    const double del = d * c;
    h *= del;
    if (fabs(del - 1.0) < 1e-13) break;
  }
  return 1.0 - exp(-x + a * log(x) - lg) * h;
}

// x with P(a, x) = f, by bisection on a bracketing interval
double gamma_p_inv(double a, double f) {
  double lo = 0.0, hi = a + 10.0 * sqrt(a) + 10.0;
  while (gamma_p(a, hi) < f) hi *= 2.0;
  for (int it = 0; it < 200; ++it) {
    const double mid = 0.5 * (lo + hi);
    if (gamma_p(a, mid) < f) lo = mid;
    else hi = mid;
  }
  return 0.5 * (lo + hi);
}

const ConcTable& conc_table() {
  static ConcTable T = [] {
    ConcTable t;
    for (int k = 0; k < kNT; ++k) {
      const double n = 0.36 * pow(8.0 / 0.36, (double)k / (kNT - 1));
      // L(<R) / L = P(2n, b_n (R / Re)^(1/n))  =>  R80 / R20 = (x80 / x20)^n
      const double x20 = gamma_p_inv(2.0 * n, 0.2), x80 = gamma_p_inv(2.0 * n, 0.8);
      t.n[k] = (float)n;
      t.c[k] = (float)pow(x80 / x20, n);
    }
    return t;
  }();
  return T;
}

}  // namespace

double sersic_light_fraction(double n, double r_over_re) {
  return gamma_p(2.0 * n, sersic_b(n) * pow(r_over_re, 1.0 / n));
}

int batch_moment_init(const apx_batch* b, double* rep, hipStream_t stream) {
  if (!b || !b->gal || !b->data || !b->psf || !rep || b->ngal < 1)
    return set_error(APX_E_INVALID, "batch_moment_init: bad arguments");
  hipLaunchKernelGGL(moment_init_kernel, dim3(std::min(b->ngal, 16384)), dim3(256), 0, stream, *b,
                     conc_table(), rep);
  hipLaunchKernelGGL(moment_finish_kernel, dim3((b->ngal + 255) / 256), dim3(256), 0, stream, *b, rep);
  return check_launch("batch_moment_init");
}

}  // namespace apx
