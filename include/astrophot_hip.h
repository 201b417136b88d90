/*
 * astrophot_hip.h -- C ABI of the MI355X (gfx950) image-model hot path.
 *
 * Plain pointers and sizes only.  Every pointer argument is device memory
 * owned by the caller unless stated otherwise (structs are passed by host
 * pointer and copied at launch); every call is asynchronous on the HIP stream
 * passed as ``stream`` (a hipStream_t; NULL = default stream) and returns 0 on
 * success or a negative APX_E* code, with a message in apx_last_error().
 * No call allocates device memory: scratch space is passed in by the caller
 * and sized with the matching *_workspace_bytes() query.
 *
 * Reference interfaces replaced (paths relative to the AstroPhot repository):
 *   apx_render_component  -> models/_model_methods.py:82-184 (_sample_init,
 *                            _sample_integrate) with models/_shared_methods.py:
 *                            274-418 and utils/operations.py:94-247
 *   apx_psf_shift         -> models/_model_methods.py:187-207, 243
 *                            (_shift_psf + normalise), utils/interpolate.py:282-329
 *   apx_convolve          -> models/_model_methods.py:233-257 (_sample_convolve),
 *                            utils/operations.py:9-36, models/model_object.py:
 *                            342-373 (crop, reduce(1), image +=)
 *   apx_chi2              -> fit/lm.py:373-378 (_chi2), utils/optimization.py:6-30
 *   apx_normal_equations  -> fit/lm.py:387-399 (_hess, _grad)
 *   apx_rpp               -> fit/lm.py:401-406 (_rpp)
 *   apx_lm_solve          -> fit/lm.py:359-371 (_h, damped solve)
 */
#ifndef ASTROPHOT_HIP_H
#define ASTROPHOT_HIP_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define APX_OK 0
#define APX_E_INVALID (-1) /* bad argument (shape, mode, pointer) */
#define APX_E_HIP (-2)     /* a HIP runtime call failed */
#define APX_E_LIMIT (-3)   /* a size exceeds a documented limit */

/* profile kinds: models/sersic_model.py, exponential_model.py,
 * gaussian_model.py, moffat_model.py, flatsky_model.py */
#define APX_SERSIC 0
#define APX_EXPONENTIAL 1
#define APX_GAUSSIAN 2
#define APX_MOFFAT 3
#define APX_FLAT_SKY 4

/* natural parameter slots of a component */
#define APX_P_CX 0
#define APX_P_CY 1
#define APX_P_Q 2
#define APX_P_PA 3
#define APX_P_A 4 /* sersic n | exponential Re | gaussian sigma | moffat n | sky F */
#define APX_P_B 5 /* sersic Re | exponential Ie | gaussian flux | moffat Rd */
#define APX_P_C 6 /* sersic Ie | moffat I0 */
#define APX_NSLOT 7

#define APX_SAMPLE_MIDPOINT 0
#define APX_SAMPLE_QUAD 1
#define APX_SAMPLE_TRAPEZOID 2

#define APX_INTEGRATE_NONE 0      /* integrate_mode "none" */
#define APX_INTEGRATE_THRESHOLD 1 /* "threshold" (_model_methods.py:155-184) */
#define APX_INTEGRATE_RADIUS 2    /* "radius": every pixel whose centre lies within
                                     integrate_radius (plane units, inclusive to 1e-9
                                     relative) of the model centre
                                     takes the quad_level x quad_level Gauss-Legendre
                                     rule once (grid_integrate at depth 1, no
                                     refinement); no reference counterpart */

#define APX_MAX_QUAD_LEVEL 7 /* quad_level**2 <= 64 lanes */
#define APX_MAX_GRIDDING 8   /* gridding**2 <= 64 lanes */
#define APX_MAX_DEPTH 3
#define APX_MAX_KERNEL 131   /* shifted-PSF side (PSF side + 2) */
#define APX_MAX_CHAN 8       /* render planes: value + up to 7 slots */

/* One component rendered on its working grid.  Geometry is float64 from the
 * host.  Working-grid pixel (i, j) (i = column, j = row) sits at plane offset
 * (X, Y) = P . (i - ci, j - cj) + frac from the model centre. */
typedef struct apx_component {
  int32_t profile;        /* APX_SERSIC .. APX_FLAT_SKY */
  int32_t sampling;       /* APX_SAMPLE_MIDPOINT | APX_SAMPLE_QUAD | APX_SAMPLE_TRAPEZOID */
  int32_t sample_quad;    /* N of sampling_mode "quad:N"; "simpsons" (_model_methods.py:
                             97-109) is N = 3 with sq_node -1, 0, 1 and sq_weight
                             1/3, 4/3, 1/3: the 3 x 3 Simpson rule on the pixel.
                             APX_SAMPLE_TRAPEZOID ("trapezoid", _model_methods.py:
                             121-139) takes N = 2 with sq_node -1, 1 and sq_weight
                             1, 1 (the mean of the four pixel corners) and selects by
                             the Laplacian of those means, as midpoint sampling does */
  int32_t integrate;      /* APX_INTEGRATE_NONE | _THRESHOLD | _RADIUS */
  int32_t quad_level;     /* integrate_quad_level */
  int32_t gridding;       /* integrate_gridding */
  int32_t max_depth;      /* integrate_max_depth */
  int32_t mean_reference; /* 1: reference = mean of the initial samples
                             (_model_methods.py:151-152); 0: use `reference` */
  int32_t nx, ny;         /* working grid */
  int32_t ci, cj;         /* integer centre pixel on the working grid */
  int32_t nchan;          /* render planes: 1 (value) + Jacobian channels */
  int32_t chan_slot[APX_MAX_CHAN]; /* slot of render plane c (c >= 1) */
  double P[4];            /* pixelscale matrix, row-major */
  double frac[2];
  double pixel_area;
  double softening;
  double tolerance;       /* sampling_tolerance */
  double reference;       /* integrate reference when mean_reference == 0 */
  double q, pa;           /* axis ratio, position angle (radians) */
  double prm[3];          /* slot A, B, C values */
  double dvdr[APX_NSLOT]; /* d value / d representation per slot */
  /* Gauss-Legendre abscissae/weights on [-1, 1] (utils/operations.py:105-120)
   * for integrate_quad_level (gl_*) and for sampling "quad:N" (sq_*) */
  double gl_node[8], gl_weight[8];
  double sq_node[8], sq_weight[8];
  double integrate_radius; /* APX_INTEGRATE_RADIUS: selection radius (plane units) */
} apx_component;

/* Workspace (bytes) needed by apx_render_component for npix working pixels. */
int64_t apx_render_workspace_bytes(int64_t npix);

/* Render one component on its working grid into `planes` (nchan x ny x nx
 * float32).  Plane 0 is the value; plane c >= 1 is d value / d rep of slot
 * chan_slot[c].  Midpoint or quad:N sampling, then threshold-selected adaptive
 * Gauss-Legendre integration (or, APX_INTEGRATE_RADIUS, one Gauss-Legendre
 * level on the pixels within integrate_radius of the centre); selection
 * decisions and level-1 quadrature are float64, deeper levels float32 samples
 * summed in float64. */
int apx_render_component(const apx_component* comp, float* planes, void* workspace,
                         int64_t workspace_bytes, void* stream);

/* Adjoint of apx_render_component: grad[c-1] = sum over working pixels q of
 * weights[q] * d value[q] / d rep(chan_slot[c]) for c = 1 .. nchan-1, float64,
 * device.  `weights` (ny x nx) is the upstream gradient already carried back
 * through the convolution.  The value render is recomputed into
 * `value_plane` (ny x nx); supersampled pixels are re-integrated as the
 * forward render integrates them (level 1 float64, deeper levels float32
 * samples summed in float64); nothing of the forward pass is stored.
 * Replaces the reverse-mode path of models/_model_methods.py:82-184. */
int apx_render_vjp(const apx_component* comp, const float* weights, float* value_plane,
                   double* grad, void* workspace, int64_t workspace_bytes, void* stream);

/* Number of pixels the last apx_render_component on `workspace` integrated
 * (copies one int to the host; synchronises the stream). */
int apx_render_selected_count(const void* workspace, void* stream, int32_t* count);

/* Bilinear sub-pixel shift of a (ph x pw) float32 PSF with a 1-px zero pad,
 * normalised to unit sum, flipped for direct correlation, and its derivatives
 * with respect to the model centre in representation units:
 *   dK/dc_x = (dK/ds_x pinv[0] + dK/ds_y pinv[2]) dvdr_x ,
 *   dK/dc_y = (dK/ds_x pinv[1] + dK/ds_y pinv[3]) dvdr_y .
 * Output `kernels`: 3 x (ph+2) x (pw+2) float32 [K, dK/dcx, dK/dcy]. */
int apx_psf_shift(const float* psf, int32_t ph, int32_t pw, double shift_x, double shift_y,
                  const double* pinv /* host, 4 doubles */, double dvdr_x, double dvdr_y, float* kernels,
                  void* stream);

/* PSF_Model.sample's normalisation to unit sum (models/psf_model_object.py:
 * 255-257) on render planes (nchan x npix float32, as apx_render_component
 * writes them): plane 0 becomes P / S with S = sum P, and plane c >= 1
 * (dP / d rep) becomes dP / S - P (sum dP) / S^2, the derivative of the
 * normalised PSF.  float64 sums in a fixed order on one workgroup. */
int apx_normalize_planes(float* planes, int32_t nchan, int64_t npix, void* stream);

/* Kernels of a PSF that is rendered from parameters (an auxiliary PSF model,
 * models/model_object.py:133-147 and 305-310, through _model_methods.py:
 * 187-207 and 243).  T is the PSF after the sub-pixel shift: the 1-px
 * zero-padded bilinear shift of apx_psf_shift (shifted = 1, kernel side
 * (ph+2) x (pw+2)) or the PSF itself (shifted = 0, psf_subpixel_shift "none",
 * side ph x pw).  K = T / sum T and, for each derivative plane dP of dpsf
 * (nd x ph x pw), dK = dT / sum T - T (sum dT) / (sum T)^2 with dT the same
 * shift of dP.  `out` receives nd + 2 planes [K, dK_0 .. dK_(nd-1), 0], each
 * flipped for direct correlation like apx_psf_shift's, so that apx_convolve
 * with kernels = out + 2k planes and dk_col = {c(2k), c(2k+1)} writes the
 * columns of derivative planes 2k and 2k+1 (the trailing zero plane pads an
 * odd nd).  nd <= APX_NSLOT. */
int apx_psf_kernels_dparam(const float* psf, const float* dpsf, int32_t nd, int32_t ph, int32_t pw,
                           int32_t shifted, double shift_x, double shift_y, float* out,
                           void* stream);

/* Direct convolution of render planes, cropped to an output box. */
typedef struct apx_conv_job {
  int32_t nx, ny, nchan;   /* render planes (working grid) */
  int32_t kh, kw;          /* kernel side (odd); 1 x 1 = plain crop/copy */
  int32_t x0, y0;          /* working-grid pixel under output pixel (0, 0) */
  int32_t ow, oh;          /* output box */
  float* img;              /* value destination (+=), may be NULL */
  int64_t img_row;         /* img row stride (floats), >= img_w */
  int32_t img_w, img_h;    /* img extent (pixels); the box must fit inside */
  int32_t img_x0, img_y0;  /* img pixel of output (0, 0) */
  float* jac;              /* Jacobian destination (+=), pixel-major, may be NULL */
  int64_t jac_row;         /* jac row stride (floats), >= jac_w * jac_np */
  int32_t jac_w, jac_h;    /* jac extent (pixels) */
  int32_t jac_np;          /* jac pixel stride (floats) */
  int32_t jac_x0, jac_y0;  /* jac pixel of output (0, 0) */
  int32_t chan_col[APX_MAX_CHAN]; /* jac column of render plane c (c >= 1) */
  int32_t dk_col[2];       /* jac columns of conv(plane 0, dK/dc), -1 = none */
  int32_t zero_outside;    /* 1: taps reaching outside the planes read zero
                              (adjoint pass); 0: the box must stay inside */
} apx_conv_job;

/* Workspace (bytes) apx_convolve needs for a kh x kw kernel. */
int64_t apx_convolve_workspace_bytes(int32_t kh, int32_t kw);

/* out(ox, oy) = sum_ab kernel[a][b] * plane[y0+oy-(kh-1)/2+a][x0+ox-(kw-1)/2+b]
 * (kernels pre-flipped by apx_psf_shift).  `kernels` is 3 x kh x kw when
 * dk_col is used, else 1 x kh x kw.  The workspace holds the taps re-arranged
 * for the scalar cache. */
int apx_convolve(const apx_conv_job* job, const float* planes, const float* kernels,
                 void* workspace, int64_t workspace_bytes, void* stream);

#define APX_MAX_BLOCK_COLS 16

/* A model sampled on a PSF-upscaled grid (model_object.py:313-314, 348-349):
 * Image.reduce, the sum of scale x scale blocks (image_object.py:348-376),
 * then the window-aware += (image_object.py:450-457).  src is pixel-major,
 * nc floats per fine pixel, src_w fine pixels per row.  For c < nc, y < h,
 * x < w:
 *   dst[(dst_y0 + y) * dst_row + (dst_x0 + x) * dst_pix + col[c]] +=
 *     sum over a, b < scale of src[((scale * y + b) * src_w + scale * x + a) * nc + c] */
typedef struct apx_block_sum {
  int32_t scale, nc;       /* block side; channels per pixel (<= APX_MAX_BLOCK_COLS) */
  int32_t w, h;            /* coarse box */
  int32_t src_w, src_h;    /* src extent in fine pixels (>= scale * w, scale * h) */
  float* dst;
  int64_t dst_row;         /* dst row stride (floats), >= dst_w * dst_pix */
  int32_t dst_pix;         /* dst pixel stride (floats) */
  int32_t dst_w, dst_h;    /* dst extent (pixels); the box must fit inside */
  int32_t dst_x0, dst_y0;  /* dst pixel of box pixel (0, 0) */
  int32_t col[APX_MAX_BLOCK_COLS]; /* dst offset within a pixel of src channel c */
} apx_block_sum;

int apx_block_sum_add(const apx_block_sum* job, const float* src, void* stream);

/* Workspace (bytes) for apx_chi2 / apx_normal_equations / apx_rpp. */
int64_t apx_reduce_workspace_bytes(int64_t npix, int32_t np);

/* out[0] = sum over unmasked pixels of weight*(data-model)^2 (float64, device).
 * mask (uint8, nonzero = ignore) and weight may be NULL. */
int apx_chi2(const float* model, const float* data, const float* weight, const uint8_t* mask,
             int64_t npix, double* out, void* workspace, int64_t workspace_bytes, void* stream);

/* hess = J^T W J (np x np) and grad = -J^T W (model - data) (np), float64,
 * with J pixel-major (npix x np float32).  FP32 matrix-core products,
 * float64 sum over workgroups.  np <= 16. */
int apx_normal_equations(const float* J, const float* model, const float* data, const float* weight,
                         const uint8_t* mask, int64_t npix, int32_t np, double* hess, double* grad,
                         void* workspace, int64_t workspace_bytes, void* stream);

/* apx_normal_equations without a workspace argument: no counterpart in the
 * reference.  For callers that cannot allocate device memory (code under HIP
 * graph capture, tight serving loops, harnesses that forbid hipMalloc).  The
 * partial sums live in the library's static device scratch of 1,114,112 bytes
 * (512 workgroups x (16 x 16 + 16) float64), held on each GPU the library runs
 * on until the process ends; every npix fits it, np > 16 returns APX_E_LIMIT.
 * Results equal apx_normal_equations' bit for bit (same kernels, same order).
 * No call allocates or frees memory.  Calls that overlap on one GPU (two
 * streams, two threads) share that scratch and race: serialise them. */
int apx_normal_equations_noalloc(const float* J, const float* model, const float* data,
                                 const float* weight, const uint8_t* mask, int64_t npix, int32_t np,
                                 double* hess, double* grad, void* stream);

/* rpp = J^T ((2/d) (W (m1 - m0) / d - W (J h)))  (fit/lm.py:281, 401-406);
 * h and rpp float64 (np). */
int apx_rpp(const float* J, const float* m0, const float* m1, const float* weight,
            const uint8_t* mask, int64_t npix, int32_t np, const double* h, double d, double* rpp,
            void* workspace, int64_t workspace_bytes, void* stream);

/* h = A(L)^-1 g with A_ii = H_ii + L (1 + H_ii), A_ij = H_ij / (1 + L): float64
 * Cholesky on one workgroup (np <= 64).  status[0] = 0 ok, k+1 if the pivot of
 * row k is not positive (h is then NaN). */
int apx_lm_solve(const double* hess, const double* grad, int32_t np, double L, double* h,
                 int32_t* status, void* stream);

/* ---------------------------------------------------------------------------
 * Batched independent fits (north-star configuration C2): every cutout holds
 * one Sersic galaxy convolved with its own PSF (psf_mode "full", bilinear
 * sub-pixel shift, midpoint sampling, threshold integration) and is fitted by
 * the reference's Levenberg-Marquardt (fit/lm.py:248-493, defaults L0=1,
 * Lup=11, Ldn=9, 10 sub-steps, curvature limit 1, acceleration 0).  All
 * fits advance together on the device: one "tick" is one LM sub-step of every
 * fit that is inside a step, plus the Jacobian pass of every fit that starts
 * one.  A tick is a fixed sequence of launches over device-built work lists,
 * so it can be captured in a HIP graph and replayed.
 * Parameter vector per fit (representation space, float64):
 *   [center_x, center_y, q, PA, n, Re, Ie] with the maps of
 *   galaxy_model_object.py:44-53 and sersic_model.py:61-66.
 * ------------------------------------------------------------------------- */
#define APX_BATCH_NP 7

typedef struct apx_batch_galaxy {
  int32_t nx, ny;     /* cutout size */
  int32_t ph, pw;     /* PSF size (odd) */
  int64_t pix_off;    /* first cutout pixel in data / weight / model / jac */
  int64_t psf_off;    /* first PSF value in psf */
  int64_t work_off;   /* first working pixel (cutout + PSF border) in planes */
  int64_t tap_off;    /* first float of this fit's re-arranged taps */
  int64_t chunk_off;  /* first 256-pixel working chunk (global index) */
  int64_t tile_off;   /* first 64 x 8 output tile (global index) */
  double origin[2];   /* plane coordinates of the cutout corner (pixel -0.5,-0.5) */
  int64_t ref_npix;   /* pixel count the Sersic flux is divided by in the integration
                         threshold (sersic_model.py:87-89); 0 = this cutout's working
                         grid.  A source sampled as part of a larger window (a group,
                         group_model_object.py:183-231) sets that window's working grid */
  int64_t sep_off;    /* first float of this PSF's rank-one factors in psf_sep (ph column
                         values u, then pw row values v, PSF = u v^T to float32
                         rounding); read only by the separable convolution */
} apx_batch_galaxy;

typedef struct apx_batch {
  int32_t ngal;
  int32_t max_kernel;          /* largest PSF side + 2 in the batch */
  int64_t npix, nwork, nchunk, ntile, ntap;  /* totals (set by apx_batch_plan) */
  double P[4];                 /* pixelscale shared by the batch (row-major) */
  double softening, tolerance; /* softening, sampling_tolerance */
  int32_t quad_level, gridding, max_depth;   /* integrate_* */
  int32_t max_iter;            /* LM max_iter */
  double relative_tolerance;   /* LM relative_tolerance */
  double L0;                   /* initial damping */
  /* device buffers, allocated by the caller with the sizes apx_batch_plan sets */
  const apx_batch_galaxy* gal; /* ngal */
  const float* data;           /* npix */
  const float* weight;         /* npix, 1/variance */
  const float* psf;            /* sum of ph * pw */
  const float* psf_sep;        /* rank-one PSF factors (sep_off); NULL unless sep_all */
  float* model0;               /* npix: model at the current state */
  float* model1;               /* npix: spare model buffer (the LM ticks reduce their
                                  probe and trial renders in place, unstored) */
  float* jac;                  /* APX_BATCH_NP x npix, parameter-major (column c of
                                  J at jac + c * npix) */
  float* planes;               /* 6 x nwork */
  float* taps;                 /* ntap */
  void* state;                 /* ngal x apx_batch_state_bytes() */
  void* scratch;               /* apx_batch_scratch_bytes(batch) */
  /* launch shape (0 = built-in default); set by the caller's autotuner */
  int32_t conv_impl;           /* 1 = VALU convolution, 2 = MFMA (kernels <= 67 px),
                                  3 = separable (sep_all, kernels <= 61 px) */
  int32_t conv_blocks;         /* workgroups of the convolution launches */
  int32_t quad_blocks;         /* workgroups of the level-2/3 quadrature launches */
  int32_t quad_group;          /* lanes per refined pixel: 32 (gridding <= 5) or 64; 25: one
                                  lane per level-2 sub-pixel, 10 pixels a workgroup
                                  (quad_level 3, gridding 5) */
  int32_t chunk_blocks;        /* workgroups of the per-chunk render launches */
  int32_t sep_all;             /* 1: every PSF of the batch has factors in psf_sep */
  int32_t quad_group_value;    /* quad_group of the value-only renders (LM probe and trial
                                  points); 0 = as quad_group */
} apx_batch;

/* Fill the offsets of gal[] (host array) and the totals of *batch. */
int apx_batch_plan(apx_batch_galaxy* gal, int32_t ngal, apx_batch* batch);
int64_t apx_batch_state_bytes(void);
int64_t apx_batch_scratch_bytes(const apx_batch* batch);

/* Render every cutout at rep (device, ngal x 7 float64) into out (npix).
 * parts: 1 = render the working planes only, 2 = convolve planes rendered by
 * a previous parts=1 call, 3 = both, 4 = the float32 level-2/3 quadrature
 * pass of the previous parts=1 call again on its lists (planes unchanged;
 * for timing that launch alone). */
int apx_batch_render(const apx_batch* batch, const double* rep, float* out, int32_t parts,
                     void* stream);

/* Render every cutout at rep into out (npix) and its Jacobian with respect
 * to the 7 representation-space parameters into batch->jac (7 x npix,
 * parameter-major): the batched counterpart of Component_Model.jacobian(
 * as_representation=True) (models/_model_methods.py:260-347), the columns of
 * the J the LM's Jacobian stage forms (fit/lm.py:256-257).  parts as in
 * apx_batch_render.  Leaves the LM state of the fits untouched. */
int apx_batch_jacobian(const apx_batch* batch, const double* rep, float* out, int32_t parts,
                       void* stream);

/* Moment-based initial parameters of every cutout from its data alone, into
 * rep (device, ngal x 7, representation space): the batched counterpart of
 * the initialise chain Component_Model.initialize (models/model_object.py:
 * 176-233, utils/initialize/center.py:8-52), Galaxy_Model.initialize
 * (models/galaxy_model_object.py:56-113) and parametric_initialize
 * (models/_shared_methods.py:71-164).  Centre and PA follow the reference's
 * estimators; q comes from PSF-corrected second moments instead of the
 * isophote scan, and n, Re, Ie from a grid-search Sersic fit of the binned
 * radial profile instead of Nelder-Mead. */
int apx_batch_moment_init(const apx_batch* batch, double* rep, void* stream);

/* Fraction of a Sersic profile's light inside elliptical radius r (in units
 * of Re): P(2n, b_n r^(1/n)), the growth curve the initialiser inverts
 * (host function; utils/conversions/functions.py:7-22 for b_n). */
double apx_sersic_light_fraction(double n, double r_over_re);

/* Start the fits from rep0 (device, ngal x 7).  A fit whose row holds a
 * non-finite value is not run: it ends at once with status 5 (skipped).
 * On its first call on a device it also makes the second stream and the two
 * events a tick forks its trial render onto (kept until the process ends),
 * so it must run, outside any graph capture, before the first apx_batch_tick
 * on that device. */
int apx_batch_start(const apx_batch* batch, const double* rep0, void* stream);

/* Start the fits from rep0 with a fallback start per fit (device, ngal x 7):
 * a run that fails (status 3 or 4) restarts once from its fallback row within
 * the same ticks, the way a caller would re-run LM from the initialise chain's
 * start (fit/lm.py:427-493); a non-finite fallback row is not armed. */
int apx_batch_start_fallback(const apx_batch* batch, const double* rep0, const double* fallback,
                             void* stream);

/* One LM tick of every unfinished fit.  Within a sub-step the probe render
 * (x + 0.1 h) runs on `stream` and the trial render (x + h, the reference's
 * trial point at its default acceleration 0) on the device's second stream,
 * forked and joined by events, so a graph captured on `stream` holds both
 * branches.  Fails with APX_E_INVALID before apx_batch_start on the device. */
int apx_batch_tick(const apx_batch* batch, void* stream);

/* Results (device arrays): best state (res(), fit/base.py:104-117), its chi2
 * (reduced), status (0 running, 1 success, 2 success by immobility, 3 fail:
 * no improving step, 4 fail: max iterations, 5 skipped), iterations (all
 * runs), fallback (1 where the fallback start ran), and the number of
 * finished fits in done[0].  Any output but rep may be null. */
int apx_batch_results(const apx_batch* batch, double* rep, double* chi2, int32_t* status,
                      int32_t* iterations, int32_t* fallback, int32_t* done, void* stream);

/* Work counters of the last render / Jacobian / tick stage, copied to out
 * (device, 8 int32): [0] fits listed, [1] 256-pixel chunks, [2] output tiles,
 * [3] pixels refined past level 1 (each integrates gridding^2 level-2
 * sub-pixels of quad_level^2 samples), [4] undecided level-1 selections,
 * [5] pixels redone in float64, [6] level-3 sub-pixels integrated by the
 * float32 pass, [7] by the float64 pass (each quad_level^2 gridding^2
 * samples).  The profile evaluations of the float32 level-2/3 pass are
 * gridding^2 quad_level^2 ([3] + [6]).  No counterpart in the reference:
 * it measures the work of utils/operations.py:210-247 as run here. */
int apx_batch_counters(const apx_batch* batch, int32_t* out, void* stream);

/* Last error message of the calling thread. */
const char* apx_last_error(void);

/* ---------------------------------------------------------------------------
 * A group model whose sources sit on windows of one image (north-star
 * configuration C3: hundreds of Sersic sources plus a flat sky fitted
 * jointly).  Each source is one cutout of an apx_batch (its window on the
 * image), so its model and its 7 Jacobian columns (parameter-major, as
 * apx_batch_jacobian writes them) exist only on that window.  These entry
 * points give Levenberg-Marquardt (fit/lm.py:248-406) what it needs from the
 * whole group without forming the dense pixels x parameters Jacobian of
 * group_model_object.py:233-283.  The host builds the per-tile source lists
 * (64 x 16 image tiles) and the list of overlapping window pairs.
 * ------------------------------------------------------------------------- */
typedef struct apx_group {
  int32_t nx, ny;           /* image (the fit window), row-major */
  int32_t nsrc;             /* sources = cutouts of the batch, in group order */
  int32_t np;               /* group parameters: 7 per source (+ 1 sky) */
  int32_t sky_col;          /* column of the sky's F (representation), -1 = no sky */
  int32_t sky_after;        /* sources ahead of the sky in the group order; -1 = no sky */
  int32_t ntx, nty;         /* (nx + 63) / 64, (ny + 15) / 16 */
  int32_t npair;            /* overlapping window pairs, (a, a) included */
  int32_t reserved;
  const int32_t* win;       /* nsrc x 4: x0, y0, width, height on the image (inside it) */
  const int64_t* pix_off;   /* nsrc: the window's first pixel in per-source buffers */
  const int32_t* col0;      /* nsrc: the source's first column (7 consecutive) */
  const int32_t* tile_ptr;  /* ntx * nty + 1: CSR offsets into tile_src */
  const int32_t* tile_src;  /* sources whose window meets each tile, ascending */
  const int32_t* pair;      /* npair x 2: (a, b), a <= b, windows overlapping */
  int64_t nsrcpix;          /* per-source buffer length (the batch's npix) */
} apx_group;

/* Workspace (bytes) apx_group_normal and apx_group_rpp need. */
int64_t apx_group_workspace_bytes(const apx_group* group);

/* out (ny x nx float32) = the group image: every pixel sums the sources whose
 * window covers it, in group order, with the flat sky value `sky` added at
 * its place in that order (group_model_object.py:183-231). */
int apx_group_image(const apx_group* group, const float* src_model, double sky, float* out,
                    void* stream);

/* H (np x np float64, row-major) = J^T W J and grad (np) = J^T W (data -
 * model) over unmasked pixels (fit/lm.py:387-399): a 7 x 7 block per
 * overlapping pair, each source's sky-column entries, and the sky's own,
 * where the sky column of J is the constant sky_dcol = d(sky value)/d(rep of F).
 * J: 7 x nsrcpix float32 (parameter-major per-source blocks). */
int apx_group_normal(const apx_group* group, const float* J, const float* model, const float* data,
                     const float* weight, const uint8_t* mask, double sky_dcol, double* hess,
                     double* grad, void* workspace, int64_t workspace_bytes, void* stream);

/* rpp (np, float64) = J^T ((2/d) (W (m1 - m0) / d - W (J h))) over unmasked
 * pixels (fit/lm.py:401-406). */
int apx_group_rpp(const apx_group* group, const float* J, const float* m0, const float* m1,
                  const float* weight, const uint8_t* mask, const double* h, double d, double sky_dcol,
                  double* rpp, void* workspace, int64_t workspace_bytes, void* stream);

/* Damped matrix of fit/lm.py:359-371, A(L)_ii = H_ii + L (1 + H_ii), A(L)_ij =
 * H_ij / (1 + L), factored A = L L^T in place into `factor` (n x n float64,
 * lower triangle, with L^T in the upper triangle for the solve; blocked
 * right-looking Cholesky, 32-column panels).  `hess` is symmetric.  Rows that
 * start late cost less: the trailing update of a panel skips the 64 x 64 tiles
 * whose rows or columns have only zeros up to that panel (a band matrix, e.g.
 * a group's normal matrix with the sources in window order), which leaves the
 * result unchanged.  status[0] (device) = 0, or k + 1 when pivot k was not
 * positive (the factor then holds NaN and so will every solution, which the
 * caller's LM treats as a failed step). */
int apx_dense_damped_factor(int32_t n, const double* hess, double L, double* factor, int32_t* status,
                            void* stream);

/* x = A^-1 b from the factor of apx_dense_damped_factor (two blocked
 * triangular solves, two 32-row blocks a launch; float64, device). */
int apx_dense_cholesky_solve(int32_t n, const double* factor, const double* b, double* x, void* stream);

/* -------------------------------------------------------------------------
 * Learned initialiser: primitives of a small CNN (4 convolutions 3x3 /
 * stride 2 / pad 1, 32-32-64-64 channels, then a 2-layer MLP) that maps a
 * 64 x 64 asinh-normalised cutout to the 7 Sersic parameters LM starts from.
 * The reference has no counterpart: its LM starts from the initialise chain
 * (apx_batch_moment_init above), which stays the fallback.  Bf16 values are
 * uint16 (round to nearest even); activations are NHWC.
 * ------------------------------------------------------------------------- */

/* C[M,N] (= or +=) A[M,K] B[K,N] (+ bias[N], ReLU) with BF16 MFMA, float32
 * accumulate.  A(m,k) = A[m*sam + k*sak], B(k,n) = B[k*sbk + n*sbn], C row
 * pitch ldc; Cb (optional) receives a bf16 copy of C.  splits > 1 divides K
 * over that many workgroup layers whose partials (in ws, >= splits*M*N
 * floats) are summed in a fixed order. */
int apx_gemm_bf16(int32_t M, int32_t N, int32_t K, const uint16_t* A, int64_t sam, int64_t sak,
                  const uint16_t* B, int64_t sbk, int64_t sbn, float* C, int64_t ldc,
                  const float* bias, int32_t relu, uint16_t* Cb, int32_t accumulate, int32_t splits,
                  float* ws, int64_t ws_floats, void* stream);

/* Weighted mean-squared error of B x N outputs y against targets t with
 * per-column weights w: loss[0] = sum w_j (y - t)^2 / B, dy its gradient. */
int apx_mse(const float* y, const float* t, const float* w, int32_t B, int32_t N, float* dy,
            float* loss, void* stream);

/* im2col of a 3x3 / stride-2 / pad-1 convolution of X (B,H,W,C) into
 * col (B*ceil(H/2)*ceil(W/2), Kp), columns (ky*3+kx)*C + c, zero beyond 9C. */
int apx_im2col_s2(const uint16_t* X, int32_t B, int32_t H, int32_t W, int32_t C, int32_t Kp,
                  uint16_t* col, void* stream);

/* The 3x3 / stride-2 / pad-1 convolution C = im2col(X) Wt (+ bias, ReLU) in
 * one BF16 MFMA GEMM whose A operand is read straight from X (B,H,W,C)
 * NHWC bf16 (8 channels a 16-byte load when C % 8 == 0): the same result as
 * apx_im2col_s2 followed by apx_gemm_bf16 (sam = Kp, sak = 1, sbk = N,
 * sbn = 1, ldc = N), without the col buffer.  Wt is (Kp, N) bf16, Kp a
 * multiple of 32 and >= 9C; C (B*ceil(H/2)*ceil(W/2), N) float32; Cb an
 * optional bf16 copy. */
int apx_conv_s2_bf16(const uint16_t* X, int32_t B, int32_t H, int32_t W, int32_t C, int32_t Kp,
                     const uint16_t* Wt, int32_t N, float* out, const float* bias, int32_t relu,
                     uint16_t* outb, void* stream);

/* The adjoint of apx_im2col_s2: dX (B,H,W,C) float32 from dcol. */
int apx_col2im_s2(const float* dcol, int32_t B, int32_t H, int32_t W, int32_t C, int32_t Kp,
                  float* dX, void* stream);

/* dst = bf16(src), zeroed where mask <= 0 when mask is given (ReLU gate);
 * dstf (optional) receives the gated float32 values. */
int apx_cast_gate_bf16(const float* src, const float* mask, int64_t n, uint16_t* dst, float* dstf,
                       void* stream);

/* out[n] = sum_m X[m,n] (bias gradients). */
int apx_colsum(const float* X, int32_t M, int32_t N, float* out, void* stream);

/* apx_cast_gate_bf16 of src (M, N) into dst, and out[n] = sum_m of the gated
 * float32 values, in one pass.  ws: at least N floats, one partial sum row a
 * workgroup (512 N floats let every workgroup have its own). */
int apx_gate_colsum_bf16(const float* src, const float* mask, int32_t M, int32_t N, uint16_t* dst,
                         float* out, float* ws, int64_t ws_floats, void* stream);

/* One Adam step (bias-corrected, step >= 1) on float32 weights w with
 * gradient g and moments m, v; w_bf16 (optional) receives bf16(w). */
int apx_adam(float* w, const float* g, float* m, float* v, int64_t n, float lr, float beta1,
             float beta2, float eps, int32_t step, uint16_t* w_bf16, void* stream);

/* Network input: out = bf16(asinh(x / sigma[b])) for B cutouts of npx pixels. */
int apx_asinh_input(const float* x, const float* sigma, int32_t B, int32_t npx, uint16_t* out,
                    void* stream);

/* The network's input and four convolutions of B cutouts (64 x 64 float32
 * images, sigma (B,)) without the layers between in memory: out (B, 4, 4, 64)
 * bf16, the bits of apx_asinh_input and four apx_conv_s2_bf16 with bias and
 * ReLU.  w, b: host arrays of the four convolutions' device pointers, w[k]
 * (K, Cout) bf16 with K padded to 32, b[k] (Cout,) float32.  workspace (on 16
 * bytes): apx_init_features_workspace_bytes() bytes. */
int64_t apx_init_features_workspace_bytes(void);
int apx_init_features(const float* images, const float* sigma, int32_t B, const uint16_t* const* w,
                      const float* const* b, uint16_t* out, void* workspace, int64_t workspace_bytes,
                      void* stream);

#ifdef __cplusplus
}
#endif

#endif /* ASTROPHOT_HIP_H */
