// extern "C" entry points of libastrophot_hip (declared in
// include/astrophot_hip.h) and the thread-local error record.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>

#include "capi_internal.h"

namespace apx {

namespace {
thread_local char g_last_error[512] = "";
}

int set_error(int code, const char* msg) {
  std::snprintf(g_last_error, sizeof(g_last_error), "%s", msg);
  return code;
}

int check_launch(const char* where) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    std::snprintf(g_last_error, sizeof(g_last_error), "%s: %s", where, hipGetErrorString(e));
    return APX_E_HIP;
  }
  return APX_OK;
}

}  // namespace apx

extern "C" {

const char* apx_last_error(void) { return apx::g_last_error; }

int64_t apx_render_workspace_bytes(int64_t npix) { return apx::render_workspace_bytes(npix); }

int apx_render_component(const apx_component* comp, float* planes, void* workspace,
                         int64_t workspace_bytes, void* stream) {
  return apx::render_component(comp, planes, workspace, workspace_bytes,
                               static_cast<hipStream_t>(stream));
}

int apx_render_vjp(const apx_component* comp, const float* weights, float* value_plane,
                   double* grad, void* workspace, int64_t workspace_bytes, void* stream) {
  return apx::render_vjp(comp, weights, value_plane, grad, workspace, workspace_bytes,
                         static_cast<hipStream_t>(stream));
}

int apx_render_selected_count(const void* workspace, void* stream, int32_t* count) {
  return apx::render_selected_count(workspace, static_cast<hipStream_t>(stream), count);
}

int apx_psf_shift(const float* psf, int32_t ph, int32_t pw, double shift_x, double shift_y,
                  const double* pinv, double dvdr_x, double dvdr_y, float* kernels,
                  void* stream) {
  return apx::psf_shift(psf, ph, pw, shift_x, shift_y, pinv, dvdr_x, dvdr_y, kernels,
                        static_cast<hipStream_t>(stream));
}

int apx_normalize_planes(float* planes, int32_t nchan, int64_t npix, void* stream) {
  return apx::normalize_planes(planes, nchan, npix, static_cast<hipStream_t>(stream));
}

int apx_psf_kernels_dparam(const float* psf, const float* dpsf, int32_t nd, int32_t ph, int32_t pw,
                           int32_t shifted, double shift_x, double shift_y, float* out,
                           void* stream) {
  return apx::psf_kernels_dparam(psf, dpsf, nd, ph, pw, shifted, shift_x, shift_y, out,
                                 static_cast<hipStream_t>(stream));
}

int64_t apx_convolve_workspace_bytes(int32_t kh, int32_t kw) {
  return apx::convolve_workspace_bytes(kh, kw);
}

int apx_convolve(const apx_conv_job* job, const float* planes, const float* kernels,
                 void* workspace, int64_t workspace_bytes, void* stream) {
  return apx::convolve(job, planes, kernels, workspace, workspace_bytes,
                       static_cast<hipStream_t>(stream));
}

int apx_block_sum_add(const apx_block_sum* job, const float* src, void* stream) {
  return apx::block_sum_add(job, src, static_cast<hipStream_t>(stream));
}

int64_t apx_group_workspace_bytes(const apx_group* group) { return apx::group_workspace_bytes(group); }

int apx_group_image(const apx_group* group, const float* src_model, double sky, float* out, void* stream) {
  return apx::group_image(group, src_model, sky, out, static_cast<hipStream_t>(stream));
}

int apx_group_normal(const apx_group* group, const float* J, const float* model, const float* data,
                     const float* weight, const uint8_t* mask, double sky_dcol, double* hess, double* grad,
                     void* workspace, int64_t workspace_bytes, void* stream) {
  return apx::group_normal(group, J, model, data, weight, mask, sky_dcol, hess, grad, workspace,
                           workspace_bytes, static_cast<hipStream_t>(stream));
}

int apx_group_rpp(const apx_group* group, const float* J, const float* m0, const float* m1,
                  const float* weight, const uint8_t* mask, const double* h, double d, double sky_dcol,
                  double* rpp, void* workspace, int64_t workspace_bytes, void* stream) {
  return apx::group_rpp(group, J, m0, m1, weight, mask, h, d, sky_dcol, rpp, workspace, workspace_bytes,
                        static_cast<hipStream_t>(stream));
}

int apx_dense_damped_factor(int32_t n, const double* hess, double L, double* factor, int32_t* status,
                            void* stream) {
  return apx::dense_damped_factor(n, hess, L, factor, status, static_cast<hipStream_t>(stream));
}

int apx_dense_cholesky_solve(int32_t n, const double* factor, const double* b, double* x, void* stream) {
  return apx::dense_cholesky_solve(n, factor, b, x, static_cast<hipStream_t>(stream));
}

int64_t apx_reduce_workspace_bytes(int64_t npix, int32_t np) {
  return apx::reduce_workspace_bytes(npix, np);
}

int apx_chi2(const float* model, const float* data, const float* weight, const uint8_t* mask,
             int64_t npix, double* out, void* workspace, int64_t workspace_bytes, void* stream) {
  return apx::chi2(model, data, weight, mask, npix, out, workspace, workspace_bytes,
                   static_cast<hipStream_t>(stream));
}

int apx_normal_equations(const float* J, const float* model, const float* data, const float* weight,
                         const uint8_t* mask, int64_t npix, int32_t np, double* hess, double* grad,
                         void* workspace, int64_t workspace_bytes, void* stream) {
  return apx::normal_equations(J, model, data, weight, mask, npix, np, hess, grad, workspace,
                               workspace_bytes, static_cast<hipStream_t>(stream));
}

int apx_normal_equations_noalloc(const float* J, const float* model, const float* data,
                                 const float* weight, const uint8_t* mask, int64_t npix, int32_t np,
                                 double* hess, double* grad, void* stream) {
  return apx::normal_equations_noalloc(J, model, data, weight, mask, npix, np, hess, grad,
                                       static_cast<hipStream_t>(stream));
}

int apx_rpp(const float* J, const float* m0, const float* m1, const float* weight,
            const uint8_t* mask, int64_t npix, int32_t np, const double* h, double d, double* rpp,
            void* workspace, int64_t workspace_bytes, void* stream) {
  return apx::rpp(J, m0, m1, weight, mask, npix, np, h, d, rpp, workspace, workspace_bytes,
                  static_cast<hipStream_t>(stream));
}

int apx_lm_solve(const double* hess, const double* grad, int32_t np, double L, double* h,
                 int32_t* status, void* stream) {
  return apx::lm_solve(hess, grad, np, L, h, status, static_cast<hipStream_t>(stream));
}

int apx_batch_plan(apx_batch_galaxy* gal, int32_t ngal, apx_batch* batch) {
  return apx::batch_plan(gal, ngal, batch);
}

int64_t apx_batch_state_bytes(void) { return apx::batch_state_bytes(); }

int64_t apx_batch_scratch_bytes(const apx_batch* batch) { return apx::batch_scratch_bytes(batch); }

int apx_batch_render(const apx_batch* batch, const double* rep, float* out, int32_t parts,
                     void* stream) {
  return apx::batch_render(batch, rep, out, parts, static_cast<hipStream_t>(stream));
}

int apx_batch_jacobian(const apx_batch* batch, const double* rep, float* out, int32_t parts,
                       void* stream) {
  return apx::batch_jacobian(batch, rep, out, parts, static_cast<hipStream_t>(stream));
}

int apx_batch_moment_init(const apx_batch* batch, double* rep, void* stream) {
  return apx::batch_moment_init(batch, rep, static_cast<hipStream_t>(stream));
}

double apx_sersic_light_fraction(double n, double r_over_re) {
  return apx::sersic_light_fraction(n, r_over_re);
}

int apx_batch_start(const apx_batch* batch, const double* rep0, void* stream) {
  return apx::batch_start(batch, rep0, nullptr, static_cast<hipStream_t>(stream));
}

int apx_batch_start_fallback(const apx_batch* batch, const double* rep0, const double* fallback,
                             void* stream) {
  if (!fallback) return apx::set_error(APX_E_INVALID, "batch_start_fallback: null fallback");
  return apx::batch_start(batch, rep0, fallback, static_cast<hipStream_t>(stream));
}

int apx_batch_tick(const apx_batch* batch, void* stream) {
  return apx::batch_tick(batch, static_cast<hipStream_t>(stream));
}

int apx_batch_counters(const apx_batch* batch, int32_t* out, void* stream) {
  return apx::batch_counters(batch, out, static_cast<hipStream_t>(stream));
}

int apx_batch_results(const apx_batch* batch, double* rep, double* chi2, int32_t* status,
                      int32_t* iterations, int32_t* fallback, int32_t* done, void* stream) {
  return apx::batch_results(batch, rep, chi2, status, iterations, fallback, done,
                            static_cast<hipStream_t>(stream));
}


/* ---- learned initialiser: BF16 MFMA network primitives ---------------- */
int apx_gemm_bf16(int32_t M, int32_t N, int32_t K, const uint16_t* A, int64_t sam, int64_t sak,
                  const uint16_t* B, int64_t sbk, int64_t sbn, float* C, int64_t ldc,
                  const float* bias, int32_t relu, uint16_t* Cb, int32_t accumulate, int32_t splits,
                  float* ws, int64_t ws_floats, void* stream) {
  return apx::gemm_bf16(M, N, K, A, sam, sak, B, sbk, sbn, C, ldc, bias, relu, Cb, accumulate, splits,
                        ws, ws_floats, static_cast<hipStream_t>(stream));
}

int apx_mse(const float* y, const float* t, const float* w, int32_t B, int32_t N, float* dy,
            float* loss, void* stream) {
  return apx::mse(y, t, w, B, N, dy, loss, static_cast<hipStream_t>(stream));
}

int apx_im2col_s2(const uint16_t* X, int32_t B, int32_t H, int32_t W, int32_t C, int32_t Kp,
                  uint16_t* col, void* stream) {
  return apx::im2col_s2(X, B, H, W, C, Kp, col, static_cast<hipStream_t>(stream));
}

int apx_conv_s2_bf16(const uint16_t* X, int32_t B, int32_t H, int32_t W, int32_t C, int32_t Kp,
                     const uint16_t* Wt, int32_t N, float* out, const float* bias, int32_t relu,
                     uint16_t* outb, void* stream) {
  return apx::conv_s2_bf16(X, B, H, W, C, Kp, Wt, N, out, bias, relu, outb, static_cast<hipStream_t>(stream));
}

int apx_col2im_s2(const float* dcol, int32_t B, int32_t H, int32_t W, int32_t C, int32_t Kp,
                  float* dX, void* stream) {
  return apx::col2im_s2(dcol, B, H, W, C, Kp, dX, static_cast<hipStream_t>(stream));
}

int apx_cast_gate_bf16(const float* src, const float* mask, int64_t n, uint16_t* dst, float* dstf,
                       void* stream) {
  return apx::cast_gate(src, mask, n, dst, dstf, static_cast<hipStream_t>(stream));
}

int apx_gate_colsum_bf16(const float* src, const float* mask, int32_t M, int32_t N, uint16_t* dst, float* out,
                         float* ws, int64_t ws_floats, void* stream) {
  return apx::gate_colsum(src, mask, M, N, dst, out, ws, ws_floats, static_cast<hipStream_t>(stream));
}

int apx_colsum(const float* X, int32_t M, int32_t N, float* out, void* stream) {
  return apx::colsum(X, M, N, out, static_cast<hipStream_t>(stream));
}

int apx_adam(float* w, const float* g, float* m, float* v, int64_t n, float lr, float beta1,
             float beta2, float eps, int32_t step, uint16_t* w_bf16, void* stream) {
  return apx::adam(w, g, m, v, n, lr, beta1, beta2, eps, step, w_bf16, static_cast<hipStream_t>(stream));
}

int64_t apx_init_features_workspace_bytes(void) { return apx::init_features_workspace_bytes(); }

int apx_init_features(const float* images, const float* sigma, int32_t B, const uint16_t* const* w, const float* const* b,
                      uint16_t* out, void* workspace, int64_t workspace_bytes, void* stream) {
  return apx::init_features(images, sigma, B, w, b, out, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

int apx_asinh_input(const float* x, const float* sigma, int32_t B, int32_t npx, uint16_t* out,
                    void* stream) {
  return apx::asinh_input(x, sigma, B, npx, out, static_cast<hipStream_t>(stream));
}

}  // extern "C"
