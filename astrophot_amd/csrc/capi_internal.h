// Internal declarations shared by the .hip translation units of libastrophot_hip.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "../../include/astrophot_hip.h"

namespace apx {

// Records `msg` as the calling thread's last error and returns `code`.
int set_error(int code, const char* msg);
// APX_OK, or APX_E_HIP with the runtime's message if the last launch failed.
int check_launch(const char* where);

int64_t render_workspace_bytes(int64_t npix);
int render_component(const apx_component* cp, float* planes, void* workspace, int64_t ws_bytes,
                     hipStream_t stream);
int render_vjp(const apx_component* cp, const float* weights, float* value_plane, double* grad,
               void* workspace, int64_t ws_bytes, hipStream_t stream);
int render_selected_count(const void* workspace, hipStream_t stream, int32_t* count);
int normalize_planes(float* planes, int32_t nchan, int64_t npix, hipStream_t stream);

int psf_shift(const float* psf, int32_t ph, int32_t pw, double sx, double sy, const double* pinv,
              double dvdr_x, double dvdr_y, float* kernels, hipStream_t stream);
int psf_kernels_dparam(const float* psf, const float* dpsf, int32_t nd, int32_t ph, int32_t pw,
                       int32_t shifted, double sx, double sy, float* out, hipStream_t stream);
int block_sum_add(const apx_block_sum* job, const float* src, hipStream_t stream);
int64_t convolve_workspace_bytes(int32_t kh, int32_t kw);
int convolve(const apx_conv_job* job, const float* planes, const float* kernels, void* workspace,
             int64_t ws_bytes, hipStream_t stream);

int group_image(const apx_group* g, const float* src, double sky, float* out, hipStream_t stream);
int64_t group_workspace_bytes(const apx_group* g);
int group_normal(const apx_group* g, const float* J, const float* model, const float* data,
                 const float* weight, const uint8_t* mask, double sky_dcol, double* H, double* grad,
                 void* ws, int64_t ws_bytes, hipStream_t stream);
int group_rpp(const apx_group* g, const float* J, const float* m0, const float* m1, const float* weight,
              const uint8_t* mask, const double* h, double d, double sky_dcol, double* out, void* ws,
              int64_t ws_bytes, hipStream_t stream);
int dense_damped_factor(int32_t n, const double* H, double L, double* A, int32_t* status, hipStream_t stream);
int dense_cholesky_solve(int32_t n, const double* A, const double* b, double* x, hipStream_t stream);

int64_t reduce_workspace_bytes(int64_t npix, int32_t np);
int chi2(const float* model, const float* data, const float* weight, const uint8_t* mask,
         int64_t npix, double* out, void* ws, int64_t ws_bytes, hipStream_t stream);
int normal_equations(const float* J, const float* model, const float* data, const float* weight,
                     const uint8_t* mask, int64_t npix, int32_t np, double* hess, double* grad,
                     void* ws, int64_t ws_bytes, hipStream_t stream);
int normal_equations_noalloc(const float* J, const float* model, const float* data,
                             const float* weight, const uint8_t* mask, int64_t npix, int32_t np,
                             double* hess, double* grad, hipStream_t stream);
int rpp(const float* J, const float* m0, const float* m1, const float* weight, const uint8_t* mask,
        int64_t npix, int32_t np, const double* h, double d, double* out, void* ws,
        int64_t ws_bytes, hipStream_t stream);
int lm_solve(const double* hess, const double* grad, int32_t np, double L, double* h,
             int32_t* status, hipStream_t stream);

int batch_plan(apx_batch_galaxy* gal, int32_t ngal, apx_batch* b);
int64_t batch_state_bytes();
int64_t batch_scratch_bytes(const apx_batch* b);
int batch_render(const apx_batch* b, const double* rep, float* out, int32_t parts,
                 hipStream_t stream);
int batch_jacobian(const apx_batch* b, const double* rep, float* out, int32_t parts,
                 hipStream_t stream);
int batch_start(const apx_batch* b, const double* rep0, const double* fallback, hipStream_t stream);
int batch_tick(const apx_batch* b, hipStream_t stream);
int batch_moment_init(const apx_batch* b, double* rep, hipStream_t stream);
double sersic_light_fraction(double n, double r_over_re);
int gemm_bf16(int M, int N, int K, const uint16_t* A, int64_t sam, int64_t sak, const uint16_t* B,
              int64_t sbk, int64_t sbn, float* C, int64_t ldc, const float* bias, int relu,
              uint16_t* Cb, int accumulate, int splits, float* ws, int64_t ws_floats,
              hipStream_t stream);
int conv_s2_bf16(const uint16_t* X, int Bn, int H, int W, int Cin, int Kp, const uint16_t* Wt, int N,
                 float* C, const float* bias, int relu, uint16_t* Cb, hipStream_t stream);
int mse(const float* y, const float* t, const float* w, int Bn, int N, float* dy, float* loss,
        hipStream_t stream);
int im2col_s2(const uint16_t* X, int Bn, int H, int W, int Cin, int Kp, uint16_t* col,
              hipStream_t stream);
int col2im_s2(const float* dcol, int Bn, int H, int W, int Cin, int Kp, float* dX, hipStream_t stream);
int cast_gate(const float* src, const float* mask, int64_t n, uint16_t* dst, float* dstf,
              hipStream_t stream);
int colsum(const float* X, int M, int N, float* out, hipStream_t stream);
int gate_colsum(const float* src, const float* mask, int M, int N, uint16_t* dst, float* out, float* ws,
                int64_t ws_floats, hipStream_t stream);
int adam(float* w, const float* g, float* m, float* v, int64_t n, float lr, float b1, float b2,
         float eps, int step, uint16_t* wb, hipStream_t stream);
int asinh_input(const float* x, const float* sigma, int Bn, int npx, uint16_t* out, hipStream_t stream);
int64_t init_features_workspace_bytes();
int init_features(const float* images, const float* sigma, int Bn, const uint16_t* const* w, const float* const* b,
                  uint16_t* out, void* ws, int64_t ws_bytes, hipStream_t stream);
int batch_counters(const apx_batch* b, int32_t* out, hipStream_t stream);
int batch_results(const apx_batch* b, double* rep, double* chi2, int32_t* status, int32_t* iters,
                  int32_t* fallback, int32_t* done, hipStream_t stream);

}  // namespace apx
