// The block's scan parameters from its learned ones, one kernel each way.
//
// Reference behaviour: e_model.py:210-230 (TwoLevelDelta: softplus(a) + eps for
// the idle and the active level), :455-470 (A = -exp(A_log), W_B and W_C the
// halves of W_BC's rows).
//
// A few thousand values: what counts is launches. Torch runs them as nine
// kernels forward and a dozen backward (softplus, add, exp, negation, two strided
// copies, their gradients and the two halves' zero-padded sum): 20 launches
// of 1.5 to 4 us of GPU time each, and as many dispatches on the host. Here it is
// one launch each way.
#include "bcm_common.hpp"

namespace bcm {

// torch's softplus (beta 1, threshold 20) and its gradient's factor
__device__ __forceinline__ float softplus(float a) { return a > 20.0f ? a : log1pf(expf(a)); }
__device__ __forceinline__ float softplus_grad(float a, float g) {
  const float z = expf(a);
  return a > 20.0f ? g : g * z / (z + 1.0f);
}

__global__ __launch_bounds__(256) void k_block_params_fwd(const float* __restrict__ a0, const float* __restrict__ a1,
                                                          const float* __restrict__ a_log,
                                                          const float* __restrict__ w_bc, int D, int N, float eps,
                                                          float* __restrict__ dt_idle, float* __restrict__ dt_active,
                                                          float* __restrict__ A, float* __restrict__ W_B,
                                                          float* __restrict__ W_C) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)D * N) return;
  const int d = (int)(i / N), s = (int)(i - (int64_t)d * N);
  A[i] = -expf(a_log[i]);
  W_B[i] = w_bc[(int64_t)d * 2 * N + s];
  W_C[i] = w_bc[(int64_t)d * 2 * N + N + s];
  if (s == 0) {
    dt_idle[d] = softplus(a0[d]) + eps;
    dt_active[d] = softplus(a1[d]) + eps;
  }
}

// Any gradient may be missing (null: zero).
__global__ __launch_bounds__(256) void k_block_params_bwd(const float* __restrict__ a0, const float* __restrict__ a1,
                                                          const float* __restrict__ A, int D, int N,
                                                          const float* __restrict__ g_idle,
                                                          const float* __restrict__ g_active,
                                                          const float* __restrict__ gA, const float* __restrict__ gB,
                                                          const float* __restrict__ gC, float* __restrict__ da0,
                                                          float* __restrict__ da1, float* __restrict__ da_log,
                                                          float* __restrict__ dw_bc) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)D * N) return;
  const int d = (int)(i / N), s = (int)(i - (int64_t)d * N);
  da_log[i] = gA ? gA[i] * A[i] : 0.0f;  // d(-exp(a)) = -exp(a)
  dw_bc[(int64_t)d * 2 * N + s] = gB ? gB[i] : 0.0f;
  dw_bc[(int64_t)d * 2 * N + N + s] = gC ? gC[i] : 0.0f;
  if (s == 0) {
    da0[d] = g_idle ? softplus_grad(a0[d], g_idle[d]) : 0.0f;
    da1[d] = g_active ? softplus_grad(a1[d], g_active[d]) : 0.0f;
  }
}

static int params_checks(const char* fn, int64_t D, int64_t N) {
  if (D < 0 || N < 1 || D * N > INT32_MAX) return set_error(BCM_EINVAL, "%s: invalid sizes", fn);
  return BCM_OK;
}

}  // namespace bcm

using namespace bcm;

extern "C" {

int bcm_block_params_fwd(const float* a0, const float* a1, const float* a_log, const float* w_bc, int64_t D, int64_t N,
                         float eps, float* dt_idle, float* dt_active, float* A, float* W_B, float* W_C,
                         bcm_stream_t stream) {
  const char* fn = "bcm_block_params_fwd";
  const int rc = params_checks(fn, D, N);
  if (rc || D == 0) return rc;
  if (!a0 || !a1 || !a_log || !w_bc || !dt_idle || !dt_active || !A || !W_B || !W_C)
    return set_error(BCM_EINVAL, "%s: null pointer", fn);
  hipLaunchKernelGGL(k_block_params_fwd, dim3((unsigned)((D * N + 255) / 256)), dim3(256), 0, hs(stream), a0, a1, a_log,
                     w_bc, (int)D, (int)N, eps, dt_idle, dt_active, A, W_B, W_C);
  return check_launch(fn);
}

int bcm_block_params_bwd(const float* a0, const float* a1, const float* A, int64_t D, int64_t N, const float* g_idle,
                         const float* g_active, const float* gA, const float* gB, const float* gC, float* da0,
                         float* da1, float* da_log, float* dw_bc, bcm_stream_t stream) {
  const char* fn = "bcm_block_params_bwd";
  const int rc = params_checks(fn, D, N);
  if (rc || D == 0) return rc;
  if (!a0 || !a1 || !A || !da0 || !da1 || !da_log || !dw_bc) return set_error(BCM_EINVAL, "%s: null pointer", fn);
  hipLaunchKernelGGL(k_block_params_bwd, dim3((unsigned)((D * N + 255) / 256)), dim3(256), 0, hs(stream), a0, a1, A,
                     (int)D, (int)N, g_idle, g_active, gA, gB, gC, da0, da1, da_log, dw_bc);
  return check_launch(fn);
}

}  // extern "C"
