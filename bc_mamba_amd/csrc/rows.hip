// Row passes of the network around the blocks: the leaky residual with its
// layer norm, and the gradient of a spike head's logits.
//
// Reference behaviour: lra_impl.py:1381-1427 (v' = alpha v + block(s),
// h = norm(v')), e_model.py:233-254 and :326-333 (p = sigmoid(logits), the
// spikes pass p's gradient on).
//
// Bound by memory: what counts is how often a [tokens, D] array is read and
// written. Torch runs the forward as three kernels over 7 arrays (17 + 24 + 54 us
// at 51200 x 256) and the backward as six over 13 (50 + 50 + 5 us for the
// norm, 24 + 17 us for the sum and the scaled gradient); here the forward is one
// kernel over 4 arrays (33 us) and the backward one over 5 (40 us, and 5 for the
// reduction of the workgroups' column sums): near 6 TB/s, part of it from the
// last-level cache. The head's gradient and its bias gradient take one kernel
// and the reduction for torch's two (24 + 30 -> 26 + 5 us). D up to 1024, a row in the registers of at most one wave.
#include "bcm_common.hpp"

#include <algorithm>

namespace bcm {

// A row is held by LP lanes, 4 NV values each (4 LP NV >= D); a wave holds
// 64 / LP rows. D is a multiple of 4.
template <int LP, int NV> struct RowAt {
  int lane, D;
  __device__ __forceinline__ explicit RowAt(int D_) : lane(threadIdx.x % LP), D(D_) {}
  __device__ __forceinline__ int col(int i) const { return 4 * (lane + LP * i); }
  __device__ __forceinline__ bool ok(int i) const { return col(i) < D; }
  __device__ __forceinline__ void load(float4 (&x)[NV], const float* p) const {
#pragma unroll
    for (int i = 0; i < NV; ++i)
      x[i] = ok(i) ? *reinterpret_cast<const float4*>(p + col(i)) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  __device__ __forceinline__ void store(float* p, const float4 (&x)[NV]) const {
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (ok(i)) *reinterpret_cast<float4*>(p + col(i)) = x[i];
  }
  static __device__ __forceinline__ float sum(float v) {
#pragma unroll
    for (int o = LP / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
  }
};

__device__ __forceinline__ float sum4(const float4& a) { return (a.x + a.y) + (a.z + a.w); }
__device__ __forceinline__ float4 mul4(const float4& a, const float4& b) {
  return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w);
}

// v_out = alpha v + dv (v null: the norm of dv, v_out not written),
// h = (v_out - mean) rstd gamma + beta. The variance is summed around the mean.
template <int LP, int NV>
__global__ __launch_bounds__(256) void k_residual_norm_fwd(const float* __restrict__ v, const float* __restrict__ dv,
                                                           float alpha, const float* __restrict__ gamma,
                                                           const float* __restrict__ beta, int64_t rows, int D,
                                                           float eps, float* __restrict__ v_out, float* __restrict__ h,
                                                           float* __restrict__ mean, float* __restrict__ rstd) {
  const RowAt<LP, NV> at(D);
  const int64_t row = (int64_t)blockIdx.x * (256 / LP) + threadIdx.x / LP;
  if (row >= rows) return;
  float4 x[NV], g[NV], b[NV];
  at.load(x, dv + row * D);
  if (v) {
    float4 r[NV];
    at.load(r, v + row * D);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
#pragma clang fp contract(off)  // rounded after the product, as torch rounds it
      x[i].x += alpha * r[i].x, x[i].y += alpha * r[i].y, x[i].z += alpha * r[i].z, x[i].w += alpha * r[i].w;
    }
    at.store(v_out + row * D, x);
  }
  at.load(g, gamma);
  at.load(b, beta);
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; ++i) s += sum4(x[i]);
  const float mu = at.sum(s) / D;
  s = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; ++i)
    if (at.ok(i)) {
      x[i] = make_float4(x[i].x - mu, x[i].y - mu, x[i].z - mu, x[i].w - mu);
      s += sum4(mul4(x[i], x[i]));
    }
  const float rs = 1.0f / sqrtf(at.sum(s) / D + eps);
#pragma unroll
  for (int i = 0; i < NV; ++i)
    x[i] = make_float4(fmaf(x[i].x * rs, g[i].x, b[i].x), fmaf(x[i].y * rs, g[i].y, b[i].y),
                       fmaf(x[i].z * rs, g[i].z, b[i].z), fmaf(x[i].w * rs, g[i].w, b[i].w));
  at.store(h + row * D, x);
  if (at.lane == 0) mean[row] = mu, rstd[row] = rs;
}

// The workgroup's sums over its rows of acc (NA sets of column sums) into part
// [NA D]; every thread comes here.
template <int LP, int NV, int NA>
__device__ __forceinline__ void column_sums(const RowAt<LP, NV>& at, const float4 (&acc)[NA][NV], float* part) {
  constexpr int G = 256 / LP, S = 4 * LP * NV;
  __shared__ __align__(16) float sm[G][NA * S];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int i = 0; i < NV; ++i) *reinterpret_cast<float4*>(&sm[threadIdx.x / LP][a * S + at.col(i)]) = acc[a][i];
  __syncthreads();
  for (int i = threadIdx.x; i < NA * S; i += 256) {
    const int c = i % S;
    if (c >= at.D) continue;
    float v = 0.0f;
#pragma unroll
    for (int g = 0; g < G; ++g) v += sm[g][i];
    part[(i / S) * at.D + c] = v;
  }
}

// g = gv + the norm's gradient of gh at v_out; d_core = g, d_v = alpha g (null:
// not written); part [workgroup][2 D]: the workgroup's share of gamma's and beta's
// gradients. gv may be null (zero). A workgroup takes every gridDim-th set of
// rows, so that few partial sums are left.
template <int LP, int NV>
__global__ __launch_bounds__(256) void k_residual_norm_bwd(const float* __restrict__ gh, const float* __restrict__ gv,
                                                           const float* __restrict__ v_out, float alpha,
                                                           const float* __restrict__ gamma,
                                                           const float* __restrict__ mean,
                                                           const float* __restrict__ rstd, int64_t rows, int D,
                                                           float* __restrict__ d_core, float* __restrict__ d_v,
                                                           float* __restrict__ part) {
  constexpr int G = 256 / LP;
  const RowAt<LP, NV> at(D);
  float4 gm[NV], acc[2][NV] = {};
  at.load(gm, gamma);
  for (int64_t row = (int64_t)blockIdx.x * G + threadIdx.x / LP; row < rows; row += (int64_t)gridDim.x * G) {
    float4 x[NV], g[NV], r[NV];
    at.load(x, v_out + row * D);
    at.load(g, gh + row * D);
    if (gv) at.load(r, gv + row * D);
    const float mu = mean[row], rs = rstd[row];
    float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      x[i] = make_float4((x[i].x - mu) * rs, (x[i].y - mu) * rs, (x[i].z - mu) * rs, (x[i].w - mu) * rs);
      acc[0][i].x = fmaf(g[i].x, x[i].x, acc[0][i].x), acc[0][i].y = fmaf(g[i].y, x[i].y, acc[0][i].y);
      acc[0][i].z = fmaf(g[i].z, x[i].z, acc[0][i].z), acc[0][i].w = fmaf(g[i].w, x[i].w, acc[0][i].w);
      acc[1][i].x += g[i].x, acc[1][i].y += g[i].y, acc[1][i].z += g[i].z, acc[1][i].w += g[i].w;
      g[i] = mul4(g[i], gm[i]);  // zero past D
      s0 += sum4(g[i]);
      s1 += sum4(mul4(g[i], x[i]));
    }
    s0 = at.sum(s0) / D;
    s1 = at.sum(s1) / D;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      g[i] = make_float4(rs * (g[i].x - fmaf(x[i].x, s1, s0)), rs * (g[i].y - fmaf(x[i].y, s1, s0)),
                         rs * (g[i].z - fmaf(x[i].z, s1, s0)), rs * (g[i].w - fmaf(x[i].w, s1, s0)));
      if (gv) g[i] = make_float4(g[i].x + r[i].x, g[i].y + r[i].y, g[i].z + r[i].z, g[i].w + r[i].w);
      r[i] = make_float4(alpha * g[i].x, alpha * g[i].y, alpha * g[i].z, alpha * g[i].w);
    }
    at.store(d_core + row * D, g);
    if (d_v) at.store(d_v + row * D, r);
  }
  column_sums<LP, NV, 2>(at, acc, part + (int64_t)blockIdx.x * 2 * D);
}

// d_logits = ds (1 - p) p with p = sigmoid(logits), rounded as torch rounds it;
// part [workgroup][D]: the workgroup's share of the bias gradient.
template <int LP, int NV>
__global__ __launch_bounds__(256) void k_spike_head_bwd(const float* __restrict__ ds, const float* __restrict__ logits,
                                                        int64_t rows, int D, float* __restrict__ d_logits,
                                                        float* __restrict__ part) {
  constexpr int G = 256 / LP;
  const RowAt<LP, NV> at(D);
  float4 acc[1][NV] = {};
  auto grad = [](float g, float l) {
    const float p = sigmoid_f(l);
    return g * (1.0f - p) * p;
  };
  for (int64_t row = (int64_t)blockIdx.x * G + threadIdx.x / LP; row < rows; row += (int64_t)gridDim.x * G) {
    float4 g[NV], l[NV];
    at.load(g, ds + row * D);
    at.load(l, logits + row * D);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      g[i] = make_float4(grad(g[i].x, l[i].x), grad(g[i].y, l[i].y), grad(g[i].z, l[i].z), grad(g[i].w, l[i].w));
      acc[0][i].x += g[i].x, acc[0][i].y += g[i].y, acc[0][i].z += g[i].z, acc[0][i].w += g[i].w;
    }
    at.store(d_logits + row * D, g);
  }
  column_sums<LP, NV, 1>(at, acc, part + (int64_t)blockIdx.x * D);
}

// part [workgroup][D]: the workgroup's share of x's column sums, in k_spike_head_bwd's
// order (the bias gradient is the same where torch computes the sigmoid's).
template <int LP, int NV>
__global__ __launch_bounds__(256) void k_column_sums(const float* __restrict__ x, int64_t rows, int D,
                                                     float* __restrict__ part) {
  constexpr int G = 256 / LP;
  const RowAt<LP, NV> at(D);
  float4 acc[1][NV] = {};
  for (int64_t row = (int64_t)blockIdx.x * G + threadIdx.x / LP; row < rows; row += (int64_t)gridDim.x * G) {
    float4 g[NV];
    at.load(g, x + row * D);
#pragma unroll
    for (int i = 0; i < NV; ++i)
      acc[0][i].x += g[i].x, acc[0][i].y += g[i].y, acc[0][i].z += g[i].z, acc[0][i].w += g[i].w;
  }
  column_sums<LP, NV, 1>(at, acc, part + (int64_t)blockIdx.x * D);
}

// out0[c] (c < D), out1[c - D] = the sum over the workgroups' shares part [n][cols],
// in a fixed order: 16 columns a workgroup, each summed by 64 threads.
__global__ __launch_bounds__(1024) void k_column_reduce(const float* __restrict__ part, int n, int cols, int D,
                                                        float* __restrict__ out0, float* __restrict__ out1) {
  __shared__ float sm[64][17];
  const int c = blockIdx.x * 16 + threadIdx.x % 16, r = threadIdx.x / 16;
  float v = 0.0f;
  if (c < cols)
#pragma unroll 8
    for (int i = r; i < n; i += 64) v += part[(int64_t)i * cols + c];
  sm[r][threadIdx.x % 16] = v;
  __syncthreads();
  if (r > 0 || c >= cols) return;
  v = 0.0f;
#pragma unroll
  for (int i = 0; i < 64; ++i) v += sm[i][threadIdx.x];
  (c < D ? out0[c] : out1[c - D]) = v;
}

// Lanes a row and float4s a lane for D values; false: no form.
template <typename F> static bool row_form(int64_t D, F&& f) {
  using std::integral_constant;
  auto go = [&](auto lp, auto nv) { f(lp, nv); return true; };
  if (D <= 32) return go(integral_constant<int, 8>{}, integral_constant<int, 1>{});
  if (D <= 64) return go(integral_constant<int, 16>{}, integral_constant<int, 1>{});
  if (D <= 128) return go(integral_constant<int, 32>{}, integral_constant<int, 1>{});
  if (D <= 256) return go(integral_constant<int, 64>{}, integral_constant<int, 1>{});
  if (D <= 512) return go(integral_constant<int, 64>{}, integral_constant<int, 2>{});
  if (D <= 1024) return go(integral_constant<int, 64>{}, integral_constant<int, 4>{});
  return false;
}

// Workgroups of a backward pass: four a CU at most.
static int64_t row_workgroups(int64_t rows, int64_t D) {
  int64_t G = 1;
  row_form(D, [&](auto lp, auto) { G = 256 / decltype(lp)::value; });
  return std::min<int64_t>((rows + G - 1) / G, 4 * (int64_t)device_cus());
}

static int row_check(const char* fn, int64_t rows, int64_t D) {
  if (rows < 0 || rows * std::max<int64_t>(D, 1) > INT32_MAX) return set_error(BCM_EINVAL, "%s: rows * D must fit in int32", fn);
  if (D < 4 || D > 1024 || D % 4) return set_error(BCM_EINVAL, "%s: D must be a multiple of 4 up to 1024", fn);
  return BCM_OK;
}

}  // namespace bcm

using namespace bcm;

extern "C" {

int bcm_residual_norm_fwd(const float* v, const float* dv, float alpha, const float* gamma, const float* beta,
                          int64_t rows, int64_t D, float eps, float* v_out, float* h, float* mean, float* rstd,
                          bcm_stream_t stream) {
  const char* fn = "bcm_residual_norm_fwd";
  if (int rc = row_check(fn, rows, D)) return rc;
  if (rows == 0) return BCM_OK;
  if (!dv || !gamma || !beta || !h || !mean || !rstd || (v && !v_out)) return set_error(BCM_EINVAL, "%s: null pointer", fn);
  for (const void* p : {(const void*)v, (const void*)dv, (const void*)gamma, (const void*)beta, (const void*)v_out, (const void*)h})
    if (!aligned16(p)) return set_error(BCM_EINVAL, "%s: arrays must be 16-byte aligned", fn);
  row_form(D, [&](auto lp, auto nv) {
    constexpr int LP = decltype(lp)::value, NV = decltype(nv)::value;
    hipLaunchKernelGGL((k_residual_norm_fwd<LP, NV>), dim3((unsigned)((rows + 256 / LP - 1) / (256 / LP))), dim3(256), 0, hs(stream), v, dv,
                       alpha, gamma, beta, rows, (int)D, eps, v_out, h, mean, rstd);
  });
  return check_launch(fn);
}

int64_t bcm_residual_norm_workspace_bytes(int64_t rows, int64_t D) {
  return rows < 1 || D < 1 ? 0 : row_workgroups(rows, D) * 2 * D * (int64_t)sizeof(float);
}

int bcm_residual_norm_bwd(const float* gh, const float* gv, const float* v_out, float alpha, const float* gamma,
                          const float* mean, const float* rstd, int64_t rows, int64_t D, float* d_core, float* d_v,
                          float* d_gamma, float* d_beta, void* workspace, int64_t workspace_bytes,
                          bcm_stream_t stream) {
  const char* fn = "bcm_residual_norm_bwd";
  if (int rc = row_check(fn, rows, D)) return rc;
  if (!d_gamma || !d_beta) return set_error(BCM_EINVAL, "%s: null pointer", fn);
  const int64_t wgs = rows ? row_workgroups(rows, D) : 0;
  if (rows && (!gh || !v_out || !gamma || !mean || !rstd || !d_core || !workspace))
    return set_error(BCM_EINVAL, "%s: null pointer", fn);
  if (workspace_bytes < wgs * 2 * D * (int64_t)sizeof(float)) return set_error(BCM_EINVAL, "%s: workspace too small", fn);
  for (const void* p : {(const void*)gh, (const void*)gv, (const void*)v_out, (const void*)gamma, (const void*)d_core, (const void*)d_v})
    if (!aligned16(p)) return set_error(BCM_EINVAL, "%s: arrays must be 16-byte aligned", fn);
  float* part = static_cast<float*>(workspace);
  if (rows)
    row_form(D, [&](auto lp, auto nv) {
      constexpr int LP = decltype(lp)::value, NV = decltype(nv)::value;
      hipLaunchKernelGGL((k_residual_norm_bwd<LP, NV>), dim3((unsigned)wgs), dim3(256), 0, hs(stream), gh, gv, v_out,
                         alpha, gamma, mean, rstd, rows, (int)D, d_core, d_v, part);
    });
  int rc = check_launch(fn);
  if (rc) return rc;
  hipLaunchKernelGGL(k_column_reduce, dim3((unsigned)((2 * D + 15) / 16)), dim3(1024), 0, hs(stream), part, (int)wgs,
                     (int)(2 * D), (int)D, d_gamma, d_beta);
  return check_launch(fn);
}

int64_t bcm_column_sums_workspace_bytes(int64_t rows, int64_t D) {
  return rows < 1 || D < 1 ? 0 : row_workgroups(rows, D) * D * (int64_t)sizeof(float);
}

// d_logits null: the column sums of x alone (logits null then)
static int column_sums_of(const char* fn, const float* x, const float* logits, int64_t rows, int64_t D,
                          float* d_logits, float* out, void* workspace, int64_t workspace_bytes,
                          bcm_stream_t stream) {
  if (int rc = row_check(fn, rows, D)) return rc;
  const int64_t wgs = rows ? row_workgroups(rows, D) : 0;
  if (!out || (rows && (!x || !workspace))) return set_error(BCM_EINVAL, "%s: null pointer", fn);
  if (workspace_bytes < wgs * D * (int64_t)sizeof(float)) return set_error(BCM_EINVAL, "%s: workspace too small", fn);
  for (const void* p : {(const void*)x, (const void*)logits, (const void*)d_logits})
    if (!aligned16(p)) return set_error(BCM_EINVAL, "%s: arrays must be 16-byte aligned", fn);
  float* part = static_cast<float*>(workspace);
  if (rows)
    row_form(D, [&](auto lp, auto nv) {
      constexpr int LP = decltype(lp)::value, NV = decltype(nv)::value;
      const dim3 grid((unsigned)wgs), block(256);
      if (d_logits)
        hipLaunchKernelGGL((k_spike_head_bwd<LP, NV>), grid, block, 0, hs(stream), x, logits, rows, (int)D, d_logits, part);
      else hipLaunchKernelGGL((k_column_sums<LP, NV>), grid, block, 0, hs(stream), x, rows, (int)D, part);
    });
  int rc = check_launch(fn);
  if (rc) return rc;
  hipLaunchKernelGGL(k_column_reduce, dim3((unsigned)((D + 15) / 16)), dim3(1024), 0, hs(stream), part, (int)wgs, (int)D,
                     (int)D, out, out);
  return check_launch(fn);
}

int bcm_column_sums(const float* x, int64_t rows, int64_t D, float* out, void* workspace, int64_t workspace_bytes,
                    bcm_stream_t stream) {
  return column_sums_of("bcm_column_sums", x, nullptr, rows, D, nullptr, out, workspace, workspace_bytes, stream);
}

int bcm_spike_head_bwd(const float* ds, const float* logits, int64_t rows, int64_t D, float* d_logits, float* d_bias,
                       void* workspace, int64_t workspace_bytes, bcm_stream_t stream) {
  const char* fn = "bcm_spike_head_bwd";
  if (rows > 0 && (!logits || !d_logits)) return set_error(BCM_EINVAL, "%s: null pointer", fn);
  return column_sums_of(fn, ds, logits, rows, D, d_logits, d_bias, workspace, workspace_bytes, stream);
}

}  // extern "C"
