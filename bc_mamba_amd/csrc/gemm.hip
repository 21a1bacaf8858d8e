// fp32 matrix products of the block's token projections (in_proj, out_proj,
// prob_head: e_model.py:419-506) and of their gradients, on the fp16 matrix
// cores with fp32 results.
// The tile and its method are in gemm_tile.hpp. One product of a layer at
// 51 200 tokens, d_model 256, d_inner 512 takes 60-70 us (200-220 TFLOP/s;
// hipBLASLt's fp32 products 102-152 us). Timing copies of it: without the
// memory reads 6 us less, without the splits and LDS stores 10, without the
// MFMAs 15: no one part bounds it; chunks are short (8 or 16 a tile), and the
// first loads and the results of a tile are a good part of its life.
#include "gemm_tile.hpp"

#include <algorithm>

namespace bcm {

struct GemmArgs {
  const float *a, *b, *bias;
  float* c;
  int64_t lda, ldb, ldc, slice_stride;
  int M, N, K, tm, tn, k_slice, n_fast;
};

// Workgroup: one 128 x 128 tile of C over one slice of k.
template <bool AKC, bool BKC, bool WHOLE>
__global__ __launch_bounds__(256, 2) void k_gemm_f32(const GemmArgs g) {
  __shared__ GemmLds s;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles = g.tm * g.tn;
  const int item = xcd_block(blockIdx.x, gridDim.x);
  const int slice = item / tiles, t = item - slice * tiles;
  const int im = g.n_fast ? t / g.tn : t % g.tm, in = g.n_fast ? t % g.tn : t / g.tm;
  const int m0 = im * kGT, n0 = in * kGT;
  const int kb = slice * g.k_slice, ke = min(g.K, kb + g.k_slice);
  gf16v acc[2][2] = {};
  gemm_tile<AKC, BKC, WHOLE>(g.a, g.M, g.lda, g.b, g.N, g.ldb, g.K, m0, n0, kb, ke, s, acc);
  const int n = n0 + gemm_col(w), mb = m0 + gemm_row(w, 0, 0);
  // rows past M are past the buffer's end: their stores are dropped
  const __amdgpu_buffer_rsrc_t rc = buf_rsrc(g.c + slice * g.slice_stride, ((int64_t)(g.M - 1) * g.ldc + g.N) * 4);
  const float b0 = g.bias && n < g.N ? g.bias[n] : 0.0f, b1 = g.bias && n + 1 < g.N ? g.bias[n + 1] : 0.0f;
  const int eb0 = s.exp[gemm_slot_b(w, 0)], eb1 = s.exp[gemm_slot_b(w, 1)];
  if (__builtin_expect(s.inf, 0)) {  // an infinity among the operands: the tile again with plain FMAs
    for (int ta = 0; ta < 2; ++ta)
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + gemm_row(w, ta, r);
        if (m >= g.M) continue;
        for (int tb = 0; tb < 2; ++tb) {
          if (n + tb >= g.N) continue;
          float v = 0.0f;
          for (int k = kb; k < ke; ++k)
            v = fmaf(g.a[AKC ? m * g.lda + k : k * g.lda + m], g.b[BKC ? (n + tb) * g.ldb + k : k * g.ldb + n + tb], v);
          buf_store_f32(rc, (uint32_t)((int64_t)m * g.ldc + n + tb) * 4u, v + (tb ? b1 : b0));
        }
      }
    return;
  }
  const uint32_t o0 = n < g.N ? (uint32_t)((int64_t)mb * g.ldc + n) * 4u : kBufOOB;
  const bool pair = n + 1 < g.N;
#pragma unroll
  for (int ta = 0; ta < 2; ++ta)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int ea = s.exp[gemm_slot_a(w, ta, r)];
      const float v0 = gemm_value(acc[ta][0][r], ta, 0, ea + eb0) + b0;
      const float v1 = gemm_value(acc[ta][1][r], ta, 1, ea + eb1) + b1;
      const uint32_t o = o0 + (uint32_t)((int64_t)(16 * (r >> 2) + 2 * (r & 3) + ta) * g.ldc) * 4u;
      if (pair)
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(v0), __float_as_uint(v1)}, rc, o, 0, 0);
      else
        buf_store_f32(rc, o, v0);
    }
}

// C = the slices' partial products, summed in a fixed order: a workgroup
// takes 64 groups of 4 results, wave w the w-th quarter of the slices (up to
// 8 loads in flight), and the quarters are added in order (one thread per
// result with all slices in a row took 13 us for 64 slices of 512 x 256).
__global__ __launch_bounds__(256) void k_gemm_sum(const float* __restrict__ part, int64_t stride, int slices, int64_t count,
                                                  int N, int64_t ldc, float* __restrict__ c) {
  __shared__ float s_q[4][256];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t i = ((int64_t)blockIdx.x * 64 + lane) * 4;
  const int per = (slices + 3) / 4, s0 = w * per, s1 = min(slices, s0 + per);
  float v[4] = {};
  if (i + 4 <= count) {
    for (int s = s0; s < s1; s += 8) {
      float4 p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) __builtin_memcpy(&p[j], part + (int64_t)min(s + j, s1 - 1) * stride + i, 16);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool in = s + j < s1;
        v[0] += in ? p[j].x : 0.0f;
        v[1] += in ? p[j].y : 0.0f;
        v[2] += in ? p[j].z : 0.0f;
        v[3] += in ? p[j].w : 0.0f;
      }
    }
  } else {
    for (int e = 0; e < 4; ++e)
      for (int s = s0; s < s1 && i + e < count; ++s) v[e] += part[s * stride + i + e];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) s_q[w][4 * lane + e] = v[e];
  __syncthreads();
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r < count)
    c[r / N * ldc + r % N] = ((s_q[0][threadIdx.x] + s_q[1][threadIdx.x]) + s_q[2][threadIdx.x]) + s_q[3][threadIdx.x];
}

// Slices of k: enough workgroups for two on every CU, at least 8 chunks each.
static int gemm_slices(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + kGT - 1) / kGT) * ((N + kGT - 1) / kGT), want = 2 * (int64_t)device_cus();
  if (tiles * 2 > want) return 1;
  const int64_t s = std::min((want + tiles - 1) / tiles, K / (8 * kGK));
  return (int)std::max<int64_t>(1, s);
}

}  // namespace bcm

using namespace bcm;

extern "C" {

int64_t bcm_gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M < 1 || N < 1 || K < 1) return 0;
  const int s = gemm_slices(M, N, K);
  return s > 1 ? 4 * s * M * N : 0;
}

int bcm_gemm_f32(const float* a, int a_k_contiguous, int64_t lda, const float* b, int b_k_contiguous, int64_t ldb,
                 const float* bias, int64_t M, int64_t N, int64_t K, float* c, int64_t ldc, void* workspace,
                 int64_t workspace_bytes, bcm_stream_t stream) {
  const char* fn = "bcm_gemm_f32";
  if (M < 0 || N < 0 || K < 1) return set_error(BCM_EINVAL, "%s: invalid sizes", fn);
  if (M == 0 || N == 0) return BCM_OK;
  if (!a || !b || !c) return set_error(BCM_EINVAL, "%s: null pointer", fn);
  if (lda < (a_k_contiguous ? K : M) || ldb < (b_k_contiguous ? K : N) || ldc < N)
    return set_error(BCM_EINVAL, "%s: a leading dimension is below its row length", fn);
  // 32-bit buffer offsets (past the last chunk a load runs on by at most one chunk's rows)
  const int64_t lim = INT32_MAX;
  if (((a_k_contiguous ? M : K) + kGK) * lda * 4 > lim || ((b_k_contiguous ? N : K) + kGK) * ldb * 4 > lim ||
      (M + kGT) * ldc * 4 > lim)
    return set_error(BCM_EINVAL, "%s: problem too large", fn);
  if (!a_k_contiguous && b_k_contiguous) return set_error(BCM_EINVAL, "%s: no form for a k-major A with a row-major B", fn);
  int S = gemm_slices(M, N, K);
  if (bias || (S > 1 && (!workspace || workspace_bytes < 4 * S * M * N))) S = 1;
  GemmArgs g;
  g.a = a, g.b = b, g.bias = bias;
  g.lda = lda, g.ldb = ldb, g.M = (int)M, g.N = (int)N, g.K = (int)K;
  g.tm = (int)((M + kGT - 1) / kGT), g.tn = (int)((N + kGT - 1) / kGT);
  g.n_fast = g.tn <= g.tm;  // the tiles that share the longer operand's rows run side by side
  const int64_t chunks = (K + kGK - 1) / kGK, per = (chunks + S - 1) / S;
  S = (int)((chunks + per - 1) / per);
  g.k_slice = (int)per * kGK;
  g.c = S > 1 ? static_cast<float*>(workspace) : c;
  g.ldc = S > 1 ? N : ldc;
  g.slice_stride = S > 1 ? M * N : 0;
  const int64_t items = (int64_t)g.tm * g.tn * S;
  if (items > INT32_MAX / 2) return set_error(BCM_EINVAL, "%s: problem too large", fn);
  const dim3 grid((unsigned)items);
  const hipStream_t st = hs(stream);
  // whole 16-byte groups: k-contiguous operands in k, row-contiguous ones in their rows
  const bool whole = (!(a_k_contiguous || b_k_contiguous) || K % kGK == 0) && (a_k_contiguous || M % 4 == 0) &&
                     (b_k_contiguous || N % 4 == 0);
  auto go = [&](auto akc, auto bkc, auto wh) {
    hipLaunchKernelGGL((k_gemm_f32<decltype(akc)::value, decltype(bkc)::value, decltype(wh)::value>), grid, dim3(256), 0,
                       st, g);
  };
  using Y = std::true_type;
  using F = std::false_type;
  if (a_k_contiguous && b_k_contiguous) whole ? go(Y{}, Y{}, Y{}) : go(Y{}, Y{}, F{});
  else if (a_k_contiguous) whole ? go(Y{}, F{}, Y{}) : go(Y{}, F{}, F{});
  else whole ? go(F{}, F{}, Y{}) : go(F{}, F{}, F{});
  int rc = check_launch(fn);
  if (rc || S == 1) return rc;
  hipLaunchKernelGGL(k_gemm_sum, dim3((unsigned)((M * N + 255) / 256)), dim3(256), 0, st, static_cast<const float*>(workspace),
                     M * N, S, M * N, (int)N, ldc, c);
  return check_launch(fn);
}

}  // extern "C"
