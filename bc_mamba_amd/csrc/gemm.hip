// fp32 matrix products of the block's token projections (in_proj, out_proj,
// prob_head: e_model.py:419-506) and of their gradients, on the fp16 matrix
// cores with fp32 results.
//
// Method: each operand value x is scaled by a power of two of its own row
// (the row of A, the column of the result for B) and written as two fp16
// values, hi = fp16(x s) and lo = fp16(x s - hi), 22 significant bits and
// more; C = A B is then hi hi + hi lo + lo hi, accumulated in fp32 by
// v_mfma_f32_32x32x16_f16, and the result is scaled back (Ootomo and Yokota,
// "Recovering single precision accuracy from Tensor Cores while surpassing
// the FP32 theoretical peak performance", 2022). The dropped lo lo term is
// 2^-24 of a product on average, the size of one fp32 rounding; the sums over k
// round less often than a chain of fp32 FMAs does (16 products a step).
//
// Range: the row scale keeps the row's largest |x s| between 2^9 and the
// largest fp16 value, so a value down to 2^-34 of its row's largest keeps an
// absolute error of 2^-34 of that largest. Scales are found on the way: a
// row's first k-chunk sets it with 2^6 to spare, and where a later chunk
// would overflow, the row's scale and its accumulators are lowered together
// (a rare, workgroup-uniform branch). A tile that meets an infinity is
// recomputed with fp32 FMAs, so infinities and NaN come out as in a plain
// fp32 product.
#include "bcm_common.hpp"

#include <algorithm>
#include <cmath>

namespace bcm {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float gf16v __attribute__((ext_vector_type(16)));

constexpr int kGT = 128;                   // result tile edge
constexpr int kGK = 32;                    // k-chunk
constexpr int kGPlane = kGT * kGK;         // halves of one operand plane in LDS
constexpr int kGDepth = 2;                 // chunks in flight from memory
constexpr float kGMax = 65000.0f;          // largest scaled magnitude
constexpr int kGTop = 10;                  // a scale set anew puts the row's largest below 2^kGTop
constexpr int kGEmpty = 127;               // largest scale exponent, and that of a row with no nonzero value yet

// Operand rows in LDS. Row r of a 64-row half sits in slot 32 (r & 1) + r / 2,
// so the two 32-row MFMA tiles of a wave hold the even and the odd rows: a
// lane's two results of a C row are neighbours (8-byte stores). A slot is
// 32 halves in four 16-byte parts, rotated so that neighbouring slots' reads
// of one part fall on different banks. Part c holds k = 4c..4c+3 and
// 16+4c..16+4c+3 of the chunk (the same order for both operands).
__device__ __forceinline__ int g_slot_row(int s) { return (s & 64) + 2 * (s & 31) + ((s >> 5) & 1); }
__device__ __forceinline__ int g_off(int slot, int part) { return slot * kGK + ((part ^ (slot >> 2)) & 3) * 8; }

__device__ __forceinline__ float g_max3(float m, float a, float b) {
  asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(a), "v"(b));
  return m;
}
// (hi, lo) of a s and b s, packed in pairs: four v_fma_mix (the empty asm
// keeps the compiler from forming b's hi a second time).
__device__ __forceinline__ void g_split2(float a, float b, float s, uint32_t& hi, uint32_t& lo) {
  h2 h = {(_Float16)__builtin_fmaf(a, s, 0.0f), (_Float16)__builtin_fmaf(b, s, 0.0f)};
  asm("" : "+v"(h));
  const h2 l = {(_Float16)__builtin_fmaf(a, s, -(float)h[0]), (_Float16)__builtin_fmaf(b, s, -(float)h[1])};
  hi = __builtin_bit_cast(uint32_t, h);
  lo = __builtin_bit_cast(uint32_t, l);
}
// Exponent that puts a row whose largest magnitude is m below 2^kGTop.
__device__ __forceinline__ int g_exp_of(float m) {
  return m > 0.0f ? min(kGTop - __builtin_amdgcn_frexp_expf(m), kGEmpty) : kGEmpty;
}
__device__ __forceinline__ float g_pow2(int e) { return __builtin_amdgcn_ldexpf(1.0f, e); }

// One operand: 128 rows by 32 k a chunk, staged by 256 threads from global
// memory through registers. KC: k is contiguous (row-major rows); otherwise
// the rows are contiguous (k-major). A thread's values all lie in NR rows.
template <bool KC> struct GOperand {
  static constexpr int NR = KC ? 2 : 4;    // rows of a thread
  static constexpr int NV = 16 / NR;       // values of each
  struct Raw { float x[NR][NV]; };  // one chunk's values on their way
  float sc[NR];
  int ex[NR];
  __amdgpu_buffer_rsrc_t rs;
  uint32_t base[NR], step;
  int kofs, left;
  bool edge;
  int slot[NR];

  __device__ __forceinline__ void init(const float* p, int rows, int K, int64_t ld, int r0) {
    const int tid = threadIdx.x;
    rs = buf_rsrc(p, KC ? ((int64_t)(rows - 1) * ld + K) * 4 : ((int64_t)(K - 1) * ld + rows) * 4);
    if constexpr (KC) {
      kofs = 4 * (tid & 3);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        slot[i] = (tid >> 2) + 64 * i;
        const int r = r0 + g_slot_row(slot[i]);
        base[i] = r < rows ? (uint32_t)((int64_t)r * ld + kofs) * 4u : kBufOOB;
      }
      step = 4u;
    } else {
      const int lane = tid & 63, w = tid >> 6, g = lane >> 3, rq = lane & 7;
      kofs = 16 * (g & 1) + 4 * (g >> 1);
      const int r = r0 + 32 * w + 4 * rq;
#pragma unroll
      for (int j = 0; j < 4; ++j) slot[j] = 64 * (w >> 1) + 32 * (j & 1) + 16 * (w & 1) + 2 * rq + (j >> 1);
      base[0] = r < rows ? (uint32_t)((int64_t)kofs * ld + r) * 4u : kBufOOB;
      step = (uint32_t)ld * 4u;
      left = rows - r;
      edge = r0 + kGT > rows;
    }
  }
  __device__ __forceinline__ u32x4 ld4(uint32_t o) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0));
  }
  __device__ __forceinline__ float ld1(uint32_t o) { return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0)); }
  // Values of chunk k0; past ke (the slice's end) they count as 0. WHOLE: no
  // chunk or row group is cut by an edge (16-byte loads, no branch); else
  // single values where one is.
  template <bool WHOLE> __device__ __forceinline__ void load(Raw& raw, int k0, int ke) {
    auto& x = raw.x;
    const uint32_t past = k0 < ke ? 0u : kBufOOB;  // scalar
    if constexpr (KC) {
      if (WHOLE || k0 + kGK <= ke) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int v = 0; v < 2; ++v) {
            const u32x4 q = ld4((base[i] + (uint32_t)(k0 + 16 * v) * 4u) | past);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[i][4 * v + e] = __uint_as_float(q[e]);
          }
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int v = 0; v < 8; ++v) {
            const int k = k0 + 16 * (v >> 2) + (v & 3);
            x[i][v] = ld1(k + kofs < ke ? base[i] + (uint32_t)k * 4u : kBufOOB);
          }
      }
    } else {
      if (WHOLE || !edge) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const u32x4 q = ld4((base[0] + (uint32_t)(k0 + i) * step) | past);
#pragma unroll
          for (int j = 0; j < 4; ++j) x[j][i] = __uint_as_float(q[j]);
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            x[j][i] = ld1(k0 + kofs + i < ke && j < left ? base[0] + (uint32_t)(k0 + i) * step + 4u * j : kBufOOB);
      }
    }
  }
  static __device__ __forceinline__ float row_max(const Raw& raw, int r) {
    auto& x = raw.x;
    float m = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; v += 2) m = g_max3(m, x[r][v], x[r][v + 1]);
    return m;
  }
  // The row's largest over the lanes that stage it.
  __device__ __forceinline__ float across(float m) {
    if constexpr (KC) {
      m = fmaxf(m, __shfl_xor(m, 1));
      m = fmaxf(m, __shfl_xor(m, 2));
    } else {
      m = fmaxf(m, __shfl_xor(m, 8));
      m = fmaxf(m, __shfl_xor(m, 16));
      m = fmaxf(m, __shfl_xor(m, 32));
    }
    return m;
  }
  __device__ __forceinline__ void first_scale(const Raw& x, int* inf) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const float m = across(row_max(x, r));
      if (m == INFINITY) *inf = 1;
      ex[r] = g_exp_of(m);
      sc[r] = g_pow2(ex[r]);
    }
  }
  // Largest scaled magnitude of the thread's values.
  __device__ __forceinline__ float scaled_max(const Raw& x) {
    float t = 0.0f;
#pragma unroll
    for (int r = 0; r < NR; ++r) t = fmaxf(t, row_max(x, r) * sc[r]);
    return t;
  }
  // Lowers the scale of the rows that would overflow; the change goes to
  // delta (per slot) for the accumulators. All lanes of the wave come here.
  __device__ __forceinline__ void lower(const Raw& x, int* delta, int* inf) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const float m = across(row_max(x, r));
      if (m * sc[r] > kGMax) {
        if (m == INFINITY) *inf = 1;
        const int e = g_exp_of(m);
        delta[slot[r]] = e - ex[r];
        ex[r] = e;
        sc[r] = g_pow2(e);
      }
    }
  }
  // Splits the chunk into LDS: hi plane at p, lo plane kGPlane after it.
  __device__ __forceinline__ void store(const Raw& raw, _Float16* p) {
    auto& x = raw.x;
    if constexpr (KC) {
      const int part = (threadIdx.x & 3);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        u32x4 hi, lo;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          uint32_t h, l;
          g_split2(x[i][2 * v], x[i][2 * v + 1], sc[i], h, l);
          hi[v] = h;
          lo[v] = l;
        }
        _Float16* q = p + g_off(slot[i], part);
        *reinterpret_cast<u32x4*>(q) = hi;
        *reinterpret_cast<u32x4*>(q + kGPlane) = lo;
      }
    } else {
      const int g = (threadIdx.x & 63) >> 3;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        u32x2 hi, lo;
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          uint32_t h, l;
          g_split2(x[j][2 * v], x[j][2 * v + 1], sc[j], h, l);
          hi[v] = h;
          lo[v] = l;
        }
        _Float16* q = p + g_off(slot[j], g >> 1) + 4 * (g & 1);
        *reinterpret_cast<u32x2*>(q) = hi;
        *reinterpret_cast<u32x2*>(q + kGPlane) = lo;
      }
    }
  }
};

struct GemmArgs {
  const float *a, *b, *bias;
  float* c;
  int64_t lda, ldb, ldc, slice_stride;
  int M, N, K, tm, tn, k_slice, n_fast;
};

// Workgroup: one 128 x 128 tile of C over one slice of k. 4 waves, 64 x 64
// each. Two LDS stages: while chunk i is multiplied, chunk i + 1 is split
// into the other stage and later chunks are on their way from memory. With
// two waves on a SIMD the matrix cores, the VALU (the splits) and LDS each
// need about the same time a chunk, so the three are interleaved inside the
// wave: sched_group_barrier puts reads, splits, stores and loads between the
// MFMAs.
template <bool AKC, bool BKC, bool WHOLE>
__global__ __launch_bounds__(256, 2) void k_gemm_f32(const GemmArgs g) {
  __shared__ _Float16 sm[2][4 * kGPlane];  // per stage: A hi, A lo, B hi, B lo
  __shared__ int s_delta[2][2 * kGT];      // per chunk parity: change of each row's scale exponent (A, then B)
  __shared__ int s_flag[2], s_inf;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w & 1, wn = w >> 1;
  const int q = lane & 31, h = lane >> 5;
  const int tiles = g.tm * g.tn;
  const int item = xcd_block(blockIdx.x, gridDim.x);
  const int slice = item / tiles, t = item - slice * tiles;
  const int im = g.n_fast ? t / g.tn : t % g.tm, in = g.n_fast ? t % g.tn : t / g.tm;
  const int m0 = im * kGT, n0 = in * kGT;
  const int kb = slice * g.k_slice, ke = min(g.K, kb + g.k_slice);

  GOperand<AKC> oa;
  GOperand<BKC> ob;
  oa.init(g.a, g.M, g.K, g.lda, m0);
  ob.init(g.b, g.N, g.K, g.ldb, n0);
  typename GOperand<AKC>::Raw xa[kGDepth];
  typename GOperand<BKC>::Raw xb[kGDepth];
#pragma unroll
  for (int i = 0; i < kGDepth; ++i) {
    oa.template load<WHOLE>(xa[i], kb + i * kGK, ke);
    ob.template load<WHOLE>(xb[i], kb + i * kGK, ke);
  }
  for (int i = tid; i < 4 * kGT; i += 256) (&s_delta[0][0])[i] = 0;
  if (tid < 2) s_flag[tid] = 0;
  if (tid == 2) s_inf = 0;
  __syncthreads();
  oa.first_scale(xa[0], &s_inf);
  ob.first_scale(xb[0], &s_inf);
  oa.store(xa[0], sm[0]);
  ob.store(xb[0], sm[0] + 2 * kGPlane);
  oa.template load<WHOLE>(xa[0], kb + kGDepth * kGK, ke);
  ob.template load<WHOLE>(xb[0], kb + kGDepth * kGK, ke);
  __syncthreads();

  gf16v acc[2][2] = {};
  const int qa = (64 * wm + q) * kGK, qb = 2 * kGPlane + (64 * wn + q) * kGK;
  // One chunk: multiply stage ST, split the next chunk (register set NX;
  // past the end it is zeros) into the other stage, send for a later one.
  auto chunk = [&](int k0, auto stc, auto nxc) {
    constexpr int ST = decltype(stc)::value, NX = decltype(nxc)::value;
    if (__builtin_expect(s_flag[ST], 0)) {  // some row's scale was lowered for this chunk: so are its accumulators
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) {
        const int db = s_delta[ST][kGT + 64 * wn + 32 * tb + q];
#pragma unroll
        for (int ta = 0; ta < 2; ++ta)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int da = s_delta[ST][64 * wm + 32 * ta + 8 * (r >> 2) + 4 * h + (r & 3)];
            acc[ta][tb][r] = __builtin_amdgcn_ldexpf(acc[ta][tb][r], da + db);
          }
      }
      __syncthreads();  // every wave has read the changes
      s_delta[ST][tid] = 0;
      if (tid == 0) s_flag[ST] = 0;
    }
    if (__builtin_expect(__any(fmaxf(oa.scaled_max(xa[NX]), ob.scaled_max(xb[NX])) > kGMax), 0)) {
      oa.lower(xa[NX], s_delta[ST ^ 1], &s_inf);
      ob.lower(xb[NX], s_delta[ST ^ 1] + kGT, &s_inf);
      if (lane == 0) s_flag[ST ^ 1] = 1;
    }
    const _Float16* pa = sm[ST] + qa;
    const _Float16* pb = sm[ST] + qb;
    h8 ah[2][2], al[2][2], bh[2][2], bl[2][2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const int o = ((2 * kk + h) ^ (q >> 2)) & 3;  // slots 32 apart rotate alike
#pragma unroll
      for (int t2 = 0; t2 < 2; ++t2) {
        al[kk][t2] = *reinterpret_cast<const h8*>(pa + 32 * kGK * t2 + o * 8 + kGPlane);
        bh[kk][t2] = *reinterpret_cast<const h8*>(pb + 32 * kGK * t2 + o * 8);
        ah[kk][t2] = *reinterpret_cast<const h8*>(pa + 32 * kGK * t2 + o * 8);
        bl[kk][t2] = *reinterpret_cast<const h8*>(pb + 32 * kGK * t2 + o * 8 + kGPlane);
      }
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int ta = 0; ta < 2; ++ta)
#pragma unroll
          for (int tb = 0; tb < 2; ++tb)
            acc[ta][tb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(p == 0 ? al[kk][ta] : ah[kk][ta],
                                                                 p == 1 ? bl[kk][tb] : bh[kk][tb], acc[ta][tb], 0, 0, 0);
    oa.store(xa[NX], sm[ST ^ 1]);
    ob.store(xb[NX], sm[ST ^ 1] + 2 * kGPlane);
    oa.template load<WHOLE>(xa[NX], k0 + (1 + kGDepth) * kGK, ke);
    ob.template load<WHOLE>(xb[NX], k0 + (1 + kGDepth) * kGK, ke);
    __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);  // the first half's operands
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // VALU
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // memory read
    }
    __syncthreads();
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  for (int k0 = kb; k0 < ke; k0 += 2 * kGK) {
    chunk(k0, I0{}, std::integral_constant<int, 1 % kGDepth>{});
    if (k0 + kGK < ke) chunk(k0 + kGK, I1{}, I0{});
  }
  // the rows' final scale exponents, one writer for each row
  int* s_exp = reinterpret_cast<int*>(&sm[0][0]);
  __syncthreads();  // the last chunk's stores into the stages are done
#pragma unroll
  for (int r = 0; r < GOperand<AKC>::NR; ++r) s_exp[oa.slot[r]] = -oa.ex[r];
#pragma unroll
  for (int r = 0; r < GOperand<BKC>::NR; ++r) s_exp[kGT + ob.slot[r]] = -ob.ex[r];
  __syncthreads();
  const int n = n0 + 64 * wn + 2 * q, mb = m0 + 64 * wm + 8 * h;
  // rows past M are past the buffer's end: their stores are dropped
  const __amdgpu_buffer_rsrc_t rc = buf_rsrc(g.c + slice * g.slice_stride, ((int64_t)(g.M - 1) * g.ldc + g.N) * 4);
  const float b0 = g.bias && n < g.N ? g.bias[n] : 0.0f, b1 = g.bias && n + 1 < g.N ? g.bias[n + 1] : 0.0f;
  const int eb0 = s_exp[kGT + 64 * wn + q], eb1 = s_exp[kGT + 64 * wn + 32 + q];
  if (__builtin_expect(s_inf, 0)) {  // an infinity among the operands: the tile again with plain FMAs
    for (int ta = 0; ta < 2; ++ta)
      for (int r = 0; r < 16; ++r) {
        const int m = mb + 16 * (r >> 2) + 2 * (r & 3) + ta;
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
      const int ea = s_exp[64 * wm + 32 * ta + 8 * (r >> 2) + 4 * h + (r & 3)];
      const float v0 = __builtin_amdgcn_ldexpf(acc[ta][0][r], ea + eb0) + b0;
      const float v1 = __builtin_amdgcn_ldexpf(acc[ta][1][r], ea + eb1) + b1;
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
