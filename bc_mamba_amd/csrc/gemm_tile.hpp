// A 128 x 128 tile of an fp32 matrix product on the fp16 matrix cores, shared by
// the projection products (gemm.hip) and the products fused with the restore
// (restore_proj.hip).
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
// The matrix cores' fp16 sums round downwards, not to nearest: every result would
// be low by about 1e-8 of the results' size, which a later sum over many tokens
// collects (off by 2.2e-6 over 51 200 rows at K = 256, where fp32 products are
// off by 3.1e-7 and these, as follows, by 1.9e-7). So
// odd rows of A and odd columns of the result enter with their sign turned,
// and the results with an odd sum of both are turned back: neighbours are then
// off in opposite directions.
//
// Range: the row scale keeps the row's largest |x s| between 2^9 and the
// largest fp16 value, so a value down to 2^-34 of its row's largest keeps an
// absolute error of 2^-34 of that largest. Scales are found on the way: a
// row's first k-chunk sets it with 2^6 to spare, and where a later chunk
// would overflow, the row's scale and its accumulators are lowered together
// (a rare, workgroup-uniform branch). A tile that meets an infinity is
// recomputed with fp32 FMAs, so infinities and NaN come out as in a plain
// fp32 product.
#pragma once
#include "bcm_common.hpp"

#include <cmath>

namespace bcm {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float gf16v __attribute__((ext_vector_type(16)));

constexpr int kGT = 128;                   // result tile edge
constexpr int kGK = 32;                    // k-chunk
constexpr int kGPlane = kGT * kGK;         // halves of one operand plane in LDS
constexpr int kGDepth = 1;                 // chunks in flight from memory beside the one being split (2: no faster)
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
  // odd rows are taken negative
  __device__ __forceinline__ float sign(int r) const { return (slot[r] >> 5) & 1 ? -1.0f : 1.0f; }
  __device__ __forceinline__ void first_scale(const Raw& x, int* inf) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const float m = across(row_max(x, r));
      if (m == INFINITY) *inf = 1;
      ex[r] = g_exp_of(m);
      sc[r] = sign(r) * g_pow2(ex[r]);
    }
  }
  // Largest scaled magnitude of the thread's values.
  __device__ __forceinline__ float scaled_max(const Raw& x) {
    float t = 0.0f;
#pragma unroll
    for (int r = 0; r < NR; ++r) t = fmaxf(t, row_max(x, r) * fabsf(sc[r]));
    return t;
  }
  // Lowers the scale of the rows that would overflow; the change goes to
  // delta (per slot) for the accumulators. All lanes of the wave come here.
  __device__ __forceinline__ void lower(const Raw& x, int* delta, int* inf) {
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const float m = across(row_max(x, r));
      if (m * fabsf(sc[r]) > kGMax) {
        if (m == INFINITY) *inf = 1;
        const int e = g_exp_of(m);
        delta[slot[r]] = e - ex[r];
        ex[r] = e;
        sc[r] = sign(r) * g_pow2(e);
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

// The workgroup's LDS: two stages of the operands (per stage A hi, A lo, B hi,
// B lo; free again after gemm_tile), per chunk parity the change of each
// row's scale exponent (A, then B), and what the tile leaves for its results:
// the exponent that scales each slot's row back, and whether an operand held
// an infinity (the tile is then to be computed again, with plain FMAs).
struct GemmLds {
  _Float16 sm[2][4 * kGPlane];
  int delta[2][2 * kGT];
  int exp[2 * kGT];
  int flag[2], inf;
};

// Place of register r of accumulator tile ta / tb of this thread in the
// 128 x 128 tile: row = gemm_row(w, ta, r), columns gemm_col(w) + tb.
__device__ __forceinline__ int gemm_slot_a(int w, int ta, int r) {
  return 64 * (w & 1) + 32 * ta + 8 * (r >> 2) + 4 * (lane_id() >> 5) + (r & 3);
}
__device__ __forceinline__ int gemm_row(int w, int ta, int r) {
  return 64 * (w & 1) + 2 * (8 * (r >> 2) + 4 * (lane_id() >> 5) + (r & 3)) + ta;
}
// A result's value: its accumulator, turned back and scaled back.
__device__ __forceinline__ float gemm_value(float acc, int ta, int tb, int e) {
  return __builtin_amdgcn_ldexpf((ta ^ tb) & 1 ? -acc : acc, e);
}
__device__ __forceinline__ int gemm_slot_b(int w, int tb) { return kGT + 64 * (w >> 1) + 32 * tb + (lane_id() & 31); }
__device__ __forceinline__ int gemm_col(int w) { return 64 * (w >> 1) + 2 * (lane_id() & 31); }

// acc (zero on entry) = the scaled product of rows m0 .. m0 + 127 of A and n0 ..
// n0 + 127 of B over k = kb .. ke - 1. The value of a result is gemm_value(acc, ta,
// tb, s.exp[slot of the row] + s.exp[slot of the column]). 256 threads,
// 4 waves, 64 x 64 each. While chunk i is multiplied, chunk i + 1 is split into
// the other LDS stage and later chunks are on their way from memory. With
// two waves on a SIMD the matrix cores, the VALU (the splits) and LDS each
// need about the same time a chunk, so the three are interleaved inside the
// wave: sched_group_barrier puts reads, splits, stores and loads between the
// MFMAs.
template <bool AKC, bool BKC, bool WHOLE>
__device__ __forceinline__ void gemm_tile(const float* pa_, int rows_a, int64_t lda, const float* pb_, int rows_b,
                                          int64_t ldb, int K, int m0, int n0, int kb, int ke, GemmLds& s,
                                          gf16v (&acc)[2][2]) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w & 1, wn = w >> 1;
  const int q = lane & 31, h = lane >> 5;
  GOperand<AKC> oa;
  GOperand<BKC> ob;
  oa.init(pa_, rows_a, K, lda, m0);
  ob.init(pb_, rows_b, K, ldb, n0);
  typename GOperand<AKC>::Raw xa[kGDepth];
  typename GOperand<BKC>::Raw xb[kGDepth];
#pragma unroll
  for (int i = 0; i < kGDepth; ++i) {
    oa.template load<WHOLE>(xa[i], kb + i * kGK, ke);
    ob.template load<WHOLE>(xb[i], kb + i * kGK, ke);
  }
  for (int i = tid; i < 4 * kGT; i += 256) (&s.delta[0][0])[i] = 0;
  if (tid < 2) s.flag[tid] = 0;
  if (tid == 2) s.inf = 0;
  __syncthreads();
  oa.first_scale(xa[0], &s.inf);
  ob.first_scale(xb[0], &s.inf);
  oa.store(xa[0], s.sm[0]);
  ob.store(xb[0], s.sm[0] + 2 * kGPlane);
  oa.template load<WHOLE>(xa[0], kb + kGDepth * kGK, ke);
  ob.template load<WHOLE>(xb[0], kb + kGDepth * kGK, ke);
  __syncthreads();

  const int qa = (64 * wm + q) * kGK, qb = 2 * kGPlane + (64 * wn + q) * kGK;
  // One chunk: multiply stage ST, split the next chunk (register set NX;
  // past the end it is zeros) into the other stage, send for a later one.
  auto chunk = [&](int k0, auto stc, auto nxc) {
    constexpr int ST = decltype(stc)::value, NX = decltype(nxc)::value;
    if (__builtin_expect(s.flag[ST], 0)) {  // some row's scale was lowered for this chunk: so are its accumulators
#pragma unroll
      for (int tb = 0; tb < 2; ++tb) {
        const int db = s.delta[ST][kGT + 64 * wn + 32 * tb + q];
#pragma unroll
        for (int ta = 0; ta < 2; ++ta)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int da = s.delta[ST][64 * wm + 32 * ta + 8 * (r >> 2) + 4 * h + (r & 3)];
            acc[ta][tb][r] = __builtin_amdgcn_ldexpf(acc[ta][tb][r], da + db);
          }
      }
      __syncthreads();  // every wave has read the changes
      s.delta[ST][tid] = 0;
      if (tid == 0) s.flag[ST] = 0;
    }
    if (__builtin_expect(__any(fmaxf(oa.scaled_max(xa[NX]), ob.scaled_max(xb[NX])) > kGMax), 0)) {
      oa.lower(xa[NX], s.delta[ST ^ 1], &s.inf);
      ob.lower(xb[NX], s.delta[ST ^ 1] + kGT, &s.inf);
      if (lane == 0) s.flag[ST ^ 1] = 1;
    }
    const _Float16* pa = s.sm[ST] + qa;
    const _Float16* pb = s.sm[ST] + qb;
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
    oa.store(xa[NX], s.sm[ST ^ 1]);
    ob.store(xb[NX], s.sm[ST ^ 1] + 2 * kGPlane);
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
#pragma unroll
  for (int r = 0; r < GOperand<AKC>::NR; ++r) s.exp[oa.slot[r]] = -oa.ex[r];  // the lanes of a row write the same
#pragma unroll
  for (int r = 0; r < GOperand<BKC>::NR; ++r) s.exp[kGT + ob.slot[r]] = -ob.ex[r];
  __syncthreads();
}

}  // namespace bcm
