// Stage 2b: flat per-channel selective scan whose B and C are operands of
// their own instead of u·W_B / u·W_C: the legacy [dstate, E] (per event) or
// [dstate, dim] (per model channel) layout and the tiled
// [n_tiles, dstate, T] layout of fwd_flat_ch / bwd_flat_ch.
//
// Reference behaviour: selective_scan.cpp:760-776, 840-848 (layouts and
// checks), selective_scan_fwd_kernel.cuh:566-598 (B/C addressing: tiled
// B[tile_offsets[ch] + chunk, s, i], legacy B[s, ev]), :640-686 (h_i =
// a_i h_{i-1} + B_i Δ_i u_i, y_i = D u_i + Σ_s C_i h_i),
// selective_scan_bwd_kernel.cuh:902-1044 (dh recurrence, per-event dB / dC),
// :1087-1112 (constant B / C sums), selective_scan.cpp:1085-1090 (dB / dC
// mirror the B / C layout).
//
// MI355X design: one workgroup per model channel d (its channels are b·dim + d,
// so dA, ddt, dD and the constant-B/C sums reduce in LDS in a fixed order: no
// atomics, deterministic). A channel runs in passes of 128 events: 16 lanes
// (one DPP row) × 8 consecutive events per lane, four channels a wave. Per
// pass and state a lane folds its 8 items, the row combines the folds with
// the DPP scan of scan_group.hpp, and a second register pass produces the
// states; (decay product, h) and the backward's a·dh carry to the next pass
// through LDS. The backward reads the forward states from a workspace
// [dstate, E] that a forward pass over the same inputs writes first.
//
// A channel is a chain of passes × states, and each link waits on its B and C
// from memory. Two things shorten it: the waves a workgroup has to spare (8,
// less one per four channels) take a share of the states each, their sums
// over the states meeting in LDS once a pass, and every link's operands are
// sent for one link ahead, as 16-byte loads. 153 000 events of 768 channels,
// dstate 16, fp32 with z: forward 94 -> 37 us, backward 159 -> 80 us
// (16 forward waves of 2 states each: 44; without the events one pass ahead: 42
// and 90).
#include "bcm_common.hpp"
#include "scan_group.hpp"

#include <algorithm>
#include <climits>

namespace bcm {

namespace {
constexpr int kVG = 16;              // lanes per channel group
constexpr int kVR = 8;               // consecutive events per lane
constexpr int kVPass = kVG * kVR;    // events per pass
constexpr int kVWaves = 8;           // most waves of a workgroup
constexpr int kVThreads = kVWaves * kWave;
constexpr int kXChunk = 2048;        // events per saved-state chunk (selective_scan.cpp:795)
constexpr float kLog2eV = 1.4426950408889634f;
static_assert(kXChunk % kVPass == 0, "passes must tile the saved-state chunks");

// Shape of a workgroup: nq waves side by side over the channels (four each),
// ns waves behind one another over the states (wave w: channels w % nq,
// states w / nq, w / nq + ns, ...).
struct VarShape {
  int nq, ns;
  int waves() const { return nq * ns; }
  int slots() const { return nq * (kWave / kVG); }
  // floats of LDS: A log2e, A, constant B, constant C; per slot the carries
  // and (backward) the gradient accumulators; two stages of the waves'
  // partial sums over their states
  int64_t bytes(int N, bool bwd) const {
    const int64_t part = ns > 1 ? 2ll * waves() * kWave * kVR * (bwd ? 2 : 1) : 0;
    return 4ll * (4ll * N + (int64_t)slots() * (bwd ? N + 3 * N + 3 : 2 * N) + part);
  }
};

// One operand's values for the 8 items of a lane, for one state: element
// base + s * sstride + r. vec: the whole group of 8 lies in the operand's
// memory (16-byte loads; the values of items past the channel's end are
// not used); otherwise item by item.
struct VarOperand {
  const float* p;
  int64_t base;
  bool vec, on;

  // per_event: one value per event; otherwise the operand has no such values
  __device__ __forceinline__ void at(const float* ptr, bool per_event, const bcm_scan_bc& bc, bool tiled, int64_t e_first,
                                     int pos, int n, int64_t tile0, int N, int64_t E) {
    p = ptr;
    on = per_event && pos < n;
    if (!per_event) return;
    if (!tiled) {
      base = e_first;
      vec = __all(!on || e_first + kVR <= E);
    } else {
      const int T = bc.tile_chunk_size;
      const int64_t tile = tile0 + pos / T;
      base = tile * N * (int64_t)T + pos % T;
      vec = __all(!on || (T % kVR == 0 && tile >= 0 && tile < bc.n_tiles));
    }
  }
  // where vec is false: the offset of item r, or -1
  static __device__ __forceinline__ int64_t item(int r, const bcm_scan_bc& bc, bool tiled, int64_t e_first, int pos, int n,
                                                 int64_t tile0, int N) {
    pos = opaque(pos);  // worked out where it is used: offsets of 8 items for each operand would not fit the registers
    if (pos + r >= n) return -1;
    if (!tiled) return opaque(e_first) + r;
    const int T = bc.tile_chunk_size;
    const int64_t t = tile0 + (pos + r) / T;
    return t >= 0 && t < bc.n_tiles ? t * N * (int64_t)T + (pos + r) % T : -1;
  }
  template <typename F> __device__ __forceinline__ void load(float (&v)[kVR], int64_t so, F&& it) const {
#pragma unroll
    for (int r = 0; r < kVR; ++r) v[r] = 0.0f;
    if (vec) {
      if (on) __builtin_memcpy(v, p + so + base, sizeof(v));
    } else {
#pragma unroll
      for (int r = 0; r < kVR; ++r) {
        const int64_t o = on ? it(r) : -1;
        if (o >= 0) v[r] = p[so + o];
      }
    }
  }
  template <typename F> __device__ __forceinline__ void store(const float (&v)[kVR], int64_t so, int items, F&& it) const {
    float* q = const_cast<float*>(p) + so;
    if (vec && items >= kVR) {
      __builtin_memcpy(q + base, v, sizeof(v));
    } else {
#pragma unroll
      for (int r = 0; r < kVR; ++r) {
        const int64_t o = r < items ? it(r) : -1;
        if (o >= 0) q[o] = v[r];
      }
    }
  }
};

// The raw values of a lane's 8 events of one pass from one stream (on: the
// lane has events; vec: 16-byte loads, all 8 lie in the stream; items past the
// channel's end are not used).
template <typename T> struct VarEvents {
  T v[kVR];
  __device__ __forceinline__ void load(const T* p, int64_t e, bool on, bool vec, int64_t E) {
    if (vec) {
      if (on) __builtin_memcpy(v, p + e, sizeof(v));
    } else {
#pragma unroll
      for (int r = 0; r < kVR; ++r) v[r] = p[max((int64_t)0, min(e + r, E - 1))];
    }
  }
};

// Most passes of the workgroup's channels (their waves keep step at the
// partial sums).
__device__ __forceinline__ int var_passes(int np, int ns, int* s_np) {
  const int npw = wave_max_dpp(np);
  if (ns == 1) return npw;
  __syncthreads();
  if (threadIdx.x == 0) *s_np = 0;
  __syncthreads();
  if (lane_id() == 0) atomicMax(s_np, npw);
  __syncthreads();
  return *s_np;
}

}  // namespace

template <typename T, bool HAS_Z, bool VB, bool VC>
__global__ __launch_bounds__(kVThreads) void k_scan_var_fwd(const bcm_scan_args a, const bcm_scan_bc bc, int nq, int ns,
                                                            float* __restrict__ hws) {
  using Ops = Grp<kVG>;
  const int N = a.dstate;
  const int d = blockIdx.x;
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int grp = lane / kVG, j = lane % kVG;
  const int wq = wave % nq, ws = wave / nq;
  const int nslots = nq * (kWave / kVG);
  const int slot = wq * (kWave / kVG) + grp;
  const int nthr = nq * ns * kWave;
  const bool tiled = bc.layout == BCM_BC_TILED;

  extern __shared__ float smem[];
  __shared__ int s_np;
  float* sAl = smem;
  float* sB = sAl + N;  // constant B / C column of d
  float* sC = sB + N;
  float* carry = sC + 2 * N + slot * 2 * N;   // [P(N), h(N)] at the end of the previous pass
  float* part = sC + 2 * N + nslots * 2 * N;  // [2][waves][8][64] partial y

  for (int s = threadIdx.x; s < N; s += nthr) {
    sAl[s] = a.A[(int64_t)d * N + s] * kLog2eV;
    sB[s] = VB ? 0.0f : bc.B[(int64_t)s * bc.b_row_stride + d];
    sC[s] = VC ? 0.0f : bc.C[(int64_t)s * bc.c_row_stride + d];
  }
  __syncthreads();

  const float dti = a.dt_idle[d], dta = a.dt_active[d];
  const float Dv = a.D ? a.D[d] : 0.0f;
  const int NC = a.n_channels, dim = a.dim, nck = a.n_chunks;
  const int n_per_d = d < NC ? (NC - d + dim - 1) / dim : 0;
  const int64_t E = a.n_events;
  const T* __restrict__ u = static_cast<const T*>(a.u);
  const T* __restrict__ z = static_cast<const T*>(a.z);
  T* __restrict__ out = static_cast<T*>(a.out);
  T* __restrict__ out_z = static_cast<T*>(a.out_z);

  for (int b0 = 0; b0 < n_per_d; b0 += nslots) {
    const int b = b0 + slot;
    const bool act = b < n_per_d;
    const int64_t ch = (int64_t)d + (int64_t)b * dim;
    const int e0 = act ? a.cu_seqlens[ch] : 0;
    // events stay inside [0, E) whatever cu_seqlens holds
    const int n = (act && e0 >= 0) ? (int)max((int64_t)0, min((int64_t)a.cu_seqlens[ch + 1], E) - e0) : 0;
    const int np = (n + kVPass - 1) / kVPass;
    const int npw = var_passes(np, ns, &s_np);
    const int64_t tile0 = (tiled && act) ? (int64_t)bc.tile_offsets[ch] : 0;
    VarOperand ob, oc;
    float bn[kVR], cn[kVR];  // the next link's B and C
    int ppos = 0;      // the lane's first event of the pass that is fetched for
    auto operands = [&](int p) {
      ppos = p * kVPass + j * kVR;
      ob.at(bc.B, VB, bc, tiled, (int64_t)e0 + ppos, ppos, n, tile0, N, E);
      oc.at(bc.C, VC, bc, tiled, (int64_t)e0 + ppos, ppos, n, tile0, N, E);
    };
    auto item = [&](int r) { return VarOperand::item(r, bc, tiled, (int64_t)e0 + ppos, ppos, n, tile0, N); };
    auto fetch = [&](int s) {
      if (VB) ob.load(bn, s * (tiled ? (int64_t)bc.tile_chunk_size : bc.b_row_stride), item);
      if (VC) oc.load(cn, s * (tiled ? (int64_t)bc.tile_chunk_size : bc.c_row_stride), item);
    };
    // the next pass's u, k and z, on their way like the operands
    VarEvents<T> un, zn;
    VarEvents<int32_t> kn;
    auto events = [&](int p) {
      const int64_t e = (int64_t)e0 + p * kVPass + j * kVR;
      const bool on = p * kVPass + j * kVR < n, vec = __all(!on || e + kVR <= E);
      un.load(u, e, on, vec, E);
      kn.load(a.k, e, on, vec, E);
      if (HAS_Z && out) zn.load(z, e, on, vec, E);
    };
    operands(0);
    if (npw > 0) {
      events(0);
      if (ws < N) fetch(ws);
    }
    for (int p = 0; p < npw; ++p) {
      const int pos0 = p * kVPass + j * kVR;
      const int64_t eb = (int64_t)e0 + pos0;
      const int items = max(0, min(kVR, n - pos0));
      float dl[kVR], dlu[kVR], y[kVR], zv[kVR];
#pragma unroll
      for (int r = 0; r < kVR; ++r) {
        const float uu = r < items ? to_f(un.v[r]) : 0.0f;
        dl[r] = r < items ? fmaf(dti, (float)(kn.v[r] - 1), dta) : 0.0f;
        dlu[r] = dl[r] * uu;
        y[r] = ws == 0 ? Dv * uu : 0.0f;
        if (HAS_Z) zv[r] = r < items ? to_f(zn.v[r]) : 0.0f;
      }
      if (p + 1 < npw) events(p + 1);
      // the pass that holds the last event of a saved-state chunk (or of the channel)
      const int pass_end = min(n, (p + 1) * kVPass);
      const bool save_x = a.x && p < np && (pass_end % kXChunk == 0 || pass_end == n);
      const int xc = (pass_end - 1) / kXChunk;
#pragma unroll 1
      for (int s = ws; s < N; s += ns) {
        const float Al = sAl[s];
        float av[kVR], xv[kVR], cv[kVR];
#pragma unroll
        for (int r = 0; r < kVR; ++r) {
          xv[r] = r < items ? (VB ? bn[r] : sB[s]) * dlu[r] : 0.0f;
          cv[r] = VC ? cn[r] : sC[s];
        }
        if (s + ns < N) {  // the next link: the wave's next state, or its first one of the next pass
          fetch(s + ns);
        } else if (p + 1 < npw) {
          operands(p + 1);
          fetch(ws);
        }
        float P = 1.0f, H = 0.0f;
#pragma unroll
        for (int r = 0; r < kVR; ++r) {
          av[r] = r < items ? decay(dl[r] * Al) : 1.0f;
          H = fmaf(av[r], H, xv[r]);
          P *= av[r];
        }
        Ops::scan_up(P, H);
        const float h0 = p > 0 ? carry[N + s] : 0.0f;
        const float P0 = p > 0 ? carry[s] : 1.0f;
        const float hend = fmaf(P, h0, H);
        float h = Ops::prev(hend, h0);
        float hv[kVR];
#pragma unroll
        for (int r = 0; r < kVR; ++r) {
          h = fmaf(av[r], h, xv[r]);
          y[r] = r < items ? fmaf(cv[r], h, y[r]) : 0.0f;
          hv[r] = h;
        }
        if (hws) {
          float* q = hws + (int64_t)s * E + eb;
          if (items == kVR) {
            __builtin_memcpy(q, hv, sizeof(hv));
          } else {
#pragma unroll
            for (int r = 0; r < kVR; ++r)
              if (r < items) q[r] = hv[r];
          }
        }
        if (j == kVG - 1 && p < np) {
          carry[s] = P0 * P;
          carry[N + s] = hend;
          if (save_x && xc < nck) {
            float* xs = a.x + ((ch * nck + xc) * 2 * N);
            xs[2 * s] = P0 * P;
            xs[2 * s + 1] = hend;
          }
        }
      }
      if (out) {
        int r0 = 0, nr = kVR;
        if (ns > 1) {  // the waves' sums over their states: each wave adds up kVR / ns of the lane's items
          float* pp = part + (p & 1) * nq * ns * kWave * kVR;
#pragma unroll
          for (int r = 0; r < kVR; ++r) pp[(wave * kVR + r) * kWave + lane] = y[r];
          __syncthreads();
          nr = kVR / ns;
          r0 = ws * nr;
#pragma unroll
          for (int r = 0; r < kVR; ++r) {
            if (r < r0 || r >= r0 + nr) continue;
            float v = 0.0f;
            for (int q = 0; q < ns; ++q) v += pp[((q * nq + wq) * kVR + r) * kWave + lane];
            y[r] = v;
          }
        }
#pragma unroll
        for (int r = 0; r < kVR; ++r) {
          if (r >= items || r < r0 || r >= r0 + nr) continue;
          out[eb + r] = from_f<T>(y[r]);
          if (HAS_Z) out_z[eb + r] = from_f<T>(y[r] * (zv[r] / (1.0f + __expf(-zv[r]))));
        }
      }
    }
    // saved-state chunks past the channel's end keep the reference's zero state
    if (act && a.x && ws == 0) {
      const int have = (n + kXChunk - 1) / kXChunk;
      for (int c = have; c < nck; ++c)
        for (int s = j; s < 2 * N; s += kVG) a.x[(ch * nck + c) * 2 * N + s] = 0.0f;
    }
  }
}

template <typename T, bool HAS_Z, bool VB, bool VC>
__global__ __launch_bounds__(kVThreads) void k_scan_var_bwd(const bcm_scan_args a, const bcm_scan_bc bc, int nq, int ns,
                                                            const float* __restrict__ hws) {
  using Ops = Grp<kVG>;
  const int N = a.dstate;
  const int d = blockIdx.x;
  const int wave = threadIdx.x / kWave, lane = lane_id();
  const int grp = lane / kVG, j = lane % kVG;
  const int wq = wave % nq, ws = wave / nq;
  const int nslots = nq * (kWave / kVG);
  const int slot = wq * (kWave / kVG) + grp;
  const int nthr = nq * ns * kWave;
  const bool tiled = bc.layout == BCM_BC_TILED;
  const int NA = 3 * N + 3;  // per slot: dA, constant dB, constant dC, ddt_idle, ddt_active, dD

  extern __shared__ float smem[];
  __shared__ int s_np;
  float* sAl = smem;
  float* sA = sAl + N;
  float* sB = sA + N;
  float* sC = sB + N;
  float* cdh = sC + N + slot * N;                       // a·dh of the first event of the later pass
  float* sacc = sC + N + nslots * N;                    // [nslots][NA]
  float* cacc = sacc + slot * NA;
  float* part = sacc + nslots * NA;                     // [2][waves][16][64] partial du, dΔ

  for (int s = threadIdx.x; s < N; s += nthr) {
    const float Av = a.A[(int64_t)d * N + s];
    sA[s] = Av;
    sAl[s] = Av * kLog2eV;
    sB[s] = VB ? 0.0f : bc.B[(int64_t)s * bc.b_row_stride + d];
    sC[s] = VC ? 0.0f : bc.C[(int64_t)s * bc.c_row_stride + d];
  }
  for (int i = threadIdx.x; i < nslots * NA; i += nthr) sacc[i] = 0.0f;
  __syncthreads();

  const float dti = a.dt_idle[d], dta = a.dt_active[d];
  const float Dv = a.D ? a.D[d] : 0.0f;
  const int NC = a.n_channels, dim = a.dim;
  const int n_per_d = d < NC ? (NC - d + dim - 1) / dim : 0;
  const int64_t E = a.n_events;
  const T* __restrict__ u = static_cast<const T*>(a.u);
  const T* __restrict__ dout = static_cast<const T*>(a.dout);
  const T* __restrict__ z = static_cast<const T*>(a.z);
  const T* __restrict__ osv = static_cast<const T*>(a.out_saved);
  T* __restrict__ du_out = static_cast<T*>(a.du);
  T* __restrict__ dz_out = static_cast<T*>(a.dz);
  const int nr = kVR / ns, r0 = ws * nr;  // the items of a lane whose sums over the states this wave completes

  for (int b0 = 0; b0 < n_per_d; b0 += nslots) {
    const int b = b0 + slot;
    const bool act = b < n_per_d;
    const int64_t ch = (int64_t)d + (int64_t)b * dim;
    const int e0 = act ? a.cu_seqlens[ch] : 0;
    // events stay inside [0, E) whatever cu_seqlens holds
    const int n = (act && e0 >= 0) ? (int)max((int64_t)0, min((int64_t)a.cu_seqlens[ch + 1], E) - e0) : 0;
    const int np = (n + kVPass - 1) / kVPass;
    const int npw = var_passes(np, ns, &s_np);
    const int64_t tile0 = (tiled && act) ? (int64_t)bc.tile_offsets[ch] : 0;
    float ddti_l = 0.0f, ddta_l = 0.0f, dD_l = 0.0f;
    VarOperand ob, oc, oh;
    float bn[kVR], cn[kVR], hn[kVR], hp0n;  // the next link's B, C and states
    int ppos = 0;                            // the lane's first event of the pass that is fetched for
    auto operands = [&](int p) {
      ppos = p * kVPass + j * kVR;
      ob.at(bc.B, VB, bc, tiled, (int64_t)e0 + ppos, ppos, n, tile0, N, E);
      oc.at(bc.C, VC, bc, tiled, (int64_t)e0 + ppos, ppos, n, tile0, N, E);
      oh.at(hws, true, bc, false, (int64_t)e0 + ppos, ppos, n, 0, N, E);
    };
    auto item = [&](int r) { return VarOperand::item(r, bc, tiled, (int64_t)e0 + ppos, ppos, n, tile0, N); };
    auto fetch = [&](int s) {
      if (VB) ob.load(bn, s * (tiled ? (int64_t)bc.tile_chunk_size : bc.b_row_stride), item);
      if (VC) oc.load(cn, s * (tiled ? (int64_t)bc.tile_chunk_size : bc.c_row_stride), item);
      oh.load(hn, s * E, [&](int r) { return VarOperand::item(r, bc, false, (int64_t)e0 + ppos, ppos, n, 0, N); });
      // state before the lane's first item
      hp0n = (oh.on && ppos > 0) ? hws[s * E + e0 + ppos - 1] : 0.0f;
    };
    VarEvents<T> un, gn;  // the next pass's u, k and dout
    VarEvents<int32_t> kn;
    auto events = [&](int p) {
      const int64_t e = (int64_t)e0 + p * kVPass + j * kVR;
      const bool on = p * kVPass + j * kVR < n, vec = __all(!on || e + kVR <= E);
      un.load(u, e, on, vec, E);
      kn.load(a.k, e, on, vec, E);
      gn.load(dout, e, on, vec, E);
    };
    if (npw > 0) {
      events(npw - 1);
      operands(npw - 1);
      if (ws < N) fetch(ws);
    }
    for (int p = npw - 1; p >= 0; --p) {
      const int pos0 = p * kVPass + j * kVR;
      const int64_t eb = (int64_t)e0 + pos0;
      const int items = max(0, min(kVR, n - pos0));
      float uu[kVR], dl[kVR], dlu[kVR], dov[kVR], du[kVR], ddl[kVR];
      int km1[kVR];
      VarEvents<T> zz, oo;
      if (HAS_Z) {
        const bool on = items > 0, vec = __all(!on || eb + kVR <= E);
        zz.load(z, eb, on, vec, E);
        oo.load(osv, eb, on, vec, E);
      }
#pragma unroll
      for (int r = 0; r < kVR; ++r) {
        uu[r] = r < items ? to_f(un.v[r]) : 0.0f;
        dov[r] = r < items ? to_f(gn.v[r]) : 0.0f;
        km1[r] = r < items ? kn.v[r] - 1 : 0;
        dl[r] = r < items ? fmaf(dti, (float)km1[r], dta) : 0.0f;
        dlu[r] = dl[r] * uu[r];
        if (HAS_Z && r < items) {  // selective_scan_bwd_kernel.cuh:795-801
          const float zv = to_f(zz.v[r]), ov = to_f(oo.v[r]);
          const float sg = 1.0f / (1.0f + __expf(-zv));
          if (ws == 0) dz_out[eb + r] = from_f<T>(dov[r] * ov * sg * (1.0f + zv * (1.0f - sg)));
          dov[r] *= zv * sg;
        }
        du[r] = ws == 0 ? Dv * dov[r] : 0.0f;
        ddl[r] = 0.0f;
        if (ws == 0) dD_l = fmaf(dov[r], uu[r], dD_l);
      }
      if (p > 0) events(p - 1);
      VarOperand odb, odc;
      odb.at(bc.dB, VB, bc, tiled, eb, pos0, n, tile0, N, E);
      odc.at(bc.dC, VC, bc, tiled, eb, pos0, n, tile0, N, E);
      auto ditem = [&](int r) { return VarOperand::item(r, bc, tiled, eb, pos0, n, tile0, N); };
#pragma unroll 1
      for (int s = ws; s < N; s += ns) {
        const float Al = sAl[s], Av = sA[s];
        float av[kVR], bv[kVR], gv[kVR], hv[kVR];
        const float hp0 = hp0n;
#pragma unroll
        for (int r = 0; r < kVR; ++r) {
          bv[r] = VB ? bn[r] : sB[s];
          gv[r] = r < items ? (VC ? cn[r] : sC[s]) * dov[r] : 0.0f;
          hv[r] = r < items ? hn[r] : 0.0f;
        }
        if (s + ns < N) {  // the next link of the walk
          fetch(s + ns);
        } else if (p > 0) {
          operands(p - 1);
          fetch(ws);
        }
#pragma unroll
        for (int r = 0; r < kVR; ++r) av[r] = r < items ? decay(dl[r] * Al) : 1.0f;
        // dh_i = C_i dout_i + a_{i+1} dh_{i+1}; the last lane of the group
        // takes the carry a·dh of the later pass (and a "next decay" of 1)
        const float anext = Ops::next(av[0], 1.0f);
        const float ec = (p + 1 < np) ? cdh[s] : 0.0f;
        float Q = 1.0f, Ce = 0.0f;
#pragma unroll
        for (int r = kVR - 1; r >= 0; --r) {
          const float al = r == kVR - 1 ? anext : av[r + 1];
          Ce = fmaf(al, Ce, gv[r]);
          Q *= al;
        }
        Ops::scan_down(Q, Ce);
        float dh = Ops::next(fmaf(Q, ec, Ce), ec);
        float dA_l = 0.0f, dBc_l = 0.0f, dCc_l = 0.0f;
        float dbv[kVR], dcv[kVR];
#pragma unroll
        for (int r = kVR - 1; r >= 0; --r) {
          const float al = r == kVR - 1 ? anext : av[r + 1];
          dh = fmaf(al, dh, gv[r]);
          const float hp = r > 0 ? hv[r - 1] : hp0;
          const float t = r < items ? dh * av[r] * hp : 0.0f;
          dA_l = fmaf(t, dl[r], dA_l);
          const float dhb = r < items ? dh * bv[r] : 0.0f;
          ddl[r] = fmaf(dhb, uu[r], fmaf(Av, t, ddl[r]));
          du[r] = fmaf(dhb, dl[r], du[r]);
          dbv[r] = r < items ? dh * dlu[r] : 0.0f;
          dcv[r] = dov[r] * hv[r];
          dBc_l += dbv[r];
          dCc_l += dcv[r];
        }
        if (VB && odb.on) odb.store(dbv, s * (tiled ? (int64_t)bc.tile_chunk_size : bc.db_row_stride), items, ditem);
        if (VC && odc.on) odc.store(dcv, s * (tiled ? (int64_t)bc.tile_chunk_size : bc.dc_row_stride), items, ditem);
        if (j == 0 && p < np) cdh[s] = av[0] * dh;  // dh of the pass's first event
        dA_l = Ops::sum(dA_l);
        if (!VB) dBc_l = Ops::sum(dBc_l);
        if (!VC) dCc_l = Ops::sum(dCc_l);
        if (j == 0 && act) {
          cacc[s] += dA_l;
          if (!VB) cacc[N + s] += dBc_l;
          if (!VC) cacc[2 * N + s] += dCc_l;
        }
      }
      if (ns > 1) {  // the waves' sums over their states
        float* pp = part + (p & 1) * nq * ns * kWave * 2 * kVR;
#pragma unroll
        for (int r = 0; r < kVR; ++r) {
          pp[(wave * 2 * kVR + r) * kWave + lane] = du[r];
          pp[(wave * 2 * kVR + kVR + r) * kWave + lane] = ddl[r];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kVR; ++r) {
          if (r < r0 || r >= r0 + nr) continue;
          float v = 0.0f, w = 0.0f;
          for (int q = 0; q < ns; ++q) {
            v += pp[((q * nq + wq) * 2 * kVR + r) * kWave + lane];
            w += pp[((q * nq + wq) * 2 * kVR + kVR + r) * kWave + lane];
          }
          du[r] = v;
          ddl[r] = w;
        }
      }
#pragma unroll
      for (int r = 0; r < kVR; ++r) {
        if (r >= items || r < r0 || r >= r0 + nr) continue;
        du_out[eb + r] = from_f<T>(du[r]);
        ddti_l = fmaf(ddl[r], (float)km1[r], ddti_l);
        ddta_l += ddl[r];
      }
    }
    ddti_l = Ops::sum(ddti_l);
    ddta_l = Ops::sum(ddta_l);
    dD_l = Ops::sum(dD_l);
    for (int q = 0; q < ns; ++q) {  // one wave of a slot after the other: a fixed order
      if (ns > 1) __syncthreads();
      if (q == ws && j == 0 && act) {
        cacc[3 * N] += ddti_l;
        cacc[3 * N + 1] += ddta_l;
        cacc[3 * N + 2] += dD_l;
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < NA; i += nthr) {
    float v = 0.0f;
    for (int q = 0; q < nslots; ++q) v += sacc[q * NA + i];  // fixed order: deterministic
    if (i < N) {
      a.dA[(int64_t)d * N + i] = v;
    } else if (i < 2 * N) {
      if (!VB) bc.dB[(int64_t)(i - N) * bc.db_row_stride + d] = v;
    } else if (i < 3 * N) {
      if (!VC) bc.dC[(int64_t)(i - 2 * N) * bc.dc_row_stride + d] = v;
    } else if (i == 3 * N) {
      a.ddt_idle[d] = v;
    } else if (i == 3 * N + 1) {
      a.ddt_active[d] = v;
    } else if (a.dD) {
      a.dD[d] = v;
    }
  }
}

static int var_checks(const bcm_scan_args* ap, const bcm_scan_bc* bc, bool bwd, const char* fn) {
  if (!ap || !bc) return set_error(BCM_EINVAL, "%s: null args", fn);
  const bcm_scan_args& a = *ap;
  if (!dtype_ok(a.dtype)) return set_error(BCM_EINVAL, "%s: u_flat must be fp16/bf16/fp32", fn);
  if (a.n_channels < 1) return set_error(BCM_EINVAL, "%s: cu_seqlens must have at least 2 elements", fn);
  if (a.dim < 1) return set_error(BCM_EINVAL, "%s: dim must be >= 1", fn);
  if (a.dstate < 1 || a.dstate > 256) return set_error(BCM_EINVAL, "%s: dstate must be in [1, 256]", fn);
  if (a.max_seqlen < 0) return set_error(BCM_EINVAL, "%s: max_seqlen must be non-negative", fn);
  const int want = a.max_seqlen > 0 ? (a.max_seqlen + kXChunk - 1) / kXChunk : 1;
  if (a.n_chunks != want) return set_error(BCM_EINVAL, "%s: n_chunks must equal max(1, ceil(max_seqlen/2048))", fn);
  if (a.n_events < 0 || a.n_events > INT32_MAX) return set_error(BCM_EINVAL, "%s: n_events out of range", fn);
  if (!a.cu_seqlens || !a.dt_idle || !a.dt_active || !a.A) return set_error(BCM_EINVAL, "%s: null input pointer", fn);
  if (a.n_events > 0 && (!a.u || !a.k)) return set_error(BCM_EINVAL, "%s: null u/k pointer", fn);
  if (bc->layout != BCM_BC_LEGACY && bc->layout != BCM_BC_TILED)
    return set_error(BCM_EINVAL, "%s: B/C layout must be BCM_BC_LEGACY or BCM_BC_TILED", fn);
  if (!bc->B || !bc->C) return set_error(BCM_EINVAL, "%s: null B/C pointer", fn);
  if (bc->layout == BCM_BC_TILED) {
    if (!bc->b_per_event || !bc->c_per_event)
      return set_error(BCM_EINVAL, "%s: tiled B/C are per event", fn);
    if (!bc->tile_offsets || bc->tile_chunk_size < 1 || bc->n_tiles < 0)
      return set_error(BCM_EINVAL, "%s: tiled B/C need tile_offsets, tile_chunk_size >= 1 and n_tiles >= 0", fn);
  } else {
    if (bc->b_row_stride < 1 || bc->c_row_stride < 1)
      return set_error(BCM_EINVAL, "%s: legacy B/C row strides must be >= 1", fn);
  }
  const bool z = a.z != nullptr;
  if (!bwd) {
    if (!a.x || (a.n_events > 0 && !a.out)) return set_error(BCM_EINVAL, "%s: null output pointer", fn);
    if (z && a.n_events > 0 && !a.out_z) return set_error(BCM_EINVAL, "%s: out_z required with z", fn);
  } else {
    if (!a.dA || !a.ddt_idle || !a.ddt_active || !bc->dB || !bc->dC)
      return set_error(BCM_EINVAL, "%s: null gradient pointer", fn);
    if (bc->layout == BCM_BC_LEGACY && (bc->db_row_stride < 1 || bc->dc_row_stride < 1))
      return set_error(BCM_EINVAL, "%s: legacy dB/dC row strides must be >= 1", fn);
    if (a.n_events > 0 && (!a.dout || !a.du)) return set_error(BCM_EINVAL, "%s: null dout/du pointer", fn);
    if (z && a.n_events > 0 && (!a.out_saved || !a.dz))
      return set_error(BCM_EINVAL, "%s: out and dz required with z", fn);
  }
  return BCM_OK;
}

// Waves over the channels first, the rest over the states (a power of two of
// them, at most one per state and item), as far as LDS allows.
static VarShape var_shape(const bcm_scan_args& a, bool bwd) {
  const int64_t per_d = (a.n_channels + a.dim - 1) / a.dim, quads = (per_d + 3) / 4;
  VarShape v{(int)std::max<int64_t>(1, std::min<int64_t>(kVWaves, quads)), 1};
  while (v.nq * v.ns * 2 <= kVWaves && v.ns * 2 <= kVR && v.ns * 2 <= a.dstate) v.ns *= 2;
  const int64_t lds = max_lds_bytes() - 256;
  while (v.bytes(a.dstate, bwd) > lds && v.ns > 1) v.ns /= 2;
  while (v.bytes(a.dstate, bwd) > lds && v.nq > 1) --v.nq;
  return v;
}

template <bool BWD, typename T, bool Z, bool VB, bool VC>
static int var_launch(const bcm_scan_args& a, const bcm_scan_bc& bc, float* hws, hipStream_t s, const char* fn) {
  const VarShape v = var_shape(a, BWD);
  const int64_t lds = v.bytes(a.dstate, BWD);
  if (lds > max_lds_bytes())
    return set_error(BCM_EINVAL, "%s: dstate %d needs %lld bytes of LDS", fn, a.dstate, (long long)lds);
  const dim3 block((unsigned)(v.waves() * kWave));
  if (BWD)
    hipLaunchKernelGGL((k_scan_var_bwd<T, Z, VB, VC>), dim3(a.dim), block, (size_t)lds, s, a, bc, v.nq, v.ns, hws);
  else
    hipLaunchKernelGGL((k_scan_var_fwd<T, Z, VB, VC>), dim3(a.dim), block, (size_t)lds, s, a, bc, v.nq, v.ns, hws);
  return check_launch(fn);
}

template <bool BWD>
static int var_dispatch(const bcm_scan_args& a, const bcm_scan_bc& bc, float* hws, hipStream_t s, const char* fn) {
  int rc = BCM_OK;
  const bool z = a.z != nullptr;
  const int mode = (bc.b_per_event ? 2 : 0) | (bc.c_per_event ? 1 : 0);
  dispatch_dtype(a.dtype, [&](auto tag) {
    using T = decltype(tag);
    auto go = [&](auto zt) {
      constexpr bool Z = decltype(zt)::value;
      switch (mode) {
        case 3: rc = var_launch<BWD, T, Z, true, true>(a, bc, hws, s, fn); break;
        case 2: rc = var_launch<BWD, T, Z, true, false>(a, bc, hws, s, fn); break;
        case 1: rc = var_launch<BWD, T, Z, false, true>(a, bc, hws, s, fn); break;
        default: rc = var_launch<BWD, T, Z, false, false>(a, bc, hws, s, fn); break;
      }
    };
    if (z) go(std::true_type{});
    else go(std::false_type{});
  });
  return rc;
}

}  // namespace bcm

extern "C" {

int64_t bcm_scan_var_workspace_bytes(int64_t n_events, int dstate) {
  return (n_events < 0 || dstate < 1) ? 0 : 4 * n_events * (int64_t)dstate;
}

int bcm_scan_var_fwd(const bcm_scan_args* args, const bcm_scan_bc* bc, bcm_stream_t stream) {
  const char* fn = "bcm_scan_var_fwd";
  int rc = bcm::var_checks(args, bc, false, fn);
  if (rc) return rc;
  return bcm::var_dispatch<false>(*args, *bc, nullptr, bcm::hs(stream), fn);
}

int bcm_scan_var_bwd(const bcm_scan_args* args, const bcm_scan_bc* bc, void* workspace, int64_t workspace_bytes,
                     bcm_stream_t stream) {
  const char* fn = "bcm_scan_var_bwd";
  int rc = bcm::var_checks(args, bc, true, fn);
  if (rc) return rc;
  const int64_t need = bcm_scan_var_workspace_bytes(args->n_events, args->dstate);
  if (need > 0 && (!workspace || workspace_bytes < need))
    return bcm::set_error(BCM_EINVAL, "%s: workspace of %lld bytes needed", fn, (long long)need);
  // forward states h[s, e] of the same inputs (outputs and x not written)
  bcm_scan_args f = *args;
  f.out = nullptr;
  f.out_z = nullptr;
  f.x = nullptr;
  float* hws = static_cast<float*>(workspace);
  rc = bcm::var_dispatch<false>(f, *bc, hws, bcm::hs(stream), fn);
  if (rc) return rc;
  return bcm::var_dispatch<true>(*args, *bc, hws, bcm::hs(stream), fn);
}

}  // extern "C"
