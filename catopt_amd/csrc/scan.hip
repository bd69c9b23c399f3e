// Diagonal affine scans on gfx950 (fp32).
//
// Both kernels are HBM-streaming: every lane owns state elements and walks
// the time axis.  The loads of a block of U steps are issued one block ahead
// of the arithmetic (register double buffering), so each wave keeps
// U x 16 B x 64 lanes of reads in flight while it computes.
//
// Schedules (the int64 chunk table chunk_starts[0..n] cuts [0, T)):
//   STREAM  — one pass; a lane walks the chunks in table order.  HBM-optimal
//             (a is read once) and used whenever the lanes fill the GPU.
//   CHUNKED — three launches: (1) every chunk composes its own map
//             (P = prod a, H = local state from 0), chunk-parallel;
//             (2) per lane, fold the carries over chunks in table order,
//             leaving the carry-in of each chunk in the workspace;
//             (3) every chunk re-runs from its carry-in and emits outputs.
//             This is the two-level blocked scan of the reference's
//             all-prefix path; it trades a second read of the inputs for
//             chunk-level parallelism when B*D*N alone cannot fill the GPU.
// The selective SSM scan streams in T-segments of its own choosing instead
// (ssm_segment below); only an explicit CHUNKED schedule walks the table.
#include <mutex>

#include "common.hpp"

namespace catopt {
namespace {

constexpr int kThreads = 256;

// Chunk bounds clamped to [0, T]: a malformed table can only shorten the
// walk, never index outside the inputs (the host validates the table too).
__device__ __forceinline__ int64_t cclamp(int64_t v, int64_t T) { return v < 0 ? 0 : (v > T ? T : v); }

// ---------------------------------------------------------------- affd scan
// h_t = a_t * h_{t-1} + u_t over [t0, t1) for lane s.
__device__ __forceinline__ float affd_run(const float* __restrict__ a, int64_t lda,
                                          const float* __restrict__ u, int64_t ldu,
                                          float* __restrict__ states, int64_t S, int64_t s,
                                          int64_t t0, int64_t t1, float h, float* prod) {
  constexpr int U = 8;
  float p = 1.f;
  int64_t t = t0;
  for (; t + U <= t1; t += U) {
    float av[U], uv[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      av[i] = a[(t + i) * lda + s];
      uv[i] = u[(t + i) * ldu + s];
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      h = av[i] * h + uv[i];
      p *= av[i];
      if (states) states[(t + i) * S + s] = h;
    }
  }
  for (; t < t1; ++t) {
    const float av = a[t * lda + s];
    h = av * h + u[t * ldu + s];
    p *= av;
    if (states) states[t * S + s] = h;
  }
  if (prod) *prod = p;
  return h;
}

__global__ __launch_bounds__(kThreads) void affd_stream(
    const float* __restrict__ a, int64_t lda, const float* __restrict__ u, int64_t ldu,
    const float* __restrict__ h0, const int64_t* __restrict__ cs, int64_t nc, int64_t T, int64_t S,
    float* __restrict__ states, float* __restrict__ hf) {
  const int64_t s = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (s >= S) return;
  float h = h0 ? h0[s] : 0.f;
  for (int64_t c = 0; c < nc; ++c)
    h = affd_run(a, lda, u, ldu, states, S, s, cclamp(cs[c], T), cclamp(cs[c + 1], T), h, nullptr);
  if (hf) hf[s] = h;
}

// Phase 1: ws_p[c, s] = prod of a over chunk c; ws_h[c, s] = chunk-local state.
__global__ __launch_bounds__(kThreads) void affd_chunk_local(
    const float* __restrict__ a, int64_t lda, const float* __restrict__ u, int64_t ldu,
    const int64_t* __restrict__ cs, int64_t T, int64_t S, float* __restrict__ ws_p,
    float* __restrict__ ws_h) {
  const int64_t s = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t c = blockIdx.y;
  if (s >= S) return;
  float p;
  const float h = affd_run(a, lda, u, ldu, nullptr, S, s, cclamp(cs[c], T), cclamp(cs[c + 1], T), 0.f, &p);
  ws_p[c * S + s] = p;
  ws_h[c * S + s] = h;
}

// Phase 2: carry fold; ws_h[c, s] becomes the state entering chunk c.
__global__ __launch_bounds__(kThreads) void scan_carry(const float* __restrict__ h0, int64_t nc,
                                                       int64_t S, const float* __restrict__ ws_p,
                                                       float* __restrict__ ws_h,
                                                       float* __restrict__ hf) {
  const int64_t s = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (s >= S) return;
  float cin = h0 ? h0[s] : 0.f;
  // the chunk summaries do not depend on the carry: load a batch of them
  // before the batch's stores (which the compiler cannot reorder across
  // ws_h's loads), so a batch costs one memory latency, not one per chunk
  constexpr int kBatch = 16;
  for (int64_t c0 = 0; c0 < nc; c0 += kBatch) {
    const int n = (int)(nc - c0 < kBatch ? nc - c0 : kBatch);
    float p[kBatch], h[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i)
      if (i < n) {
        p[i] = ws_p[(c0 + i) * S + s];
        h[i] = ws_h[(c0 + i) * S + s];
      }
#pragma unroll
    for (int i = 0; i < kBatch; ++i)
      if (i < n) {
        ws_h[(c0 + i) * S + s] = cin;
        cin = p[i] * cin + h[i];
      }
  }
  if (hf) hf[s] = cin;
}

// Phase 3: re-run each chunk from its carry-in, writing the prefix states.
__global__ __launch_bounds__(kThreads) void affd_chunk_apply(
    const float* __restrict__ a, int64_t lda, const float* __restrict__ u, int64_t ldu,
    const int64_t* __restrict__ cs, int64_t T, int64_t S, const float* __restrict__ ws_h,
    float* __restrict__ states) {
  const int64_t s = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t c = blockIdx.y;
  if (s >= S) return;
  affd_run(a, lda, u, ldu, states, S, s, cclamp(cs[c], T), cclamp(cs[c + 1], T), ws_h[c * S + s], nullptr);
}

// ---------------------------------------------------------------- SSM scan
// Thread layout: TPD = N/4 threads per channel d, each owning 4 consecutive
// state elements n (one 16-byte load of a per step); DPW = 256/TPD channels
// per workgroup; grid.y = batch.  y[b,t,d] is reduced across the TPD lanes
// of a channel with DPP moves.
template <int N>
struct SsmLayout {
  static constexpr int TPD = N / 4;
  static constexpr int DPW = kThreads / TPD;
};

template <int N, bool APS>
struct SsmStep {
  f32x4 a;
  f32x4 bx;
  f32x4 c;
  float x;
};

template <int N, bool APS>
__device__ __forceinline__ void ssm_load(SsmStep<N, APS>& st, const float* __restrict__ a,
                                         const float* __restrict__ bx,
                                         const float* __restrict__ c,
                                         const float* __restrict__ x, int64_t b, int64_t t,
                                         int64_t T, int64_t D, int64_t d, int n0) {
  const int64_t bt = b * T + t;
  if (APS) {
    st.a = *reinterpret_cast<const f32x4*>(a + (bt * D + d) * N + n0);
  } else {
    const float av = a[bt * D + d];
    st.a = f32x4{av, av, av, av};
  }
  st.bx = *reinterpret_cast<const f32x4*>(bx + bt * N + n0);
  st.c = *reinterpret_cast<const f32x4*>(c + bt * N + n0);
  st.x = x[bt * D + d];
}

// p plus the DPP-moved p of another lane.
template <int CTRL>
__device__ __forceinline__ float add_dpp(float p) {
  return p + __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(p), CTRL, 0xf, 0xf, true));
}

// The sum over the TPD lanes of a channel, on every one of them: quad
// permutations (lane ^ 1, lane ^ 2), then the mirror of 8 and of 16 lanes,
// whose halves are uniform by then.  A shuffle through LDS per level put
// four LDS latencies on every step of the streaming scan: 0.21 us a step.
template <int N>
__device__ __forceinline__ float lane_reduce(float p) {
  constexpr int TPD = SsmLayout<N>::TPD;
  static_assert(TPD <= 16, "a channel's lanes lie in one DPP row");
  if (TPD >= 2) p = add_dpp<0xB1>(p);    // quad_perm [1, 0, 3, 2]
  if (TPD >= 4) p = add_dpp<0x4E>(p);    // quad_perm [2, 3, 0, 1]
  if (TPD >= 8) p = add_dpp<0x141>(p);   // row_half_mirror
  if (TPD >= 16) p = add_dpp<0x140>(p);  // row_mirror
  return p;
}

// Run steps [t0, t1) from state h; optionally emit y and the product of a.
template <int N, bool APS, bool EMIT>
__device__ __forceinline__ f32x4 ssm_run(const float* __restrict__ a,
                                         const float* __restrict__ bx,
                                         const float* __restrict__ c,
                                         const float* __restrict__ x, float* __restrict__ y,
                                         int64_t b, int64_t T, int64_t D, int64_t d, bool dok,
                                         int n0, int64_t t0, int64_t t1, f32x4 h, f32x4* prod) {
  constexpr int U = 8;
  const int64_t dd = dok ? d : 0;  // out-of-range channels shadow channel 0, never store
  f32x4 p = f32x4{1.f, 1.f, 1.f, 1.f};
  SsmStep<N, APS> cur[U], nxt[U];
  int64_t t = t0;
  if (t + U <= t1) {
#pragma unroll
    for (int i = 0; i < U; ++i) ssm_load(cur[i], a, bx, c, x, b, t + i, T, D, dd, n0);
  }
  for (; t + U <= t1; t += U) {
    const bool more = t + 2 * U <= t1;
    if (more) {
#pragma unroll
      for (int i = 0; i < U; ++i) ssm_load(nxt[i], a, bx, c, x, b, t + U + i, T, D, dd, n0);
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      h = cur[i].a * h + cur[i].bx * cur[i].x;
      if (!EMIT) p *= cur[i].a;
      if (EMIT) {
        const f32x4 ch = cur[i].c * h;
        const float r = lane_reduce<N>(ch[0] + ch[1] + ch[2] + ch[3]);
        if (dok && n0 == 0) y[(b * T + t + i) * D + d] = r;
      }
    }
    if (more) {
#pragma unroll
      for (int i = 0; i < U; ++i) cur[i] = nxt[i];
    }
  }
  for (; t < t1; ++t) {
    SsmStep<N, APS> st;
    ssm_load(st, a, bx, c, x, b, t, T, D, dd, n0);
    h = st.a * h + st.bx * st.x;
    if (!EMIT) p *= st.a;
    if (EMIT) {
      const f32x4 ch = st.c * h;
      const float r = lane_reduce<N>(ch[0] + ch[1] + ch[2] + ch[3]);
      if (dok && n0 == 0) y[(b * T + t) * D + d] = r;
    }
  }
  if (prod) *prod = p;
  return h;
}

template <int N>
struct SsmIdx {
  int64_t d;
  bool dok;
  int n0;
};

template <int N>
__device__ __forceinline__ SsmIdx<N> ssm_idx(int64_t D) {
  SsmIdx<N> r;
  const int tl = threadIdx.x;
  r.d = (int64_t)blockIdx.x * SsmLayout<N>::DPW + tl / SsmLayout<N>::TPD;
  r.dok = r.d < D;
  r.n0 = (tl % SsmLayout<N>::TPD) * 4;
  return r;
}

template <int N, bool APS>
__global__ __launch_bounds__(kThreads) void ssm_chunk_local(
    const float* __restrict__ a, const float* __restrict__ bx, const float* __restrict__ c,
    const float* __restrict__ x, const int64_t* __restrict__ cs, int64_t T, int64_t D,
    int64_t S, float* __restrict__ ws_p, float* __restrict__ ws_h) {
  const SsmIdx<N> ix = ssm_idx<N>(D);
  const int64_t b = blockIdx.y, k = blockIdx.z;
  f32x4 p;
  const f32x4 h = ssm_run<N, APS, false>(a, bx, c, x, nullptr, b, T, D, ix.d, ix.dok, ix.n0,
                                         cclamp(cs[k], T), cclamp(cs[k + 1], T),
                                         f32x4{0.f, 0.f, 0.f, 0.f}, &p);
  if (!ix.dok) return;
  const int64_t sidx = (b * D + ix.d) * N + ix.n0;
  *reinterpret_cast<f32x4*>(ws_p + k * S + sidx) = p;
  *reinterpret_cast<f32x4*>(ws_h + k * S + sidx) = h;
}

template <int N, bool APS>
__global__ __launch_bounds__(kThreads) void ssm_chunk_apply(
    const float* __restrict__ a, const float* __restrict__ bx, const float* __restrict__ c,
    const float* __restrict__ x, const int64_t* __restrict__ cs, int64_t T, int64_t D,
    int64_t S, const float* __restrict__ ws_h, float* __restrict__ y) {
  const SsmIdx<N> ix = ssm_idx<N>(D);
  const int64_t b = blockIdx.y, k = blockIdx.z;
  const int64_t sidx = (b * D + (ix.dok ? ix.d : 0)) * N + ix.n0;
  const f32x4 h = *reinterpret_cast<const f32x4*>(ws_h + k * S + sidx);
  ssm_run<N, APS, true>(a, bx, c, x, y, b, T, D, ix.d, ix.dok, ix.n0, cclamp(cs[k], T),
                        cclamp(cs[k + 1], T), h, nullptr);
}

// ------------------------------------------------------- streaming segments
// The scan over T-segments: a workgroup owns DPW channels x N states (one
// 4 KB slice of a per step, 16 bytes per thread) and walks one segment of
// the steps.  With one segment (enough workgroups to fill the chip) that is
// a single pass over a; with P segments two launches:
//   EMIT = false  composes each segment but the last into (prod a, local
//                 state), reading a, b and x;
//   EMIT = true   starts each segment from h0 folded through the segments
//                 before it, and emits y.  It reads the copy of h0 that the
//                 first launch left in the workspace: its last segment
//                 writes h_final, which may be h0's own buffer, while the
//                 others may not have begun.
// 8 x 8192 x 2048 x 16: 1790 us a call (5.4 TB/s) where the chunk-parallel
// schedule, which reads a twice in three launches, took 4300.
// HBM bounds both, and below two workgroups per CU what bounds a workgroup
// is the latency of its loads: with loads one stage ahead a stage took 1.66 us
// (20 GB/s per workgroup).  So everything is loaded two stages ahead, into
// one of three register sets: a's slices for RSU steps and this thread's
// share of the small x, b and c streams.  The share goes to LDS (one copy per
// workgroup, three buffers) one stage before it is read, and y leaves
// through LDS as whole rows.  Every load is an ordinary load into registers,
// so the compiler derives every wait and no result depends on the order in
// which it places them.  No load has a branch around it: a lane past the end
// of a small stream repeats another lane's slot.  In two stages of three the
// derived waits leave the newest two stages in flight.  The loop's back edge
// joins paths of one, two and three stages, and there the compiler waits for
// every load, so the run-ahead starts anew with each third stage.
// y's stores are non-temporal (written once, never read back here): 1.5%
// faster at C5's shape than plain stores.  What y costs beyond that is
// HBM's turnaround between reads and writes; a plain streaming kernel with
// the same 16:1 read/write mix pays it as well.  Steps past the last whole
// stage run unpipelined.
constexpr int RSU = 8;  // steps per stage

template <int N>
struct SsmSmall {
  static constexpr int TPD = N / 4, DPW = kThreads / TPD;
  static constexpr int X_SLOTS = RSU * DPW, V_SLOTS = 2 * RSU * N;  // 4-byte slots: x (and y); b, then c
  static constexpr int STAGE = (X_SLOTS + V_SLOTS) * 4;
  static constexpr int Y_BYTES = X_SLOTS * 4;
  static constexpr int BYTES = 3 * (STAGE + Y_BYTES);
  static constexpr int XPT = (X_SLOTS + kThreads - 1) / kThreads;  // x loads (and y stores) per thread
  static constexpr int VPT = (V_SLOTS + kThreads - 1) / kThreads;  // b and c loads per thread
  static_assert(X_SLOTS % 64 == 0, "store_y's guards are wave-uniform");
};

// One thread's loads of a stage: a's slices, and its slots of x and of b, c.
template <int N>
struct SsmStage {
  f32x4 a[RSU];
  float x[SsmSmall<N>::XPT], v[SsmSmall<N>::VPT];
};

// The stages [first, second) of RSU steps that segment seg of P walks (the
// steps past the last whole stage belong to the last segment).
__device__ __forceinline__ int64_t seg_stage(int64_t T, int64_t seg, int64_t P) { return (T / RSU) * seg / P; }

// a ⊙ h + b x, rounding a h and fusing b x: with a in (0, 1) the rounded
// product is the smaller one, and the states' error against 64 bits is 12%
// less than with the other product rounded.
__device__ __forceinline__ f32x4 ssm_step(f32x4 a, f32x4 h, f32x4 b, float x) {
  const f32x4 ah = a * h;
  f32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_fmaf(b[i], x, ah[i]);
  return r;
}

template <int N, bool APS, bool EMIT>
__global__ __launch_bounds__(kThreads, 2) void ssm_segment(
    const float* __restrict__ a, const float* __restrict__ bx, const float* __restrict__ c,
    const float* __restrict__ x, const float* __restrict__ h0, int64_t T, int64_t D, int64_t S,
    int64_t P, float* __restrict__ ws_p, float* __restrict__ ws_h, float* __restrict__ y,
    float* __restrict__ hf) {
  using L = SsmSmall<N>;
  __shared__ __attribute__((aligned(16))) char lds[L::BYTES];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t b = blockIdx.y, seg = blockIdx.z;
  const int64_t d0 = (int64_t)blockIdx.x * L::DPW;
  const int ch = tid / L::TPD, n0 = (tid % L::TPD) * 4;
  const int64_t d = d0 + ch;
  const bool dok = d < D;
  const int64_t dd = dok ? d : D - 1;  // channels past D shadow the last one, never stored
  const int64_t st0 = seg_stage(T, seg, P), st1 = seg_stage(T, seg + 1, P);
  // this thread's x slots (step u, channel), clamped to valid channels: their
  // elements' offsets in a stage of x and of y, and their words in LDS.  All
  // per-stage address arithmetic is on wave-uniform bases.
  int64_t xo[L::XPT];
  int xw[L::XPT];
#pragma unroll
  for (int i = 0; i < L::XPT; ++i) {
    const int s = (i * kThreads + tid) % L::X_SLOTS, u = s / L::DPW;
    const int cc = (int)(d0 + s % L::DPW < D ? s % L::DPW : D - 1 - d0);
    xo[i] = u * D + d0 + cc;
    xw[i] = u * L::DPW + cc;
  }
  // and its b and c slots: RSU * N of b, then of c (not emitting, b alone)
  constexpr int VS = EMIT ? L::V_SLOTS : L::V_SLOTS / 2, VPT = (VS + kThreads - 1) / kThreads;
  const uint32_t ao = (uint32_t)(APS ? (dd - d0) * N + n0 : dd - d0);

  // stage st into registers, the small streams first (they are used first)
  auto load = [&](int64_t st, SsmStage<N>& r) {
    const int64_t bt = b * T + st * RSU;
#pragma unroll
    for (int i = 0; i < L::XPT; ++i) r.x[i] = x[bt * D + xo[i]];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int s = (i * kThreads + tid) % VS;
      r.v[i] = s < RSU * N ? bx[bt * N + s] : c[bt * N + s - RSU * N];
    }
    const float* ar = a + (bt * D + d0) * (APS ? N : 1);
    const int64_t row = D * (APS ? N : 1);
#pragma unroll
    for (int u = 0; u < RSU; ++u) {
      if (APS) {
        r.a[u] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(ar + u * row + ao));
      } else {
        const float av = (ar + u * row)[ao];
        r.a[u] = f32x4{av, av, av, av};
      }
    }
  };
  // a stage's small streams into LDS buffer `buf` (a repeated slot: the same
  // value to the same word)
  auto put = [&](const SsmStage<N>& r, int buf) {
    float* xb = reinterpret_cast<float*>(lds + buf * L::STAGE);
#pragma unroll
    for (int i = 0; i < L::XPT; ++i) xb[(i * kThreads + tid) % L::X_SLOTS] = r.x[i];
#pragma unroll
    for (int i = 0; i < VPT; ++i) xb[L::X_SLOTS + (i * kThreads + tid) % VS] = r.v[i];
  };

  f32x4 h = f32x4{0.f, 0.f, 0.f, 0.f}, p = f32x4{1.f, 1.f, 1.f, 1.f};
  const int64_t sidx = (b * D + dd) * N + n0;
  if (EMIT) {
    if (h0) h = *reinterpret_cast<const f32x4*>(h0 + sidx);
    // the segments before this one, in order; their summaries do not depend
    // on the carry, so a batch of them costs one memory latency
    constexpr int kBatch = 8;
    for (int64_t k0 = 0; k0 < seg; k0 += kBatch) {
      f32x4 pk[kBatch], hk[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {  // past the last: that one again, not used (no branch between the loads)
        const int64_t k = k0 + i < seg ? k0 + i : seg - 1;
        pk[i] = *reinterpret_cast<const f32x4*>(ws_p + k * S + sidx);
        hk[i] = *reinterpret_cast<const f32x4*>(ws_h + k * S + sidx);
      }
#pragma unroll
      for (int i = 0; i < kBatch; ++i)
        if (k0 + i < seg) h = pk[i] * h + hk[i];
    }
  }
  auto compute = [&](int buf, const f32x4* ra, char* yb) {
    const char* xb = lds + buf * L::STAGE;
    const char* vb = xb + L::X_SLOTS * 4;
    float r[RSU];
#pragma unroll
    for (int u = 0; u < RSU; ++u) {
      const f32x4 bv = *reinterpret_cast<const f32x4*>(vb + (u * N + n0) * 4);
      const float xv = *reinterpret_cast<const float*>(xb + (u * L::DPW + ch) * 4);
      h = ssm_step(ra[u], h, bv, xv);
      if (EMIT) {
        const f32x4 cv = *reinterpret_cast<const f32x4*>(vb + (RSU * N + u * N + n0) * 4);
        const f32x4 chv = cv * h;
        r[u] = lane_reduce<N>(chv[0] + chv[1] + chv[2] + chv[3]);
      } else {
        p *= ra[u];
      }
    }
    if (!EMIT) return;
    // every lane of a channel has every step's sum: lane j writes steps j,
    // j + TPD, ... (a write under a lane mask per step would keep the next
    // step's reads from being issued ahead of it)
    const int j = (tid % L::TPD) % RSU;
#pragma unroll
    for (int k = 0; k < RSU; k += L::TPD) {
      float v = r[k];
#pragma unroll
      for (int i = 1; i < L::TPD && i < RSU; ++i) v = j == i ? r[k + i] : v;
      *reinterpret_cast<float*>(yb + ((k + j) * L::DPW + ch) * 4) = v;
    }
  };
  // y rows of a stage from LDS: row u, channels d0 .. d0 + DPW - 1
  auto store_y = [&](int64_t st, const char* yb) {
    float* yr = y + (b * T + st * RSU) * D;
#pragma unroll
    for (int i = 0; i < L::XPT; ++i) {
      // a channel past D (last, partial workgroup) writes channel D - 1's
      // value to it again: no lane mask around the store
      if (i * kThreads + wave * 64 < L::X_SLOTS)
        __builtin_nontemporal_store(*reinterpret_cast<const float*>(yb + xw[i] * 4), yr + xo[i]);
    }
  };
  auto issue = [&](int64_t st, SsmStage<N>& r) {
    load(st < st1 ? st : st1 - 1, r);    // past the end: the last stage again, not used
    __builtin_amdgcn_sched_barrier(0);  // ahead of the products that hide it
  };
  // stage st from register set `cur` and buffer `buf`; stage st + 1's small
  // streams go to buffer `nbuf`, stage st + 2 into `ahead`.  A buffer is
  // written two barriers after its last reader's stage began, and read past
  // the barrier that follows the write.
  auto step = [&](int64_t st, int buf, const SsmStage<N>& cur, int nbuf, const SsmStage<N>& nxt, SsmStage<N>& ahead) {
    issue(st + 2, ahead);
    char* yb = lds + 3 * L::STAGE + buf * L::Y_BYTES;
    compute(buf, cur.a, yb);
    put(nxt, nbuf);
    __syncthreads();
    if (EMIT) store_y(st, yb);
  };
  SsmStage<N> r0, r1, r2;
  if (st0 < st1) {
    issue(st0, r0);
    issue(st0 + 1, r1);
    put(r0, 0);
    __syncthreads();
    for (int64_t st = st0; st < st1; st += 3) {
      step(st, 0, r0, 1, r1, r2);
      if (st + 1 < st1) step(st + 1, 1, r1, 2, r2, r0);
      if (st + 2 < st1) step(st + 2, 2, r2, 0, r0, r1);
    }
  }
  if (!EMIT) {
    if (!dok) return;
    // the last segment's place in ws_h is not used: h0's copy
    if (seg == 0 && h0)
      *reinterpret_cast<f32x4*>(ws_h + (P - 1) * S + sidx) = *reinterpret_cast<const f32x4*>(h0 + sidx);
    *reinterpret_cast<f32x4*>(ws_p + seg * S + sidx) = p;
    *reinterpret_cast<f32x4*>(ws_h + seg * S + sidx) = h;
    return;
  }
  if (seg + 1 < P) return;
  // steps past the last whole stage
  for (int64_t t = T / RSU * RSU; t < T; ++t) {
    SsmStep<N, APS> sp;
    ssm_load(sp, a, bx, c, x, b, t, T, D, dd, n0);
    h = ssm_step(sp.a, h, sp.bx, sp.x);
    const f32x4 chv = sp.c * h;
    const float r = lane_reduce<N>(chv[0] + chv[1] + chv[2] + chv[3]);
    if (dok && n0 == 0) y[(b * T + t) * D + d] = r;
  }
  if (hf && dok) *reinterpret_cast<f32x4*>(hf + sidx) = h;
}

// Lanes that fill the GPU: 256 CUs x 8 waves x 64 lanes.
constexpr int64_t kFillThreads = 256LL * 8 * 64;

// The schedule a launch runs: the automatic choice streams when the lanes
// fill the GPU and goes chunk-parallel otherwise.  The workspace queries use
// the same functions, so a caller sizes exactly what the launch will read.
bool affd_chunked(int64_t S, int64_t nc, int32_t schedule) {
  if (schedule == CATOPT_SCAN_CHUNKED) return true;
  return schedule == CATOPT_SCAN_AUTO && nc > 1 && S < kFillThreads;
}

// Segments of the SSM scan under the automatic schedule, at most one per chunk
// of the caller's table (which sizes the workspace).  One pass reads a once
// but takes 0.86 us per stage however few workgroups walk it; P segments read
// it 2 - 1/P times.  One pass wins from about 84 workgroups up (D = 2048,
// N = 16, T = 8192: 128 workgroups 1033 us against 1307 at P = 2, 64
// workgroups 906 against 701 at P = 4).  Below that the best P puts one
// workgroup on each CU: more, and the pass ends in a part-filled second round
// (32 workgroups, T = 8192: P = 8 365 us, P = 10 438, P = 16 396).  Many
// segments are taken odd in number, so that their starts do not lie a power
// of two of bytes apart (16 workgroups, T = 2048: P = 15 50 us, P = 16 61).
int64_t ssm_segments(int64_t B, int64_t T, int64_t D, int64_t N, int64_t nc) {
  constexpr int64_t kOnePass = 84, kCus = 256, kMinStages = 2;
  const int64_t dpw = kThreads / (N / 4);  // channels per workgroup
  const int64_t wgs = (D + dpw - 1) / dpw * B;
  if (wgs <= 0 || wgs >= kOnePass || nc <= 1) return 1;
  int64_t P = kCus / wgs;
  if (P > 8 && P % 2 == 0) --P;
  if (P > T / (RSU * kMinStages)) P = T / (RSU * kMinStages);
  if (P > nc) P = nc;
  return P < 2 ? 1 : P;
}

bool ssm_chunked(int64_t B, int64_t T, int64_t D, int64_t N, int64_t nc, int32_t schedule) {
  if (schedule == CATOPT_SCAN_CHUNKED) return true;
  return schedule == CATOPT_SCAN_AUTO && ssm_segments(B, T, D, N, nc) > 1;
}

template <int N, bool APS>
int32_t ssm_launch(int64_t B, int64_t T, int64_t D, const float* a, const float* bx,
                   const float* c, const float* x, const float* h0, const int64_t* cs,
                   int64_t nc, int32_t schedule, float* y, float* hf, void* ws, int64_t wsb,
                   hipStream_t s) {
  const int64_t gx = (D + SsmLayout<N>::DPW - 1) / SsmLayout<N>::DPW;
  const int64_t S = B * D * N;
  static_assert(SsmLayout<N>::TPD == N / 4, "ssm_segments assumes four states per thread");
  if (gx > 0x7fffffff || B > 65535 || nc > 65535) return CATOPT_E_UNSUPPORTED;
  if (schedule != CATOPT_SCAN_CHUNKED) {
    int64_t P = schedule == CATOPT_SCAN_AUTO ? ssm_segments(B, T, D, N, nc) : 1;
    float* ws_p = static_cast<float*>(ws);
    float* ws_h = ws_p + P * S;
    if (P > 1) {
      if (!ws || wsb < catopt_hip_scan_workspace_bytes(S, nc)) return CATOPT_E_WORKSPACE;
      ssm_segment<N, APS, false><<<dim3((uint32_t)gx, (uint32_t)B, (uint32_t)(P - 1)), dim3(kThreads), 0, s>>>(
          a, bx, c, x, h0, T, D, S, P, ws_p, ws_h, y, hf);
      CATOPT_LAUNCH_CHECK();
      if (h0) h0 = ws_h + (P - 1) * S;
    }
    ssm_segment<N, APS, true><<<dim3((uint32_t)gx, (uint32_t)B, (uint32_t)P), dim3(kThreads), 0, s>>>(
        a, bx, c, x, h0, T, D, S, P, ws_p, ws_h, y, hf);
    CATOPT_LAUNCH_CHECK();
    return CATOPT_OK;
  }
  if (!ws || wsb < catopt_hip_scan_workspace_bytes(S, nc)) return CATOPT_E_WORKSPACE;
  float* ws_p = static_cast<float*>(ws);
  float* ws_h = ws_p + nc * S;
  ssm_chunk_local<N, APS><<<dim3((uint32_t)gx, (uint32_t)B, (uint32_t)nc), dim3(kThreads), 0, s>>>(
      a, bx, c, x, cs, T, D, S, ws_p, ws_h);
  CATOPT_LAUNCH_CHECK();
  scan_carry<<<dim3((uint32_t)((S + kThreads - 1) / kThreads)), dim3(kThreads), 0, s>>>(
      h0, nc, S, ws_p, ws_h, hf);
  CATOPT_LAUNCH_CHECK();
  ssm_chunk_apply<N, APS><<<dim3((uint32_t)gx, (uint32_t)B, (uint32_t)nc), dim3(kThreads), 0, s>>>(
      a, bx, c, x, cs, T, D, S, ws_h, y);
  CATOPT_LAUNCH_CHECK();
  return CATOPT_OK;
}

}  // namespace
}  // namespace catopt

using namespace catopt;

extern "C" int64_t catopt_hip_scan_workspace_bytes(int64_t S, int64_t n_chunks) {
  if (S < 0 || n_chunks < 0) return -1;
  return 2 * S * n_chunks * (int64_t)sizeof(float);
}

extern "C" int64_t catopt_hip_affd_scan_workspace_bytes(int64_t T, int64_t S, int64_t n_chunks,
                                                         int32_t schedule) {
  if (T < 0 || S < 0 || n_chunks < 1) return -1;
  if (schedule < CATOPT_SCAN_AUTO || schedule > CATOPT_SCAN_CHUNKED) return -1;
  return affd_chunked(S, n_chunks, schedule) ? catopt_hip_scan_workspace_bytes(S, n_chunks) : 0;
}

extern "C" int64_t catopt_hip_ssm_scan_workspace_bytes(int64_t B, int64_t T, int64_t D, int64_t N,
                                                        int64_t n_chunks, int32_t schedule) {
  if (B < 0 || T < 0 || D < 0 || n_chunks < 1) return -1;
  if (schedule < CATOPT_SCAN_AUTO || schedule > CATOPT_SCAN_CHUNKED) return -1;
  if (N != 4 && N != 8 && N != 16 && N != 32 && N != 64) return -1;
  return ssm_chunked(B, T, D, N, n_chunks, schedule) ? catopt_hip_scan_workspace_bytes(B * D * N, n_chunks)
                                                  : 0;
}

namespace catopt {
namespace {

// Argument checks and launches of catopt_hip_affd_scan, with the workspace
// resolved by the caller: `ws_cap` is the bytes available at `ws` (a caller
// buffer, or the static scratch array of the no-allocation entry point).
int32_t affd_scan_body(int64_t T, int64_t S, const float* a, int64_t lda, const float* u,
                       int64_t ldu, const float* h0, const int64_t* chunk_starts,
                       int64_t n_chunks, int32_t schedule, float* states, float* h_final,
                       void* ws, int64_t ws_cap, hipStream_t s) {
  if (S > 0x7fffffffLL * kThreads || n_chunks > 65535) return CATOPT_E_UNSUPPORTED;
  const int64_t gx = (S + kThreads - 1) / kThreads;
  const bool chunked = affd_chunked(S, n_chunks, schedule);
  if (!chunked) {
    affd_stream<<<dim3((uint32_t)gx), dim3(kThreads), 0, s>>>(a, lda, u, ldu, h0, chunk_starts,
                                                              n_chunks, T, S, states, h_final);
    CATOPT_LAUNCH_CHECK();
    return CATOPT_OK;
  }
  if (!ws || ws_cap < catopt_hip_scan_workspace_bytes(S, n_chunks)) return CATOPT_E_WORKSPACE;
  float* ws_p = static_cast<float*>(ws);
  float* ws_h = ws_p + n_chunks * S;
  affd_chunk_local<<<dim3((uint32_t)gx, (uint32_t)n_chunks), dim3(kThreads), 0, s>>>(
      a, lda, u, ldu, chunk_starts, T, S, ws_p, ws_h);
  CATOPT_LAUNCH_CHECK();
  scan_carry<<<dim3((uint32_t)gx), dim3(kThreads), 0, s>>>(h0, n_chunks, S, ws_p, ws_h, h_final);
  CATOPT_LAUNCH_CHECK();
  if (states) {
    affd_chunk_apply<<<dim3((uint32_t)gx, (uint32_t)n_chunks), dim3(kThreads), 0, s>>>(
        a, lda, u, ldu, chunk_starts, T, S, ws_h, states);
    CATOPT_LAUNCH_CHECK();
  }
  return CATOPT_OK;
}

int32_t affd_scan_args_ok(int64_t T, int64_t S, const float* a, int64_t lda, const float* u,
                          int64_t ldu, const int64_t* chunk_starts, int64_t n_chunks,
                          int32_t schedule) {
  if (T < 0 || S < 0 || n_chunks < 1 || lda < 0 || ldu < S) return CATOPT_E_INVAL;
  if (lda != 0 && lda < S) return CATOPT_E_INVAL;
  if (schedule < CATOPT_SCAN_AUTO || schedule > CATOPT_SCAN_CHUNKED) return CATOPT_E_INVAL;
  if (S > 0 && (!chunk_starts || (T > 0 && (!a || !u)))) return CATOPT_E_INVAL;
  return CATOPT_OK;
}

// Scratch of the no-allocation entry point: a file-scope device array that
// each GPU holds from the library's load to the end of the process.  Its
// name is a host-side stand-in, not a device address: host code uses only
// the per-device address that hipGetSymbolAddress returns for it.  The
// chunk-parallel schedule writes every word it later reads (chunk maps and
// local states, then the carries), so nothing in it has to start at zero.
constexpr int64_t kAffdScratchBytes = CATOPT_AFFD_SCAN_SCRATCH_BYTES;
static __device__ __align__(256) float scratch[kAffdScratchBytes / sizeof(float)];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The address of `scratch` on the stream's device, looked up once per
// device with that device current (made current for the lookup when the
// caller's current device is another one, then restored).
int32_t affd_scratch(hipStream_t stream, void** out) {
  hipDevice_t dev = -1;
  hipError_t e = hipStreamGetDevice(stream, &dev);
  if (e != hipSuccess) return set_hip_error(e);
  if (dev < 0 || dev >= kMaxDevices) return CATOPT_E_UNSUPPORTED;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    int cur = -1;
    e = hipGetDevice(&cur);
    if (e != hipSuccess) return set_hip_error(e);
    if (cur != dev) {
      e = hipSetDevice(dev);
      if (e != hipSuccess) return set_hip_error(e);
    }
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    const hipError_t back = cur != dev ? hipSetDevice(cur) : hipSuccess;
    if (e != hipSuccess) return set_hip_error(e);
    if (back != hipSuccess) return set_hip_error(back);
    if (!p) return CATOPT_E_HIP;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return CATOPT_OK;
}

}  // namespace
}  // namespace catopt

extern "C" int32_t catopt_hip_affd_scan(int64_t T, int64_t S, const float* a, int64_t lda,
                                        const float* u, int64_t ldu, const float* h0,
                                        const int64_t* chunk_starts, int64_t n_chunks,
                                        int32_t schedule, float* states, float* h_final,
                                        void* workspace, int64_t workspace_bytes, void* stream) {
  const int32_t st = affd_scan_args_ok(T, S, a, lda, u, ldu, chunk_starts, n_chunks, schedule);
  if (st != CATOPT_OK) return st;
  if (S == 0) return CATOPT_OK;
  return affd_scan_body(T, S, a, lda, u, ldu, h0, chunk_starts, n_chunks, schedule, states, h_final,
                        workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

extern "C" int64_t catopt_hip_affd_scan_noalloc_max_bytes(void) { return kAffdScratchBytes; }

extern "C" int32_t catopt_hip_affd_scan_noalloc(int64_t T, int64_t S, const float* a, int64_t lda,
                                                const float* u, int64_t ldu, const float* h0,
                                                const int64_t* chunk_starts, int64_t n_chunks,
                                                int32_t schedule, float* states, float* h_final,
                                                void* stream) {
  int32_t st = affd_scan_args_ok(T, S, a, lda, u, ldu, chunk_starts, n_chunks, schedule);
  if (st != CATOPT_OK) return st;
  if (S == 0) return CATOPT_OK;
  void* ws = nullptr;
  if (affd_chunked(S, n_chunks, schedule)) {
    // reject before touching the device: the chunked workspace must fit
    if (catopt_hip_scan_workspace_bytes(S, n_chunks) > kAffdScratchBytes) return CATOPT_E_WORKSPACE;
    st = affd_scratch(static_cast<hipStream_t>(stream), &ws);
    if (st != CATOPT_OK) return st;
  }
  return affd_scan_body(T, S, a, lda, u, ldu, h0, chunk_starts, n_chunks, schedule, states, h_final,
                        ws, ws ? kAffdScratchBytes : 0, static_cast<hipStream_t>(stream));
}

extern "C" int32_t catopt_hip_ssm_scan(int64_t B, int64_t T, int64_t D, int64_t N,
                                       const float* a, int32_t a_per_state, const float* bx,
                                       const float* c, const float* x, const float* h0,
                                       const int64_t* chunk_starts, int64_t n_chunks,
                                       int32_t schedule, float* y, float* h_final,
                                       void* workspace, int64_t workspace_bytes, void* stream) {
  if (B < 0 || T < 0 || D < 0 || n_chunks < 1) return CATOPT_E_INVAL;
  if (schedule < CATOPT_SCAN_AUTO || schedule > CATOPT_SCAN_CHUNKED) return CATOPT_E_INVAL;
  if (B == 0 || D == 0) return CATOPT_OK;
  if (!chunk_starts || (T > 0 && (!a || !bx || !c || !x || !y))) return CATOPT_E_INVAL;
  if (!aligned16(a) && a_per_state) return CATOPT_E_INVAL;
  if (!aligned16(bx) || !aligned16(c) || (h0 && !aligned16(h0)) || (h_final && !aligned16(h_final)))
    return CATOPT_E_INVAL;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define CATOPT_SSM(NN)                                                                                \
  case NN:                                                                                            \
    return a_per_state ? ssm_launch<NN, true>(B, T, D, a, bx, c, x, h0, chunk_starts, n_chunks,     \
                                              schedule, y, h_final, workspace, workspace_bytes, s)  \
                       : ssm_launch<NN, false>(B, T, D, a, bx, c, x, h0, chunk_starts, n_chunks,    \
                                               schedule, y, h_final, workspace, workspace_bytes, s);
  switch (N) {
    CATOPT_SSM(4)
    CATOPT_SSM(8)
    CATOPT_SSM(16)
    CATOPT_SSM(32)
    CATOPT_SSM(64)
    default:
      return CATOPT_E_UNSUPPORTED;
  }
#undef CATOPT_SSM
}
