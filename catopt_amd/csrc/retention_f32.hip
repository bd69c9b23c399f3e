// Chunked decayed retention on fp32 operands (gfx950 fp32 MFMA,
// v_mfma_f32_32x32x2_f32):
//
//   o[t] = scale · Σ_{s ≤ t} γ^(t−s) (q[t]·k[s]) v[s]
//
// in chunks of C = 32 steps: for chunk n with carried state S (d × d),
//   o_n = scale · ( (q_n k_nᵀ ⊙ D) v_n + diag(γ^a) q_n S ),   D[a, b] = γ^(a−b) (a ≥ b)
//   S  ← γ^C S + k_nᵀ diag(γ^(C−b)) v_n
// which is the bf16 kernel's algebra with every operand, product and the
// state in fp32 (no rounding to bf16 anywhere).
//
// Work split.  The fp32 MFMA bounds it (64 cycles for 32 x 32 x 2), so the
// split computes nothing twice and puts a wave on every SIMD.  Each head's
// chunks are cut into P segments; retention_f32<STATE> folds each segment
// but the last into its state from zero, and retention_f32<OUT> starts each
// segment from the fold of those before it and emits the outputs.  In a
// workgroup wave w owns value columns 32w .. 32w + 31 and the state tiles
// S[:, 32w..]; the 32 x 32 scores of a chunk are split over the waves by q/k
// columns and their partial sums meet in LDS.  160 MFMAs per wave and chunk
// at d = 128.  (With a workgroup per 32 value columns and all of a head's
// chunks in order, each slice recomputed the scores and each wave the whole
// P v.)  Measured, that kernel and this one: 32 heads x 2048 steps x 128
// 255 / 96 us, 64 x 8192 x 128 1009 / 588, 32 x 2048 x 64 219 / 45.  A product
// takes 38-40 ns here (27 at 2.4 GHz; without the loads the 64 x 8192 output
// pass still takes 409 of 471 us).  With MFMA accumulators in VGPRs
// (-amdgpu-mfma-vgpr-form) d = 128 is 5% faster and d = 64 16-25% slower: two
// waves then fit a SIMD and both of a workgroup's may land on one.
//
// The q, k and v rows of a chunk go global->LDS directly, one chunk ahead.
// LDS rows are XOR-swizzled by a permutation of the row's low four bits that
// keeps both reads free of bank conflicts: 16-byte reads along a row by 32
// lanes on 32 rows, and 4-byte reads of 32 columns of rows j and j + 4 by the
// two lane halves.
//
// Operand layouts (32x32x2 f32 MFMA: lane l gives A row l%32 and B column
// l%32 at k index l/32; the accumulator of lane l holds column l%32, rows
// acc_row(r, l/32) in register r).  The k index of a product is a summation
// order, so k-step t with half-wave g can take any inner index as long as A
// and B agree; every product here takes inner index acc_row(t, g) (plus the
// tile base), which lets accumulators feed the next product directly:
//   * the state accumulator S[dd, c] (lane: column c, register t: row dd)
//     is the B operand of the inter term O = Q S;
//   * the score accumulator Pᵀ[j, i] (lane: query i, register t: key j) is
//     the A operand of O += P V.
// Loads go through buffer resources over the head's rows: rows past T and
// columns past d read zeros, and stores there are dropped.
#include "common.hpp"

namespace catopt {
namespace {

constexpr int kC = 32;                  // chunk length (steps)
constexpr uint32_t kOOB = 0x80000000u;  // a buffer offset past every range: loads 0, stores nothing
constexpr int64_t kMaxSeg = 16;

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// N steps of one or two products with `read` behind them.  With one wave per
// SIMD an LDS read right before its use is waited out, so every stream of
// products carries the reads of the next one; and a product that adds to the
// result of the one before it waits for it, so streams alternate between two
// accumulators.
template <int N, typename Product, typename Read>
__device__ __forceinline__ void stream(Product product, Read read) {
#pragma unroll
  for (int x = 0; x < N; ++x) {
    product(x);
    read(x);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// ND tiles of 32 columns (d <= 32 ND) and as many waves.
template <int ND>
struct Ret {
  static constexpr int NT = 64 * ND, ROW = 128 * ND;        // threads; bytes of an LDS row
  static constexpr int CH = 8 * ND;                         // 16-byte chunks of a row
  static constexpr int MAT = kC * ROW;                      // one matrix of a chunk
  static constexpr int LOADS = MAT / 1024 / ND;             // 1 KB loads per wave and matrix
  static constexpr int64_t STATE = 1024LL * ND * ND;        // floats
  static_assert(CH >= 16, "the swizzle permutes 16 chunks");
};

// The swizzle of row r: its low four bits with bits 2 and 3 traded.
__device__ __forceinline__ int row_swz(int r) { return (r & 3) | ((r & 4) << 1) | ((r & 8) >> 1); }

// Chunks [first, ...) of segment seg.
__host__ __device__ inline int64_t seg_first(int64_t nch, int64_t seg, int64_t P) { return nch * seg / P; }

template <int ND, bool OUT>
__global__ __launch_bounds__(64 * ND, 1) void retention_f32(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ gamma, float scale, float* __restrict__ o, float* __restrict__ pieces, int H, int T,
    int d, int P) {
  using L = Ret<ND>;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr int NMAT = OUT ? 3 : 2, STAGE = NMAT * L::MAT;  // (q,) k, v
  const int nseg = OUT ? P : P - 1;
  const int64_t bh = blockIdx.x / nseg;
  const int seg = blockIdx.x % nseg;
  const int h = (int)(bh % H);
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t base = bh * (int64_t)T * d;
  const uint32_t bytes = (uint32_t)T * (uint32_t)d * 4u;
  const u32x4 rq = make_rsrc(q + base, bytes), rk = make_rsrc(k + base, bytes), rv = make_rsrc(v + base, bytes);
  const int nch = (T + kC - 1) / kC;
  const int c0 = (int)seg_first(nch, seg, P), c1 = (int)seg_first(nch, seg + 1, P);

  // decay factors of this lane, fixed over the chunks (exp2 domain)
  const float gam = gamma[h];
  const float lg = log2f(fabsf(gam));
  const bool neg = gam < 0.f;
  float rowf[16], diagf[16], wv[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int ar = acc_row(r, g);
    rowf[r] = pow_k(lg, neg, ar);                            // γ^a, a = row in chunk
    diagf[r] = ar <= l32 ? pow_k(lg, neg, l32 - ar) : 0.f;    // D
    wv[r] = pow_k(lg, neg, kC - ar);                         // γ^(C − b)
  }
  const float gC = pow_k(lg, neg, kC);

  // this wave's loads of a matrix: 1 KB blocks of 1024 / ROW rows
  uint32_t off[L::LOADS];
#pragma unroll
  for (int i = 0; i < L::LOADS; ++i) {
    const int slot = 64 * (L::LOADS * w + i) + lane, row = slot / L::CH, chunk = (slot % L::CH) ^ row_swz(row);
    off[i] = 4 * chunk < d ? (uint32_t)(row * d + 4 * chunk) * 4u : kOOB;
  }
  const uint32_t lds0 = lds_u32(lds);
  auto issue = [&](int n, int stage) {
    const uint32_t sb = (uint32_t)n * (uint32_t)(kC * d * 4);  // the chunk's first row
    const uint32_t dst = lds0 + stage * STAGE + L::LOADS * w * 1024;
#pragma unroll
    for (int i = 0; i < L::LOADS; ++i) {
      // a column past d keeps its out-of-range offset (row offsets stay below 2^31)
      const uint32_t src = off[i] + sb;
      if (OUT) dma_buf(rq, src, dst + 2 * L::MAT + i * 1024);
      dma_buf(rk, src, dst + i * 1024);
      dma_buf(rv, src, dst + L::MAT + i * 1024);
    }
  };
  // X[l32][32 tile + 8 u + 4 g + e], e = 0 .. 3: inner index acc_row(4 u + e, g) of the tile
  auto row4 = [&](const char* X, int tile, int u) {
    return *reinterpret_cast<const f32x4*>(X + l32 * L::ROW + (((8 * tile + 2 * u + g) ^ row_swz(l32)) << 4));
  };
  // X[acc_row(t, g)][32 tile + l32]
  auto col1 = [&](const char* X, int tile, int t) {
    const int j = acc_row(t, g);
    return *reinterpret_cast<const float*>(X + j * L::ROW + (((8 * tile + (l32 >> 2)) ^ row_swz(j)) << 4) +
                                           4 * (l32 & 3));
  };

  if (c0 < c1) issue(c0, 0);
  f32x16 S[ND];  // S[32 tile + acc_row(r, g)][32 w + l32]
#pragma unroll
  for (int t = 0; t < ND; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) S[t][r] = 0.f;
  // a state piece in memory: 16 bytes per lane, lanes contiguous
  auto piece = [&](int64_t s) { return pieces + (bh * (P - 1) + s) * L::STATE + (w * ND * 4 * 64 + lane) * 4; };
  if (OUT) {  // 64 KB per segment before this one (ND = 4): about 2 us each, bound by one CU's load rate
    for (int s = 0; s < seg; ++s) {
      const float f = pow_k(lg, neg, kC * (int)(seg_first(nch, s + 1, P) - seg_first(nch, s, P)));
      const float* src = piece(s);
#pragma unroll
      for (int t = 0; t < ND; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(src + (4 * t + u) * 256);
#pragma unroll
          for (int e = 0; e < 4; ++e) S[t][4 * u + e] = __builtin_fmaf(f, S[t][4 * u + e], x[e]);
        }
    }
  }
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(o + base, (short)0, (int)bytes, 0x00020000);
  const uint32_t ocol = 32 * w + l32 < d ? (uint32_t)(32 * w + l32 + 4 * g * d) * 4u : kOOB;
  float* part = reinterpret_cast<float*>(lds + 2 * STAGE);
  __builtin_amdgcn_s_waitcnt(0);  // the first chunk: no stores behind its loads yet

  for (int n = c0; n < c1; ++n) {
    const int stage = (n - c0) & 1;
    // chunk n has landed (its loads are older than the 16 stores of the
    // chunk before), and every wave is done with the other half and with the
    // partial scores
    __builtin_amdgcn_s_waitcnt(OUT ? ((16 & 15) | (7 << 4) | ((16 >> 4) << 14)) : 0);
    __syncthreads();
    if (n + 1 < c1) issue(n + 1, stage ^ 1);
    const char* Ks = lds + stage * STAGE;
    const char* Vs = Ks + L::MAT;
    const char* Qs = Vs + L::MAT;
    float vr[16], kc[ND][16];
    f32x16 oacc;
    if (OUT) {
      f32x16 p, o2;
#pragma unroll
      for (int r = 0; r < 16; ++r) p[r] = oacc[r] = o2[r] = 0.f;
      f32x4 kf[4], qw[4], qf[ND][4], ps[ND][4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        kf[u] = row4(Ks, w, u);
        qw[u] = row4(Qs, w, u);
        qf[0][u] = row4(Qs, 0, u);
      }
      __builtin_amdgcn_sched_barrier(0);
      // scores Pᵀ[j, i] over this wave's q/k columns, and the inter-chunk
      // term's first tile
      stream<16>(
          [&](int x) {
            p = mfma_f32(kf[x >> 2][x & 3], qw[x >> 2][x & 3], p);
            oacc = mfma_f32(qf[0][x >> 2][x & 3], S[0][x], oacc);
          },
          [&](int x) {
            if (x % 4 == 0) qf[1][x >> 2] = row4(Qs, 1, x >> 2);
            if (ND == 4 && x % 4 == 2) qf[ND - 2][x >> 2] = row4(Qs, ND - 2, x >> 2);
          });
      // the partial scores go to LDS; the inter-chunk term's next tiles
      auto put = [&](int u) {
        *reinterpret_cast<f32x4*>(part + ((4 * w + u) * 64 + lane) * 4) =
            f32x4{p[4 * u], p[4 * u + 1], p[4 * u + 2], p[4 * u + 3]};
      };
      if (ND == 4) {
        stream<16>(
            [&](int x) {
              oacc = mfma_f32(qf[1][x >> 2][x & 3], S[1][x], oacc);
              o2 = mfma_f32(qf[ND - 2][x >> 2][x & 3], S[ND - 2][x], o2);
            },
            [&](int x) {
              if (x % 4 == 0) qf[ND - 1][x >> 2] = row4(Qs, ND - 1, x >> 2);
              if (x % 4 == 3) put(x >> 2);
            });
      } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) put(u);
      }
      __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (3 << 14));  // lgkmcnt 0
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
      // the last tile, while the partial scores come back from all waves
      stream<8>(
          [&](int x) {
            const int y = 2 * x;
            oacc = mfma_f32(qf[ND - 1][y >> 2][y & 3], S[ND - 1][y], oacc);
            o2 = mfma_f32(qf[ND - 1][y >> 2][(y & 3) + 1], S[ND - 1][y + 1], o2);
          },
          [&](int x) {
#pragma unroll
            for (int y = 2 * x; y < 2 * x + 2; ++y) {
              vr[y] = col1(Vs, w, y);
              if (y < 4 * ND) ps[y >> 2][y & 3] = *reinterpret_cast<const f32x4*>(part + (y * 64 + lane) * 4);
            }
          });
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        oacc[r] = (oacc[r] + o2[r]) * rowf[r];  // the per-row decay γ^a
        o2[r] = 0.f;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int y = 1; y < ND; ++y) ps[0][u] += ps[y][u];
#pragma unroll
        for (int e = 0; e < 4; ++e) ps[0][u][e] *= diagf[4 * u + e];
      }
      __builtin_amdgcn_sched_barrier(0);
      // intra-chunk term O += P V
      stream<8>(
          [&](int x) {
            const int y = 2 * x;
            oacc = mfma_f32(ps[0][y >> 2][y & 3], vr[y], oacc);
            o2 = mfma_f32(ps[0][y >> 2][(y & 3) + 1], vr[y + 1], o2);
          },
          [&](int x) {
#pragma unroll
            for (int y = 2 * x; y < 2 * x + 2; ++y) {
              kc[0][y] = col1(Ks, 0, y);
              kc[1][y] = col1(Ks, 1, y);
            }
          });
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[r] += o2[r];
    } else {
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        vr[x] = col1(Vs, w, x);
        kc[0][x] = col1(Ks, 0, x);
        kc[1][x] = col1(Ks, 1, x);
      }
    }
    // state update S ← γ^C S + kᵀ diag(γ^(C−b)) v (not read again past the last chunk)
    if (!OUT || n + 1 < c1) {
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        vr[x] *= wv[x];
        S[0][x] *= gC;
        S[1][x] *= gC;
      }
#pragma unroll
      for (int t = 0; t < ND; t += 2) {
        __builtin_amdgcn_sched_barrier(0);
        stream<16>(
            [&](int x) {
              S[t] = mfma_f32(kc[t][x], vr[x], S[t]);
              S[t + 1] = mfma_f32(kc[t + 1][x], vr[x], S[t + 1]);
            },
            [&](int x) {
#pragma unroll
              for (int y = t + 2; y < t + 4 && y < ND; ++y) {
                kc[y][x] = col1(Ks, y, x);
                S[y][x] *= gC;
              }
            });
      }
    }
    if (OUT) {
      const uint32_t sb = (uint32_t)n * (uint32_t)(kC * d * 4);
#pragma unroll
      for (int r = 0; r < 16; ++r)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, scale * oacc[r]), ro,
                                              (int)(ocol + sb + (uint32_t)((8 * (r >> 2) + (r & 3)) * d * 4)), 0, 0);
    }
  }
  if (!OUT) {
    float* dst = piece(seg);
#pragma unroll
    for (int t = 0; t < ND; ++t)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        *reinterpret_cast<f32x4*>(dst + (4 * t + u) * 256) =
            f32x4{S[t][4 * u], S[t][4 * u + 1], S[t][4 * u + 2], S[t][4 * u + 3]};
  }
}

// Segments per head: one workgroup per CU (two at ND = 2, whose LDS is half),
// at least two chunks each; past 16 the fold of the start state costs what
// the shorter segments give.
int64_t n_segments(int64_t BH, int64_t T, int64_t d) {
  const int64_t slots = d > 64 ? 256 : 512, nch = (T + kC - 1) / kC;
  int64_t P = BH > 0 ? slots / BH : 1;
  if (P > kMaxSeg) P = kMaxSeg;
  if (P > nch / 2) P = nch / 2;
  return P < 1 ? 1 : P;
}

template <int ND>
int32_t launch(int64_t BH, int64_t H, int64_t T, int64_t d, const float* q, const float* k, const float* v,
               const float* gamma, float scale, float* o, float* ws, int64_t P, hipStream_t s) {
  using L = Ret<ND>;
  constexpr int LDS_STATE = 4 * L::MAT, LDS_OUT = 6 * L::MAT + ND * 4096;
  static bool attr_done = false;  // idempotent; benign race (same value written)
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&retention_f32<ND, true>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, LDS_OUT);
    if (e != hipSuccess) return set_hip_error(e);
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(&retention_f32<ND, false>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, LDS_STATE);
    if (e != hipSuccess) return set_hip_error(e);
    attr_done = true;
  }
  if (P > 1) {
    retention_f32<ND, false><<<dim3((uint32_t)(BH * (P - 1))), dim3(L::NT), LDS_STATE, s>>>(
        q, k, v, gamma, scale, o, ws, (int)H, (int)T, (int)d, (int)P);
    CATOPT_LAUNCH_CHECK();
  }
  retention_f32<ND, true><<<dim3((uint32_t)(BH * P)), dim3(L::NT), LDS_OUT, s>>>(q, k, v, gamma, scale, o, ws, (int)H,
                                                                                (int)T, (int)d, (int)P);
  CATOPT_LAUNCH_CHECK();
  return CATOPT_OK;
}

}  // namespace

int64_t retention_f32_workspace(int64_t B, int64_t H, int64_t T, int64_t d) {
  const int64_t P = n_segments(B * H, T, d);
  return B * H * (P - 1) * (d > 64 ? Ret<4>::STATE : Ret<2>::STATE) * (int64_t)sizeof(float);
}

int32_t retention_f32_launch(int64_t B, int64_t H, int64_t T, int64_t d, const float* q, const float* k,
                             const float* v, const float* gamma, float scale, float* o, void* ws, int64_t ws_bytes,
                             hipStream_t s) {
  if (d < 1 || d > 128 || d % 4) return CATOPT_E_UNSUPPORTED;
  if (T * d * 4 + 2 * (int64_t)kC * d * 4 > 0x7fffffffLL) return CATOPT_E_UNSUPPORTED;  // 32-bit buffer offsets
  if (B * H > 0x7fffffffLL) return CATOPT_E_UNSUPPORTED;  // more segments than one: B H <= 256
  int64_t P = n_segments(B * H, T, d);
  if (P > 1 && (!ws || !aligned16(ws) || ws_bytes < retention_f32_workspace(B, H, T, d))) P = 1;
  float* pieces = static_cast<float*>(ws);
  return d > 64 ? launch<4>(B * H, H, T, d, q, k, v, gamma, scale, o, pieces, P, s)
                : launch<2>(B * H, H, T, d, q, k, v, gamma, scale, o, pieces, P, s);
}

}  // namespace catopt
