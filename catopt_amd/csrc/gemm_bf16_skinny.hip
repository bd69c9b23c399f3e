// bf16 "NT" GEMM for few rows (M <= 64): C[m, n] = epi(sum_k X[m, k] W[n, k]).
//
// With few rows the product streams W once and does little with it (at M = 8,
// 8 flop per byte of W), so HBM is the bound and what counts is how many
// bytes of W are in flight.  The 256 x 256 tiles of gemm_bf16.hip give such a
// call one workgroup per 256 weight rows: 16 workgroups for a 4096-wide
// projection, each walking all of K by itself (195 us at 8 x 11008 -> 4096,
// 0.46 TB/s).  Here a workgroup owns 16 weight rows (paired epilogues: 16 of
// each projection) and its waves split K, so the same call has 256
// workgroups: 22.6 us (4.0 TB/s; a device copy moves 4.9).
//
// The waves take 64-wide K chunks in turn (wave w chunks w, w + WAVES, ...),
// so the workgroup reads runs of WAVES x 128 bytes of each weight row.  Both
// operands go straight from memory into the 16x16x32 MFMA's operand layout
// (lane l: row l % 16, 8 consecutive k of group l / 16), UNROLL chunks of
// loads in flight per wave before the first product.  No operand passes through LDS: W is used by one wave only, and
// X's few rows come from L2.  Loads go through buffer resources: k past K
// reads as zero (both operands, so that no Inf or NaN of a neighbouring row
// meets a zero), rows past M or N read a clamped, valid row whose results
// are not stored.  The partial sums are added through LDS in wave order
// (deterministic), then the epilogue runs once.
//
// W rows feed the MFMA's A operand, so accumulator register r of lane l is
// C[16 mb + l % 16][n0 + 4 (l / 16) + r].
#include "common.hpp"
#include "gemm_bf16.hpp"

namespace catopt {
namespace {

constexpr int SKN = 16;       // weight rows per workgroup (per projection)
constexpr int SKC = 64;       // K per chunk: one cache line of a row
constexpr uint32_t kOutOfRange = 0x80000000u;

__device__ __forceinline__ bf16x8 load8(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}

// Waves per workgroup and 64-wide chunks in flight per wave, by 16-row blocks
// MB and projections NP.  At 11008 -> 4096 with 1 / 16 rows: 16 waves x 2
// chunks 21.1 / 24.6 us, 8 x 4 22.0 / 25.4, 8 x 8 23.3 / 26.3; paired
// 4096 -> 2 x 11008: 16 x 1 34.5 / 38.7, 8 x 2 34.6 / 40.9.  At three and four
// blocks the 16 partial sums would not fit 64 KB of LDS.
constexpr int rows_waves(int mb) { return mb <= 2 ? 16 : 8; }
constexpr int rows_unroll(int mb, int np) { return mb <= 2 && np == 2 ? 1 : 2; }

template <int EPI, int MB>
__global__ __launch_bounds__(64 * rows_waves(MB)) void gemm_bf16_rows(
    const uint16_t* __restrict__ X, int64_t ldx, const uint16_t* __restrict__ W, int64_t ldw,
    const uint16_t* __restrict__ bias, const uint16_t* __restrict__ bias2, uint16_t* __restrict__ C,
    int64_t ldc, int M, int N, int K, int64_t sX, int64_t sW, int64_t sC, int vec_store) {
  constexpr bool PAIRED = (EPI == CATOPT_EPI_SILU_MUL || EPI == CATOPT_EPI_GLU);
  constexpr int NP = PAIRED ? 2 : 1;
  constexpr int WAVES = rows_waves(MB), UNROLL = rows_unroll(MB, NP);
  __shared__ __attribute__((aligned(16))) f32x4 part[WAVES][NP * MB][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * SKN;
  X += (int64_t)blockIdx.y * sX;
  W += (int64_t)blockIdx.y * sW;
  C += (int64_t)blockIdx.y * sC;

  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(X), (short)0, (int)(((int64_t)(M - 1) * ldx + K) * 2), 0x00020000);
  __amdgpu_buffer_rsrc_t rw[NP];
  const int nlim = min(N - 1 - n0, SKN - 1);
#pragma unroll
  for (int p = 0; p < NP; ++p)
    rw[p] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(W + ((int64_t)n0 + (p ? (int64_t)N : 0)) * ldw), (short)0,
        (int)(((int64_t)nlim * ldw + K) * 2), 0x00020000);
  const uint32_t wrow = (uint32_t)(min(r16, nlim) * ldw * 2) + kg * 16;
  uint32_t xrow[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) xrow[mb] = (uint32_t)(min(16 * mb + r16, M - 1) * ldx * 2) + kg * 16;

  f32x4 acc[NP][MB];
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[p][mb] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nch = (K + SKC - 1) / SKC;
  for (int c0 = wave; c0 < nch; c0 += WAVES * UNROLL) {
    bf16x8 wf[UNROLL][2][NP], xf[UNROLL][2][MB];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = (c0 + WAVES * u) * SKC + 32 * h;  // this lane's first k is k + 8 kg
        const bool ok = k + 8 * kg < K;               // K % 8 == 0: a lane's 8 are wholly in or out
#pragma unroll
        for (int p = 0; p < NP; ++p) wf[u][h][p] = load8(rw[p], ok ? wrow + 2 * k : kOutOfRange);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) xf[u][h][mb] = load8(rx, ok ? xrow[mb] + 2 * k : kOutOfRange);
      }
    __builtin_amdgcn_sched_barrier(0);  // every load of the pass before its first product
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb)
            acc[p][mb] = mfma16(wf[u][h][p], xf[u][h][mb], acc[p][mb]);
  }
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) part[wave][p * MB + mb][lane] = acc[p][mb];
  __syncthreads();

  // wave mb sums and stores block mb: lane l's four columns of one row
  if (wave >= MB) return;
  f32x4 s[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    s[p] = part[0][p * MB + wave][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) s[p] += part[w][p * MB + wave][lane];
  }
  const int m = 16 * wave + r16, n = n0 + 4 * kg;
  if (m >= M || n >= N) return;
  float o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int nn = min(n + r, N - 1);
    const float b1 = EPI == CATOPT_EPI_BIAS || EPI == CATOPT_EPI_BIAS_ADD2 ? bf16_to_f32(bias[nn]) : 0.f;
    const float b2 = EPI == CATOPT_EPI_BIAS_ADD2 ? bf16_to_f32(bias2[nn]) : 0.f;
    o[r] = epilogue_value<EPI>(s[0][r], s[NP - 1][r], b1, b2);
  }
  uint16_t* dst = C + (int64_t)m * ldc + n;
  if (vec_store && n + 3 < N) {
    *reinterpret_cast<u32x2*>(dst) = u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < N) dst[r] = f32_to_bf16(o[r]);
  }
}

template <int EPI>
int32_t launch_rows(const uint16_t* X, int64_t ldx, const uint16_t* W, int64_t ldw, const uint16_t* bias,
                    const uint16_t* bias2, uint16_t* C, int64_t ldc, int M, int N, int K, int64_t batch,
                    int64_t sX, int64_t sW, int64_t sC, hipStream_t s) {
  if (batch > 65535) return CATOPT_E_UNSUPPORTED;
  const dim3 grid((uint32_t)((N + SKN - 1) / SKN), (uint32_t)batch), block(64 * rows_waves((M + 15) / 16));
  const int vec_store = ldc % 4 == 0 && sC % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 7) == 0;
#define CATOPT_ROWS(MB)                                                                                    \
  gemm_bf16_rows<EPI, MB><<<grid, block, 0, s>>>(X, ldx, W, ldw, bias, bias2, C, ldc, M, N, K, sX, sW, sC, \
                                                 vec_store)
  switch ((M + 15) / 16) {
    case 1: CATOPT_ROWS(1); break;
    case 2: CATOPT_ROWS(2); break;
    case 3: CATOPT_ROWS(3); break;
    case 4: CATOPT_ROWS(4); break;
    default: return CATOPT_E_INVAL;
  }
#undef CATOPT_ROWS
  CATOPT_LAUNCH_CHECK();
  return CATOPT_OK;
}

}  // namespace

bool gemm_bf16_rows_ok(int64_t M, int64_t N) {
  return M <= 64 && grid_fits((N + SKN - 1) / SKN, 64 * rows_waves((int)((M + 15) / 16)));
}

int32_t gemm_bf16_rows_launch(int32_t epi, int64_t M, int64_t N, int64_t K, const void* x, int64_t ldx,
                              const void* w, int64_t ldw, const void* bias, const void* bias2, void* y,
                              int64_t ldy, int64_t batch, int64_t sX, int64_t sW, int64_t sC,
                              hipStream_t s) {
  auto A = static_cast<const uint16_t*>(x);
  auto B = static_cast<const uint16_t*>(w);
  auto b1 = static_cast<const uint16_t*>(bias);
  auto b2 = static_cast<const uint16_t*>(bias2);
  auto C = static_cast<uint16_t*>(y);
#define CATOPT_EPI_CASE(E) \
  case E: return launch_rows<E>(A, ldx, B, ldw, b1, b2, C, ldy, (int)M, (int)N, (int)K, batch, sX, sW, sC, s);
  switch (epi) {
    CATOPT_EPI_CASE(CATOPT_EPI_NONE)
    CATOPT_EPI_CASE(CATOPT_EPI_BIAS)
    CATOPT_EPI_CASE(CATOPT_EPI_BIAS_ADD2)
    CATOPT_EPI_CASE(CATOPT_EPI_SILU_MUL)
    CATOPT_EPI_CASE(CATOPT_EPI_GLU)
    default: return CATOPT_E_INVAL;
  }
#undef CATOPT_EPI_CASE
}

}  // namespace catopt
