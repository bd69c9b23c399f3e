// What the bf16 "NT" GEMM kernels share: the LDS row swizzle, waits, the
// MFMA, the epilogue of a wave's accumulator blocks, and the launchers'
// declarations.
#pragma once
#include "common.hpp"

namespace catopt {

constexpr int ROW_BYTES = 128;  // one tile row of a K stage of 64: one cache line

// Byte offset of (row, 16-byte chunk) in a tile of ROW_BYTES rows.
__device__ __forceinline__ constexpr int swz(int row, int chunk) {
  return row * ROW_BYTES + ((chunk ^ ((row >> 1) & 7)) << 4);
}

// s_waitcnt with lgkmcnt(0) and vmcnt <= n (gfx9 encoding; expcnt not waited on).
template <int n>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(n >= 0 && n < 64, "vmcnt field");
  __builtin_amdgcn_s_waitcnt((n & 15) | (7 << 4) | ((n >> 4) << 14));
}
__device__ __forceinline__ void wait_lgkm0() { __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (3 << 14)); }

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

struct TileMap {
  int tm, tn;
};

// Logical tile -> (M-tile, N-tile): groups of 8 M-tiles, N-tiles in order.
__device__ __forceinline__ TileMap tile_of(int lt, int tiles_m, int tiles_n) {
  constexpr int GM = 8;
  const int per_group = GM * tiles_n;
  const int group = lt / per_group;
  const int first_m = group * GM;
  const int gsize = min(tiles_m - first_m, GM);
  const int in_group = lt - group * per_group;
  TileMap t;
  t.tm = first_m + in_group % gsize;
  t.tn = in_group / gsize;
  return t;
}

// One output value from its sum `a` (paired: `b` the second projection's).
template <int EPI>
__device__ __forceinline__ float epilogue_value(float a, float b, float bias, float bias2) {
  if constexpr (EPI == CATOPT_EPI_SILU_MUL) return a * __builtin_amdgcn_rcpf(1.0f + __expf(-a)) * b;
  if constexpr (EPI == CATOPT_EPI_GLU) return a * __builtin_amdgcn_rcpf(1.0f + __expf(-b));
  if constexpr (EPI == CATOPT_EPI_BIAS_ADD2) return (a + bias) + bias2;
  return a + bias;
}

// Stores a wave's blocks.  acc[i][j][r] is C[m][n] with m = mrow + 16 j
// (mrow: this lane's row of block 0) and n = (first column of block i) +
// 4 (l / 16) + r; the wave's columns start at nw and its blocks are 16 wide
// (paired: blocks 0-1 the first projection's, 2-3 the second's).  Adjacent
// blocks i, i+1 trade halves between lane rows (v_permlane16_swap) so each
// lane holds 8 consecutive columns: one 16-byte store per lane, 64 contiguous
// bytes per output row (8-byte stores of 32-byte row pieces cost 2-7% more
// kernel time).
template <int EPI, int FM>
__device__ __forceinline__ void gemm_epilogue(const f32x4 (&acc)[4][FM], int mrow, int nw, int M, int N,
                                              const uint16_t* bias, const uint16_t* bias2, uint16_t* C,
                                              int64_t ldc, int vec_store) {
  constexpr bool PAIRED = (EPI == CATOPT_EPI_SILU_MUL || EPI == CATOPT_EPI_GLU);
  const int q = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int i = 0; i < (PAIRED ? 2 : 4); i += 2) {
    const int nb = nw + i * 16;
    float bv[2][4], bv2[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = nb + 16 * h + 4 * q + r;
        bv[h][r] = (EPI == CATOPT_EPI_BIAS || EPI == CATOPT_EPI_BIAS_ADD2) && n < N ? bf16_to_f32(bias[n]) : 0.f;
        bv2[h][r] = (EPI == CATOPT_EPI_BIAS_ADD2) && n < N ? bf16_to_f32(bias2[n]) : 0.f;
      }
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      uint32_t pk[2][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          o[r] = epilogue_value<EPI>(acc[i + h][j][r], PAIRED ? acc[(i + h + 2) & 3][j][r] : 0.f, bv[h][r], bv2[h][r]);
        pk[h][0] = pack_bf16x2(o[0], o[1]);
        pk[h][1] = pack_bf16x2(o[2], o[3]);
      }
      // rows q = 1, 3 take block i+1 columns 0-3 / 8-11 of rows 0, 2 and
      // give them their block i columns 4-7 / 12-15
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        auto sw = __builtin_amdgcn_permlane16_swap(pk[0][w], pk[1][w], false, false);
        pk[0][w] = sw[0];
        pk[1][w] = sw[1];
      }
      const int m = mrow + 16 * j;
      const int n = nb + 16 * (q & 1) + 8 * (q >> 1);
      if (m >= M || n >= N) continue;
      uint16_t* dst = C + (int64_t)m * ldc + n;
      if (vec_store && n + 7 < N) {
        *reinterpret_cast<u32x4*>(dst) = u32x4{pk[0][0], pk[0][1], pk[1][0], pk[1][1]};
      } else {
        const uint32_t wv[4] = {pk[0][0], pk[0][1], pk[1][0], pk[1][1]};
#pragma unroll
        for (int r = 0; r < 8; ++r)
          if (n + r < N) dst[r] = (uint16_t)(wv[r >> 1] >> (16 * (r & 1)));
      }
    }
  }
}

// ------------------------------------------------------------------ launchers

// The current device's CU count.
int32_t gemm_cu_count(int* out);

// Whether the bf16 kernels take these operands (K-contiguous, 16-byte
// aligned, 32-bit offsets within a tile's rows).
bool gemm_bf16_nt_fast_ok(int64_t M, int64_t N, int64_t K, const void* x, int64_t ldx,
                          const void* w, int64_t ldw, const void* y, int64_t ldy);

// Runs one product (or a batch) on the kernel its sizes call for; `ws` may be
// null (then no tile's K is split).
int32_t gemm_bf16_nt_launch(int32_t epi, int64_t M, int64_t N, int64_t K, const void* x,
                            int64_t ldx, const void* w, int64_t ldw, const void* bias,
                            const void* bias2, void* y, int64_t ldy, int64_t batch,
                            int64_t strideA, int64_t strideB, int64_t strideC, void* ws,
                            int64_t ws_bytes, hipStream_t s);

// Few rows, M <= 64 (gemm_bf16_skinny.hip), where its grid can be launched.
bool gemm_bf16_rows_ok(int64_t M, int64_t N);
int32_t gemm_bf16_rows_launch(int32_t epi, int64_t M, int64_t N, int64_t K, const void* x, int64_t ldx,
                              const void* w, int64_t ldw, const void* bias, const void* bias2, void* y,
                              int64_t ldy, int64_t batch, int64_t sX, int64_t sW, int64_t sC,
                              hipStream_t s);

// The kernel that runs one product (gemm_bf16_mid.hip): the large tiles
// (NONE), the few-rows kernel, or a middle tile shape with the tiles done
// whole (a multiple of the workgroups per round, or all of them) and the K
// ranges of each other tile.
enum { GEMM_MID_NONE = 0, GEMM_ROWS, GEMM_MID_128x256, GEMM_MID_64x128 };
struct GemmMidPlan {
  int shape, direct, round, splits;
};
// The plan of a launch with `ws_bytes` of workspace (0: none).
GemmMidPlan gemm_bf16_plan(int64_t batch, int64_t M, int64_t N, int64_t K, bool paired, int n_cu, int64_t ws_bytes);
int64_t gemm_bf16_mid_workspace(const GemmMidPlan& p, int64_t M, int64_t N, bool paired);
int32_t gemm_bf16_mid_launch(const GemmMidPlan& plan, int32_t epi, int64_t M, int64_t N, int64_t K, const void* x,
                             int64_t ldx, const void* w, int64_t ldw, const void* bias, const void* bias2, void* y,
                             int64_t ldy, void* ws, hipStream_t s);

// fp32 tiles (gemm_f32_tile.hip).  ta: A stored K x M; tb: B stored N x K.
bool gemm_f32_tile_ok(int64_t batch, int64_t M, int64_t N, int64_t K, const void* A, int64_t lda, int64_t sA, bool ta,
                      const void* B, int64_t ldb, int64_t sB, bool tb);
int32_t gemm_f32_tile_launch(int32_t epi, int64_t batch, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda,
                             int64_t sA, bool ta, const float* B, int64_t ldb, int64_t sB, bool tb, const float* bias,
                             const float* bias2, float* C, int64_t ldc, int64_t sC, hipStream_t s);

}  // namespace catopt
