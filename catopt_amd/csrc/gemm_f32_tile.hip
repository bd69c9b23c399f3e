// fp32 GEMM tiles on the 32x32x2 fp32 MFMA: C[b] = epi(op(A[b]) op(B[b])).
//
// The fp32 MFMA takes 64 cycles for 4 KB of products, so a 64 x 64 tile needs
// 16 KB of operands per 1024 cycles and neither LDS nor L2 is near its rate:
// all that is asked of the loop is that loads are wide and never waited for.
// (The general kernel of gemm.hip loads element by element between two
// barriers.  4096 x 512 x 512: 97 us there, 21 here, 102 TFLOP/s;
// 2048 x 2048 x 2048 400 and 146.)
//
// A workgroup is 4 waves in a 2 x 2 grid, one 32 x 32 block each.  K runs in
// stages of 32 through three LDS slots filled by direct global->LDS loads two
// stages ahead, one barrier per stage; three workgroups share a CU.
//
// Operands are taken as they lie.  K-contiguous (linear's X and W): 128-byte
// rows of 32 k, 16-byte chunks XOR-swizzled by (row / 2) % 8; lane l reads 4
// consecutive k of row l % 32 with one 16-byte read (k 8 s + 4 (l / 32) + e
// for MFMA e: the k index is a summation order, the same on both sides).
// K-strided (a product's plain B, or A transposed): 256-byte rows of 64
// columns, one per k; lane l reads its column in the same four k rows with
// 4-byte reads, the two lane halves on different banks by a swizzle of 32
// columns.  B feeds the MFMA's A operand, so accumulator register r of lane l
// is C[m = l % 32][n = acc_row(r, l / 32)] of the block: 16-byte stores.
#include "common.hpp"
#include "gemm_bf16.hpp"

namespace catopt {
namespace {

constexpr int FT = 64, FK = 32, FNT = 256, FSTAGES = 3;
constexpr int OPERAND_BYTES = FT * FK * 4, FSTAGE = 2 * OPERAND_BYTES;  // 8 KB each

// One operand's loads of a workgroup: 64 rows (m or n) of a stage.
template <bool KSTRIDED>
struct F32Operand {
  u32x4 rsrc;
  uint32_t off[2];  // this wave's two 1 KB blocks
  int kfirst[2];    // the k (K-contiguous) or k row (K-strided) of a lane's chunk in its stage
  uint32_t stage_bytes;

  __device__ __forceinline__ void setup(const float* base, int64_t ld, int row0, int rows, int K, int wave, int lane) {
    if (KSTRIDED) {  // element (k, row) at base + k ld + row; block i: k rows 8 wave + 4 i .. + 3
      const int64_t span = (int64_t)(K - 1) * ld + rows;
      rsrc = make_rsrc(base, (uint32_t)(span * 4));
      stage_bytes = (uint32_t)(FK * ld * 4);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int kr = 8 * wave + 4 * i + (lane >> 4);
        const int chunk = (lane & 15) ^ (8 * ((kr >> 2) & 1));
        const int col = row0 + 4 * chunk;
        kfirst[i] = col < rows ? kr : 0x40000000;  // columns past the matrix read out of range
        off[i] = (uint32_t)(((int64_t)kr * ld + col) * 4);
      }
    } else {
      const int lim = min(rows - 1 - row0, FT - 1);
      rsrc = make_rsrc(base + (int64_t)row0 * ld, (uint32_t)(((int64_t)lim * ld + K) * 4));
      stage_bytes = FK * 4;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = 16 * wave + 8 * i + (lane >> 3);
        kfirst[i] = 4 * ((lane & 7) ^ ((row >> 1) & 7));
        off[i] = (uint32_t)(((int64_t)min(row, lim) * ld + kfirst[i]) * 4);
      }
    }
  }
  // stage T into LDS at `dst`; k past K reads out of range: zeros
  __device__ __forceinline__ void load(int T, int K, int wave, uint32_t dst) const {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      dma_buf(rsrc, T * FK + kfirst[i] < K ? off[i] + (uint32_t)T * stage_bytes : 0x80000000u,
              dst + (2 * wave + i) * 1024);
  }
};

// Four k of row `row` of a stage: k = 8 s + 4 g + e, e = 0 .. 3.
template <bool KSTRIDED>
__device__ __forceinline__ f32x4 f32_frag(const char* lds, int row, int s, int g) {
  if (!KSTRIDED) return *reinterpret_cast<const f32x4*>(lds + swz(row, 2 * s + g));
  f32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    r[e] = *reinterpret_cast<const float*>(lds + (8 * s + 4 * g + e) * 256 + ((row ^ (32 * g)) * 4));
  return r;
}

template <bool TA, bool TB, int EPI>
__global__ __launch_bounds__(FNT, 2) void gemm_f32_tile(
    const float* __restrict__ A, int64_t lda, int64_t sA, const float* __restrict__ B, int64_t ldb, int64_t sB,
    const float* __restrict__ bias, const float* __restrict__ bias2, float* __restrict__ C, int64_t ldc, int64_t sC,
    int M, int N, int K, int tiles_m, int tiles_n, int vec_store) {
  __shared__ __attribute__((aligned(16))) char lds[FSTAGES * FSTAGE];
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  A += (int64_t)blockIdx.y * sA;
  B += (int64_t)blockIdx.y * sB;
  C += (int64_t)blockIdx.y * sC;
  // an XCD takes a contiguous run of tiles (8 M-tiles at a time)
  const int per = gridDim.x >> 3, rem = gridDim.x & 7, xcd = blockIdx.x & 7;
  const TileMap t = tile_of(xcd * per + min(xcd, rem) + (int)(blockIdx.x >> 3), tiles_m, tiles_n);
  const int m0 = t.tm * FT, n0 = t.tn * FT;
  F32Operand<TA> oa;   // TA: A stored K x M
  F32Operand<!TB> ob;  // TB: B stored N x K
  oa.setup(A, lda, m0, M, K, wave, lane);
  ob.setup(B, ldb, n0, N, K, wave, lane);
  const uint32_t lds0 = lds_u32(lds);
  const int kst = (K + FK - 1) / FK;
  // past the last stage: out of range, into a slot that is not read again, so
  // that every stage issues the same loads
  auto load = [&](int T, int slot) {
    oa.load(T, K, wave, lds0 + slot * FSTAGE);
    ob.load(T, K, wave, lds0 + slot * FSTAGE + OPERAND_BYTES);
  };
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
  for (int p = 0; p < FSTAGES - 1; ++p) load(p, p);
  int slot = 0;
  for (int T = 0; T < kst; ++T) {
    wait_vm_lgkm0<(FSTAGES - 2) * 4>();
    __syncthreads();  // stage T has landed for every wave, and the slot before it is free
    load(T + FSTAGES - 1, slot == 0 ? FSTAGES - 1 : slot - 1);
    const char* as = lds + slot * FSTAGE;
    const char* bs = as + OPERAND_BYTES;
    f32x4 af[4], bf[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      bf[s] = f32_frag<!TB>(bs, 32 * wn + l32, s, g);
      af[s] = f32_frag<TA>(as, 32 * wm + l32, s, g);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(bf[s][e], af[s][e], acc, 0, 0, 0);
    slot = slot == FSTAGES - 1 ? 0 : slot + 1;
  }
  __builtin_amdgcn_s_waitcnt(0);  // the loads past the last stage have landed

  const int m = m0 + 32 * wm + l32;
  if (m >= M) return;
#pragma unroll
  for (int rg = 0; rg < 4; ++rg) {
    const int n = n0 + 32 * wn + 8 * rg + 4 * g;
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int nn = min(n + e, N - 1);
      o[e] = acc[4 * rg + e];
      if (EPI == CATOPT_EPI_BIAS || EPI == CATOPT_EPI_BIAS_ADD2) o[e] += bias[nn];
      if (EPI == CATOPT_EPI_BIAS_ADD2) o[e] += bias2[nn];
    }
    float* dst = C + (int64_t)m * ldc + n;
    if (vec_store && n + 3 < N) {
      *reinterpret_cast<f32x4*>(dst) = o;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) dst[e] = o[e];
    }
  }
}

template <bool TA, bool TB, int EPI>
int32_t launch_f32(const float* A, int64_t lda, int64_t sA, const float* B, int64_t ldb, int64_t sB,
                   const float* bias, const float* bias2, float* C, int64_t ldc, int64_t sC, int64_t batch, int M,
                   int N, int K, hipStream_t s) {
  const int tiles_m = (M + FT - 1) / FT, tiles_n = (N + FT - 1) / FT;
  const int vec_store = ldc % 4 == 0 && sC % 4 == 0 && aligned16(C);
  gemm_f32_tile<TA, TB, EPI><<<dim3((uint32_t)(tiles_m * tiles_n), (uint32_t)batch), dim3(FNT), 0, s>>>(
      A, lda, sA, B, ldb, sB, bias, bias2, C, ldc, sC, M, N, K, tiles_m, tiles_n, vec_store);
  CATOPT_LAUNCH_CHECK();
  return CATOPT_OK;
}

// An operand of `rows` rows: 16-byte chunks aligned and wholly in or out, offsets below 2^31.
bool operand_ok(const void* p, int64_t ld, int64_t stride, int64_t rows, int64_t K, bool kstrided) {
  if (!aligned16(p) || ld % 4 || stride % 4) return false;
  if (kstrided) return rows % 4 == 0 && ((K + FK * FSTAGES) * ld + rows + FT) * 4 < 0x7fffffffLL;
  return K % 4 == 0 && (FT * ld + K + FK * FSTAGES) * 4 < 0x7fffffffLL;
}

}  // namespace

bool gemm_f32_tile_ok(int64_t batch, int64_t M, int64_t N, int64_t K, const void* A, int64_t lda, int64_t sA, bool ta,
                      const void* B, int64_t ldb, int64_t sB, bool tb) {
  const int64_t tiles = ((M + FT - 1) / FT) * ((N + FT - 1) / FT);
  return grid_fits(tiles, FNT) && batch <= 65535 && M < 0x40000000LL && N < 0x40000000LL && K < 0x40000000LL &&
         operand_ok(A, lda, sA, M, K, ta) && operand_ok(B, ldb, sB, N, K, !tb);
}

int32_t gemm_f32_tile_launch(int32_t epi, int64_t batch, int64_t M, int64_t N, int64_t K, const float* A, int64_t lda,
                             int64_t sA, bool ta, const float* B, int64_t ldb, int64_t sB, bool tb, const float* bias,
                             const float* bias2, float* C, int64_t ldc, int64_t sC, hipStream_t s) {
#define CATOPT_F32(TA, TB, E) \
  launch_f32<TA, TB, E>(A, lda, sA, B, ldb, sB, bias, bias2, C, ldc, sC, batch, (int)M, (int)N, (int)K, s)
  if (epi == CATOPT_EPI_BIAS && !ta && tb) return CATOPT_F32(false, true, CATOPT_EPI_BIAS);
  if (epi == CATOPT_EPI_BIAS_ADD2 && !ta && tb) return CATOPT_F32(false, true, CATOPT_EPI_BIAS_ADD2);
  if (epi != CATOPT_EPI_NONE) return CATOPT_E_INVAL;
  if (!ta) return tb ? CATOPT_F32(false, true, CATOPT_EPI_NONE) : CATOPT_F32(false, false, CATOPT_EPI_NONE);
  return tb ? CATOPT_F32(true, true, CATOPT_EPI_NONE) : CATOPT_F32(true, false, CATOPT_EPI_NONE);
#undef CATOPT_F32
}

}  // namespace catopt
