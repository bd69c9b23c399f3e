// bf16 "NT" GEMM on gfx950 MFMA with fused epilogues: a persistent
// ping-pong kernel.
//
//   C[m, n] = epi( sum_k X[m, k] * W[n, k] )
//
// X is the activation (rows of length K, K contiguous), W the weight in
// nn.Linear layout (out_features x in_features, K contiguous): both operands
// are K-contiguous, the layout the 16x16x32 bf16 MFMA consumes directly (each
// lane supplies 8 consecutive k of one row).  W rows feed the MFMA's A
// operand and X rows its B operand, so a lane's accumulators hold four
// consecutive output columns n of one row m; the epilogue trades halves of
// adjacent blocks between lane rows (v_permlane16_swap) so that each lane
// stores 8 consecutive columns with one 16-byte store.
//
// Tiling: a 256 (m) x 256 (n) output tile per workgroup of 8 waves, two per
// SIMD.  Wave w owns m rows [128 (w / 4), +128) and n columns [64 (w % 4),
// +64): 8 x 4 MFMA blocks of 16 x 16, 128 accumulator registers.
//
// Schedule.  The waves form two groups, 0-3 and 4-7, one wave of each per
// SIMD.  Phases are separated by workgroup barriers; in each phase one group
// computes and the other does memory work, and group 1 runs one phase behind
// group 0, so on every SIMD one wave issues MFMAs back to back while its
// partner reads its next fragments.  A K stage of 64 is two steps of 32:
//   memory phase, first step:  read the wave's 12 fragments of the step
//     from LDS (ds_read_b128) and issue 4 global->LDS loads of the wave's W
//     rows of the next stage;
//   memory phase, second step:  read the fragments, issue 4 loads of the
//     wave's X rows two stages ahead, wait for every load but those 4;
//   compute phase:  32 MFMAs over the fragment registers, nothing else.
// LDS holds ten 16 KB slots (160 KB): a ring of 3 stages for each group's
// 128 X rows and a ring of 2 stages for the 256 W rows.  Each load goes
// into the slot of a stage that every wave finished reading in an earlier
// phase; the detailed slot schedule is written at the main loop.
//
// Persistent tiles: the grid is one workgroup per CU, and each workgroup
// walks its tiles in rounds.  The loads run one stage ahead across tile
// boundaries (the last stage of a tile prefetches the first of the next),
// and a tile's epilogue is issued in the first memory phase of the next
// tile, so the stores overlap the next tile's MFMAs instead of all
// workgroups storing at once.
//
// Loads go global->LDS directly (buffer_load_dwordx4 ... lds) through buffer
// resources over the tile's rows, issued as inline asm: the compiler then
// places no vmcnt wait of its own in front of the fragment reads (it cannot
// tell which stage a pending load writes), and the explicit waits are the
// only ones.  Each load moves 8 rows x 128 bytes, whole cache lines (a
// 64-byte row per load costs about 10% more time).  Rows past M or N read a
// clamped, valid row and are never stored; 16-byte chunks past K read out of
// the resource's range, which returns zeros.  Each 128-byte LDS row is
// XOR-swizzled by (row / 2) % 8 so that the 16 rows of a fragment read hit
// 16 distinct 16-byte bank groups.
//
// Paired epilogues (SILU_MUL / GLU): the W tile holds 128 rows of the first
// projection and the 128 matching rows of the second (row n and row n + N of
// the concatenated weight), and each wave owns 32 columns of both, so the
// gate is applied in registers and chunk / silu / mul never touch HBM.
//
// Tile order is XCD-aware: the hardware deals workgroups round robin over 8
// XCDs, so in each round the 32 workgroups of one XCD take a contiguous range
// of logical tiles (grouped 8 M-tiles at a time), which march through K
// together and share that XCD's L2.
#include "common.hpp"
#include "gemm_bf16.hpp"

namespace catopt {
namespace {

constexpr int BM = 256, BN = 256, BK = 64;     // tile; K per stage (two MFMA steps of 32)
constexpr int NT = 512;                        // 8 waves
constexpr int SLOT_ROWS = 128;                 // an LDS slot: 128 rows of one stage
constexpr int SLOT_BYTES = SLOT_ROWS * ROW_BYTES;  // 16 KB
// LDS slots: X rows 0-127 in a ring of 3 (read by waves 0-3), X rows
// 128-255 in a ring of 3 (waves 4-7), W rows 0-127 and 128-255 in a ring of
// 2 stages (read by all waves).
constexpr int X_RING = 3, W_RING = 2;
constexpr int W_SLOT0 = 2 * X_RING;
constexpr int N_SLOTS = 2 * X_RING + 2 * W_RING;
constexpr int LDS_BYTES = N_SLOTS * SLOT_BYTES;   // 160 KB
constexpr int DMA_PER_PHASE = 4;               // 1 KB loads per wave per compute phase
constexpr int FM = 8, FN = 4;                  // 16x16 blocks per wave along m, n
static_assert(BN == BM && LDS_BYTES <= 160 * 1024, "geometry");
static_assert(SLOT_BYTES / 1024 == 4 * DMA_PER_PHASE, "a group's 4 waves fill one slot per phase");

// The kernel's operands, shared by its helpers.
struct GemmArgs {
  const uint16_t* X;
  const uint16_t* W;
  int64_t lda, ldb;
  int M, N, K, tiles_m, tiles_n, nblocks, kst, G, slot;
};

// One load stream of a wave: the 128 rows of one matrix half that the wave's
// group loads, stage after stage, tile after tile.  `what` is 0 for X rows
// 128 h .. 128 h + 127 (h = `half`), 1 for W rows of half h (paired: h = 0 the
// gate rows, h = 1 the up rows).  Wave wq loads 1 KB blocks q = 4 wq + i
// (i < 4) of the 16 in a slot; block q covers slot rows 8 q .. 8 q + 7, lane
// l holds row 8 q + l / 8 and stored chunk l % 8, i.e. global chunk
// (l % 8) ^ ((q % 2) * 4 + l / 16).  Past the last tile the stream repeats
// its last stage (into a slot nobody reads again), so every wave issues the
// same loads every phase and the vmcnt bounds below stay exact.
template <bool PAIRED>
struct Stream {
  u32x4 rsrc;
  uint32_t voff[DMA_PER_PHASE];
  int what, half;  // 0: X rows 128 half.., 1: W rows of `half`
  int round, T;    // the stage this stream loads next
  bool live;       // a tile exists for `round`

  __device__ __forceinline__ void setup(const GemmArgs& g, int wq, int lane, const int* lchunk8) {
    const int lt = round * g.G + g.slot;
    live = lt < g.nblocks;
    if (!live) return;  // keep the last tile's resource and offsets
    const TileMap t = tile_of(lt, g.tiles_m, g.tiles_n);
    int64_t ld;
    int row0, row_lim;  // first tile row of the half; last valid tile row
    const uint16_t* base;
    if (what == 0) {
      const int m0 = t.tm * BM;
      base = g.X + (int64_t)m0 * g.lda;
      ld = g.lda;
      row0 = half * SLOT_ROWS;
      row_lim = min(g.M - 1 - m0, BM - 1);
    } else {
      const int n0 = t.tn * (PAIRED ? BN / 2 : BN);
      ld = g.ldb;
      if (PAIRED) {  // gate rows n0.. or up rows N + n0..
        base = g.W + ((int64_t)n0 + (half ? (int64_t)g.N : 0)) * g.ldb;
        row0 = 0;
        row_lim = min(g.N - 1 - n0, BN / 2 - 1);
      } else {
        base = g.W + (int64_t)n0 * g.ldb;
        row0 = half * SLOT_ROWS;
        row_lim = min(g.N - 1 - n0, BN - 1);
      }
    }
    rsrc = make_rsrc(base, (uint32_t)(((int64_t)row_lim * ld + g.K) * 2));
#pragma unroll
    for (int i = 0; i < DMA_PER_PHASE; ++i) {
      const int r = row0 + 8 * (4 * wq + i) + (lane >> 3);
      voff[i] = (uint32_t)(((int64_t)min(r, row_lim) * ld + lchunk8[i & 1]) * 2);
    }
  }
  // the offset of load i of the current stage (zero-reading past K)
  __device__ __forceinline__ uint32_t off(const GemmArgs& g, int i, const int* lchunk8) const {
    const int klim = g.K - T * BK;
    return lchunk8[i & 1] < klim ? voff[i] + (uint32_t)T * ROW_BYTES : 0x80000000u;
  }
  __device__ __forceinline__ void advance(const GemmArgs& g, int wq, int lane, const int* lchunk8) {
    if (!live) return;  // repeat the last stage
    if (++T == g.kst) {
      T = 0;
      ++round;
      setup(g, wq, lane, lchunk8);
      if (!live) T = g.kst - 1;  // nothing left: repeat the last stage of the last tile
    }
  }
};

template <int EPI>
__global__ __launch_bounds__(NT, 1) void gemm_bf16_nt(
    const uint16_t* __restrict__ X, int64_t lda, const uint16_t* __restrict__ W, int64_t ldb,
    const uint16_t* __restrict__ bias, const uint16_t* __restrict__ bias2,
    uint16_t* __restrict__ C, int64_t ldc, int M, int N, int K, int tiles_m, int tiles_n,
    int64_t sA, int64_t sB, int64_t sC, int vec_store) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  constexpr bool PAIRED = (EPI == CATOPT_EPI_SILU_MUL || EPI == CATOPT_EPI_GLU);
  constexpr int WROWS = PAIRED ? BN / 2 : BN;  // weight rows per projection in a tile
  GemmArgs ga;
  ga.X = X + (int64_t)blockIdx.y * sA;
  ga.W = W + (int64_t)blockIdx.y * sB;
  C += (int64_t)blockIdx.y * sC;
  ga.lda = lda;
  ga.ldb = ldb;
  ga.M = M;
  ga.N = N;
  ga.K = K;
  ga.tiles_m = tiles_m;
  ga.tiles_n = tiles_n;
  ga.nblocks = tiles_m * tiles_n;
  ga.kst = (K + BK - 1) / BK;
  // This workgroup's slot in a round: the workgroups of one XCD (ids
  // congruent mod 8) take consecutive logical tiles.
  ga.G = gridDim.x;
  ga.slot = (ga.G & 7) == 0 ? (blockIdx.x & 7) * (ga.G >> 3) + (blockIdx.x >> 3) : blockIdx.x;
  const int kst = ga.kst;
  if (ga.slot >= ga.nblocks) return;  // uniform over the workgroup

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wave >> 2, wq = wave & 3;
  const uint32_t lds0 = lds_u32(lds);
  const int lchunk8[2] = {((lane & 7) ^ (lane >> 4)) * 8, ((lane & 7) ^ (4 | (lane >> 4))) * 8};

  // ---- load streams.  Stage T of a tile (global stage s) is read in phases
  // 4s + 1 .. 4s + 4: group 0 in 4s + 1, 4s + 3 (its steps 2s, 2s + 1),
  // group 1 in 4s + 2, 4s + 4; group 0 computes in 4s + 2, 4s + 4 and group
  // 1 in 4s + 3, 4s + 5.  Each memory phase issues 4 loads per wave, 16 per
  // CU, among its fragment reads, so the loads are spread evenly over the
  // phases and the compute phases are MFMAs only:
  //   group 0, memory of step 2s     (4s + 1): W rows 0-127 of stage s + 1
  //   group 1, memory of step 2s     (4s + 2): W rows 128-255 of stage s + 1
  //   group 0, memory of step 2s + 1 (4s + 3): X rows 128-255 of stage s + 2
  //   group 1, memory of step 2s + 1 (4s + 4): X rows 0-127 of stage s + 2
  // W stage s + 1 goes into the W slots stage s - 1 used (last read in phase
  // 4s); X stage s + 2 into the X slots of stage s - 1 (last read in 4s - 1
  // or 4s).  At the end of its second memory phase of a stage each wave
  // waits for all its loads but the 4 it just issued: group 0's W half of
  // stage s + 1 (needed in 4s + 5) and X rows of stage s + 1 (4s + 6), group
  // 1's W half of stage s + 1 and X rows of stage s + 1 (both 4s + 5).  Every
  // wait for loads is followed by a barrier before the data is read: an
  // LDS-DMA write can become visible a little after vmcnt counts it done,
  // and a read straight after the wait (no barrier between) has seen stale
  // rows on MI355X.
  // st[0]: this wave's W stream (group 0 rows 0-127, group 1 rows 128-255);
  // st[1]: its X stream (group 0 X rows 128-255, group 1 X rows 0-127).
  Stream<PAIRED> st[2];
  st[0].what = 1;
  st[0].half = grp;
  st[1].what = 0;
  st[1].half = 1 - grp;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    st[h].round = 0;
    st[h].T = 0;
    st[h].setup(ga, wq, lane, lchunk8);
  }
  auto w_slot = [&](int stage_mod, int half) { return lds0 + (W_SLOT0 + 2 * stage_mod + half) * SLOT_BYTES; };
  auto x_slot = [&](int stage_mod, int g) { return lds0 + (X_RING * g + stage_mod) * SLOT_BYTES; };
  const uint32_t blk = 4 * wq * 1024;  // this wave's first 1 KB block in a slot

  // ---- fragments: lane l reads row (l % 16), chunk 4 h + (l / 16) of a
  // 16-row block for step h of a stage
  const int frag[2] = {swz(lane & 15, lane >> 4), swz(lane & 15, 4 + (lane >> 4))};
  // W row of the wave's n-block i (paired: blocks 0-1 gate, 2-3 up)
  auto wrow = [&](int i) { return PAIRED ? (i >> 1) * 128 + wq * 32 + (i & 1) * 16 : wq * 64 + i * 16; };
  bf16x8 xf[FM], wf[FN];
  // the step's 12 fragment reads with the phase's 4 loads of stream `ls`
  // into the slot at `dst` among them (one after every 3 reads)
  auto mem_phase = [&](int xmod, int wmod, int h, Stream<PAIRED>& ls, uint32_t dst) {
    const char* xs = lds + (X_RING * grp + xmod) * SLOT_BYTES;
    const char* ws = lds + (W_SLOT0 + 2 * wmod) * SLOT_BYTES;
#pragma unroll
    for (int i = 0; i < FN; ++i) {
      wf[i] = *reinterpret_cast<const bf16x8*>(ws + wrow(i) * ROW_BYTES + frag[h]);
      xf[2 * i] = *reinterpret_cast<const bf16x8*>(xs + 32 * i * ROW_BYTES + frag[h]);
      xf[2 * i + 1] = *reinterpret_cast<const bf16x8*>(xs + (32 * i + 16) * ROW_BYTES + frag[h]);
      dma_buf(ls.rsrc, ls.off(ga, i, lchunk8), dst + blk + i * 1024);
    }
    ls.advance(ga, wq, lane, lchunk8);
  };

  f32x4 acc[FN][FM];
  auto zero_acc = [&]() {
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto compute = [&]() {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = mfma16(wf[i], xf[j], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- epilogue of the tile at (m0, n0): the wave's 128 rows and 64 columns
  // (paired: 32 of each projection)
  auto epilogue = [&](int m0, int n0) {
    gemm_epilogue<EPI, FM>(acc, m0 + 128 * grp + (lane & 15), n0 + wq * (PAIRED ? 32 : 64), M, N, bias, bias2, C,
                           ldc, vec_store);
  };

  // ---- prologue: stage 0 (each wave its W and X rows) and X of stage 1
  for (int i = 0; i < DMA_PER_PHASE; ++i) dma_buf(st[0].rsrc, st[0].off(ga, i, lchunk8), w_slot(0, grp) + blk + i * 1024);
  st[0].advance(ga, wq, lane, lchunk8);
  for (int p = 0; p < 2; ++p) {
    for (int i = 0; i < DMA_PER_PHASE; ++i) dma_buf(st[1].rsrc, st[1].off(ga, i, lchunk8), x_slot(p, 1 - grp) + blk + i * 1024);
    st[1].advance(ga, wq, lane, lchunk8);
  }
  zero_acc();
  wait_vm_lgkm0<0>();
  __syncthreads();
  if (grp == 1) __syncthreads();  // group 1 runs one phase behind

  int round = 0, T = 0;      // the stage being computed (tile round, stage in tile)
  int xmod = 0, wmod = 0;    // its X and W slot indices
  int pm0 = -1, pn0 = -1;    // tile whose epilogue is pending
  int lt = ga.slot;
  TileMap tile = tile_of(lt, tiles_m, tiles_n);
  for (;;) {
    // ---- first step of the stage: fragments, and this wave's W rows of
    // the next stage into the W slot of the previous one
    __builtin_amdgcn_sched_barrier(0);
    if (pm0 >= 0) {  // first stage of a tile: the previous tile's stores, fresh accumulators
      epilogue(pm0, pn0);
      zero_acc();
      pm0 = -1;
    }
    const int xnext2 = xmod == 0 ? 2 : xmod - 1;  // (stage + 2) mod 3 == (stage - 1) mod 3
    mem_phase(xmod, wmod, 0, st[0], w_slot(wmod ^ 1, grp));
    wait_lgkm0();
    __syncthreads();
    compute();
    __syncthreads();
    // ---- second step: fragments, and this wave's X rows of stage + 2 into
    // the X slot of stage - 1; then everything but those landed
    __builtin_amdgcn_sched_barrier(0);
    mem_phase(xmod, wmod, 1, st[1], x_slot(xnext2, 1 - grp));
    wait_vm_lgkm0<DMA_PER_PHASE>();
    __syncthreads();
    compute();
    __syncthreads();
    // ---- next stage
    xmod = xmod == X_RING - 1 ? 0 : xmod + 1;
    wmod ^= 1;
    if (++T == kst) {
      T = 0;
      pm0 = tile.tm * BM;
      pn0 = tile.tn * WROWS;
      lt = (++round) * ga.G + ga.slot;
      if (lt >= ga.nblocks) break;
      tile = tile_of(lt, tiles_m, tiles_n);
    }
  }
  if (grp == 0) __syncthreads();  // match group 1's extra barrier
  epilogue(pm0, pn0);
  __builtin_amdgcn_s_waitcnt(0);  // the repeat loads past the last tile have landed
}

template <int EPI>
int32_t launch(const uint16_t* A, int64_t lda, const uint16_t* B, int64_t ldb,
               const uint16_t* bias, const uint16_t* bias2, uint16_t* C, int64_t ldc, int M,
               int N, int K, int64_t batch, int64_t sA, int64_t sB, int64_t sC, hipStream_t s) {
  constexpr bool PAIRED = (EPI == CATOPT_EPI_SILU_MUL || EPI == CATOPT_EPI_GLU);
  static bool attr_done = false;  // idempotent; benign race (same value written)
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_bf16_nt<EPI>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
    if (e != hipSuccess) return set_hip_error(e);
    attr_done = true;
  }
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles_n = (N + (PAIRED ? BN / 2 : BN) - 1) / (PAIRED ? BN / 2 : BN);
  const int64_t nblocks = (int64_t)tiles_m * tiles_n;
  if (nblocks > 0x7fffffff || batch > 65535) return CATOPT_E_UNSUPPORTED;
  // persistent: one workgroup per CU (each walks its tiles in rounds)
  int n_cu = 0;
  const int32_t st = gemm_cu_count(&n_cu);
  if (st != CATOPT_OK) return st;
  const int64_t grid = nblocks < n_cu ? nblocks : n_cu;
  // the epilogue's 16-byte stores of eight columns need every row of every
  // batch of C 16-byte aligned; otherwise it stores columns one by one
  const int vec_store = (ldc % 8 == 0) && (sC % 8 == 0) && aligned16(C);
  gemm_bf16_nt<EPI><<<dim3((uint32_t)grid, (uint32_t)batch), dim3(NT), LDS_BYTES, s>>>(
      A, lda, B, ldb, bias, bias2, C, ldc, M, N, K, tiles_m, tiles_n, sA, sB, sC, vec_store);
  CATOPT_LAUNCH_CHECK();
  return CATOPT_OK;
}

}  // namespace

// The current device's CU count, read once per device (idempotent; a race
// writes the same value).
int32_t gemm_cu_count(int* out) {
  static int cu_count[64] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return set_hip_error(e);
  int n = dev >= 0 && dev < 64 ? cu_count[dev] : 0;
  if (n == 0) {
    e = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return set_hip_error(e);
    if (n <= 0) n = 1;
    if (dev >= 0 && dev < 64) cu_count[dev] = n;
  }
  *out = n;
  return CATOPT_OK;
}

// Fast-path predicate shared with the dispatcher in gemm.hip.
bool gemm_bf16_nt_fast_ok(int64_t M, int64_t N, int64_t K, const void* x, int64_t ldx,
                          const void* w, int64_t ldw, const void* y, int64_t ldy) {
  // buffer offsets within one tile's rows: (255 * ld + K) * 2 bytes < 2^31
  const bool offsets_fit = (256 * (ldx > ldw ? ldx : ldw) + K) * 2 < (1LL << 31);
  return M > 0 && N > 0 && K > 0 && M < (1LL << 31) && N < (1LL << 30) && K < (1LL << 31) &&
         K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldx >= K && ldw >= K && offsets_fit &&
         aligned16(x) && aligned16(w) && ldy >= 1 && y != nullptr;
}

int32_t gemm_bf16_nt_launch(int32_t epi, int64_t M, int64_t N, int64_t K, const void* x,
                            int64_t ldx, const void* w, int64_t ldw, const void* bias,
                            const void* bias2, void* y, int64_t ldy, int64_t batch,
                            int64_t sA, int64_t sB, int64_t sC, void* ws, int64_t ws_bytes, hipStream_t s) {
  const bool paired = epi == CATOPT_EPI_SILU_MUL || epi == CATOPT_EPI_GLU;
  int n_cu = 0;
  const int32_t st = gemm_cu_count(&n_cu);
  if (st != CATOPT_OK) return st;
  const GemmMidPlan plan =
      gemm_bf16_plan(batch, M, N, K, paired, n_cu, ws != nullptr && aligned16(ws) && ws_bytes > 0 ? ws_bytes : 0);
  if (plan.shape == GEMM_ROWS)
    return gemm_bf16_rows_launch(epi, M, N, K, x, ldx, w, ldw, bias, bias2, y, ldy, batch, sA, sB, sC, s);
  if (plan.shape != GEMM_MID_NONE)
    return gemm_bf16_mid_launch(plan, epi, M, N, K, x, ldx, w, ldw, bias, bias2, y, ldy, ws, s);
  auto A = static_cast<const uint16_t*>(x);
  auto B = static_cast<const uint16_t*>(w);
  auto b1 = static_cast<const uint16_t*>(bias);
  auto b2 = static_cast<const uint16_t*>(bias2);
  auto C = static_cast<uint16_t*>(y);
  switch (epi) {
    case CATOPT_EPI_NONE: return launch<CATOPT_EPI_NONE>(A, ldx, B, ldw, b1, b2, C, ldy, (int)M, (int)N, (int)K, batch, sA, sB, sC, s);
    case CATOPT_EPI_BIAS: return launch<CATOPT_EPI_BIAS>(A, ldx, B, ldw, b1, b2, C, ldy, (int)M, (int)N, (int)K, batch, sA, sB, sC, s);
    case CATOPT_EPI_BIAS_ADD2: return launch<CATOPT_EPI_BIAS_ADD2>(A, ldx, B, ldw, b1, b2, C, ldy, (int)M, (int)N, (int)K, batch, sA, sB, sC, s);
    case CATOPT_EPI_SILU_MUL: return launch<CATOPT_EPI_SILU_MUL>(A, ldx, B, ldw, b1, b2, C, ldy, (int)M, (int)N, (int)K, batch, sA, sB, sC, s);
    case CATOPT_EPI_GLU: return launch<CATOPT_EPI_GLU>(A, ldx, B, ldw, b1, b2, C, ldy, (int)M, (int)N, (int)K, batch, sA, sB, sC, s);
    default: return CATOPT_E_INVAL;
  }
}

}  // namespace catopt
