// bf16 "NT" GEMM for middle row counts: C[m, n] = epi(sum_k X[m, k] W[n, k]).
//
// The 256 x 256 tiles of gemm_bf16.hip need several times 256 of them to keep
// the chip full; a 333-row batch through a 11008 -> 4096 projection has 32.
// Here a tile is BM x BN with BM = 64 or 128, and the tiles past the last
// whole round of workgroups split K: each (tile, K range) writes its fp32
// partial sums to the caller's workspace and gemm_bf16_reduce adds them in
// range order and applies the epilogue, so the result does not depend on
// timing and nothing is rounded before the end.
//
// A workgroup's waves form a 2 x (BN / 64) grid, each owning BM / 2 rows and
// 64 columns as 16 x 16 blocks of the 16x16x32 MFMA (W rows feed the A
// operand, X rows the B operand, as in gemm_bf16.hip).  K runs in stages of
// 64 through a ring of STAGES LDS slots: both operands' rows go global->LDS
// directly (whole 128-byte lines, rows XOR-swizzled so that a fragment read
// hits 16 distinct 16-byte bank groups), STAGES - 1 stages ahead, with one
// barrier per stage.  What bounds the loop is the stage's loads, by latency or
// bytes: 0.63 us per 128 x 256 x 64 stage with the operands cached, 0.80 us
// with W from HBM, where the MFMAs take 0.4 us.  A two-slot ring of 128 x 128
// tiles, two workgroups per CU, needed 0.83 us for the same work and cached
// operands.
#include "common.hpp"
#include "gemm_bf16.hpp"

namespace catopt {
namespace {

constexpr int BK = 64;

template <int BM, int BN, int STAGES>
struct Mid {
  static constexpr int WAVES_N = BN / 64, WAVES = 2 * WAVES_N, NT = 64 * WAVES;
  static constexpr int X_BYTES = BM * ROW_BYTES, STAGE = (BM + BN) * ROW_BYTES, BYTES = STAGES * STAGE;
  static constexpr int FM = BM / 32, FN = 4;                            // 16x16 blocks per wave along m, n
  static constexpr int XL = BM / 8 / WAVES, WL = BN / 8 / WAVES;        // 1 KB loads (8 rows) per wave and stage
  static_assert(XL >= 1 && WL >= 2 && BYTES <= 160 * 1024, "geometry");
};

struct MidArgs {
  const uint16_t* X;
  const uint16_t* W;
  const uint16_t* bias;
  const uint16_t* bias2;
  uint16_t* C;
  float* part;  // [splits][split tiles][BM][BN]
  int64_t ldx, ldw, ldc;
  int M, N, K, tiles_m, tiles_n, vec_store;
  int direct;   // tiles done whole: the first `direct` workgroups
  int round;    // workgroups per round (dealt to the XCDs in runs)
  int splits;   // K ranges of each tile after them
};

template <int EPI, int BM, int BN, int STAGES>
__global__ __launch_bounds__(2 * BN, 2) void gemm_bf16_mid(MidArgs g) {
  using G = Mid<BM, BN, STAGES>;
  constexpr bool PAIRED = (EPI == CATOPT_EPI_SILU_MUL || EPI == CATOPT_EPI_GLU);
  constexpr int COLS = PAIRED ? BN / 2 : BN;  // output columns of a tile
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / G::WAVES_N, wn = wave % G::WAVES_N;

  // Workgroups are dealt round robin over 8 XCDs: in each round an XCD takes a
  // contiguous run of tiles, so that those sharing X or W rows share its L2.
  const int ntiles = g.tiles_m * g.tiles_n, nsplit = ntiles - g.direct;
  int b = blockIdx.x, base = 0, count = g.direct;
  if (b < g.direct) {
    base = b / g.round * g.round;
    count = min(g.round, g.direct - base);
    b -= base;
  } else {
    b -= g.direct;
    count = nsplit * g.splits;
  }
  const int xcd = b & 7, per = count >> 3, rem = count & 7;
  const int pos = base + xcd * per + min(xcd, rem) + (b >> 3);
  const bool whole = (int)blockIdx.x < g.direct;
  const int split = whole ? 0 : pos / nsplit, st = whole ? 0 : pos % nsplit;
  const TileMap t = tile_of(whole ? pos : g.direct + st, g.tiles_m, g.tiles_n);
  const int m0 = t.tm * BM, n0 = t.tn * COLS;
  const int kst = (g.K + BK - 1) / BK;
  const int s0 = whole ? 0 : (int)((int64_t)kst * split / g.splits);
  const int s1 = whole ? kst : (int)((int64_t)kst * (split + 1) / g.splits);

  // this wave's loads: 1 KB blocks of 8 rows, lane l row l / 8, stored chunk
  // l % 8, i.e. global chunk (l % 8) ^ ((row / 2) % 8)
  const int mlim = min(g.M - 1 - m0, BM - 1), nlim = min(g.N - 1 - n0, COLS - 1);
  const u32x4 rx = make_rsrc(g.X + (int64_t)m0 * g.ldx, (uint32_t)(((int64_t)mlim * g.ldx + g.K) * 2));
  // W rows 0 .. BN - 1 of the tile; paired: the first half of the waves loads
  // rows of the first projection, the second half the matching ones of the second
  const bool second = PAIRED && wave >= G::WAVES / 2;
  const u32x4 rw = make_rsrc(g.W + ((int64_t)n0 + (second ? (int64_t)g.N : 0)) * g.ldw,
                             (uint32_t)(((int64_t)nlim * g.ldw + g.K) * 2));
  uint32_t xoff[G::XL], woff[G::WL];
  int xk[G::XL], wk[G::WL];
#pragma unroll
  for (int i = 0; i < G::XL; ++i) {
    const int row = 8 * (G::XL * wave + i) + (lane >> 3);
    xk[i] = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
    xoff[i] = (uint32_t)(((int64_t)min(row, mlim) * g.ldx + xk[i]) * 2);
  }
#pragma unroll
  for (int i = 0; i < G::WL; ++i) {
    const int row = 8 * (G::WL * wave + i) + (lane >> 3);
    wk[i] = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
    woff[i] = (uint32_t)(((int64_t)min(second ? row - COLS : row, nlim) * g.ldw + wk[i]) * 2);
  }
  const uint32_t lds0 = lds_u32(lds);
  // Load i of stage T into slot `slot`.  Past the unit's last stage the loads
  // read out of range (zeros, into a slot that is not read again), so that
  // every stage issues the same loads and the vmcnt bounds below stay exact.
  auto load = [&](int T, int slot, int i) {
    const int klim = T < s1 ? g.K - T * BK : 0;
    const uint32_t kb = (uint32_t)T * ROW_BYTES, base = lds0 + slot * G::STAGE;
    if (i < G::XL)
      dma_buf(rx, xk[i] < klim ? xoff[i] + kb : 0x80000000u, base + (G::XL * wave + i) * 1024);
    else
      dma_buf(rw, wk[i - G::XL] < klim ? woff[i - G::XL] + kb : 0x80000000u,
              base + G::X_BYTES + (G::WL * wave + i - G::XL) * 1024);
  };

  f32x4 acc[G::FN][G::FM];
#pragma unroll
  for (int i = 0; i < G::FN; ++i)
#pragma unroll
    for (int j = 0; j < G::FM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // fragments: lane l reads row l % 16, chunk 4 h + l / 16 of a 16-row block
  const int frag[2] = {swz(lane & 15, lane >> 4), swz(lane & 15, 4 + (lane >> 4))};
  auto wrow = [&](int i) { return PAIRED ? (i >> 1) * COLS + wn * 32 + (i & 1) * 16 : wn * 64 + i * 16; };

  bf16x8 wf[2][G::FN], xf[2][G::FM];
  auto read = [&](int slot, int h, int i) {
    const char* base = lds + slot * G::STAGE + frag[h];
    if (i < G::FN)
      wf[h][i] = *reinterpret_cast<const bf16x8*>(base + G::X_BYTES + wrow(i) * ROW_BYTES);
    else
      xf[h][i - G::FN] = *reinterpret_cast<const bf16x8*>(base + (wm * (BM / 2) + 16 * (i - G::FN)) * ROW_BYTES);
  };
  // One half stage: the products of half h with the reads of the next half and
  // some loads among them, one memory instruction between two MFMAs.  Issued in
  // a block, the reads and loads of all waves queue up in front of the first
  // product: 64 rows x 5504 -> 2048 without K ranges took 72 us for 55 with W
  // cached, and the same time with W from HBM.
  constexpr int NMEM = G::FN + G::FM, NLOAD = G::XL + G::WL, NLOAD_A = NLOAD / 2;
  auto half = [&](int h, int rslot, int rh, int T, int lslot, int l0, int l1) {
    constexpr int NM = G::FN * G::FM;
    int nr = 0, nl = l0;
#pragma unroll
    for (int x = 0; x < NM; ++x) {
      const int i = x / G::FM, j = x % G::FM;
      acc[i][j] = mfma16(wf[h][i], xf[h][j], acc[i][j]);
#pragma unroll
      for (; nr < NMEM && nr * NM < (x + 1) * NMEM; ++nr) read(rslot, rh, nr);
#pragma unroll
      for (; nl < l1 && (nl - l0) * NM < (x + 1) * (l1 - l0); ++nl) load(T, lslot, nl);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // The fragments of each half stage are read while the half before it is
  // multiplied.  A stage's slot is free once every wave has read its second
  // half, which the barrier in the middle of the stage establishes; the loads
  // of stage T + STAGES go there, the first ones in the second half of stage T
  // and the others in the first half of stage T + 1.
#pragma unroll
  for (int p = 0; p < STAGES; ++p)
#pragma unroll
    for (int i = 0; i < (p < STAGES - 1 ? NLOAD : NLOAD_A); ++i) load(s0 + p, p, i);
  wait_vm_lgkm0<(STAGES - 2) * NLOAD + NLOAD_A>();
  __syncthreads();
  int slot = 0, prev = STAGES - 1;
#pragma unroll
  for (int i = 0; i < NMEM; ++i) read(slot, 0, i);
  for (int T = s0; T < s1; ++T) {
    const int next = slot == STAGES - 1 ? 0 : slot + 1;
    __builtin_amdgcn_sched_barrier(0);
    half(0, slot, 1, T + STAGES - 1, prev, NLOAD_A, NLOAD);
    wait_vm_lgkm0<(STAGES - 2) * NLOAD>();  // stage T + 1 has landed
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    half(1, next, 0, T + STAGES, slot, 0, NLOAD_A);  // past the last stage: zeros, not used
    prev = slot;
    slot = next;
  }
  __builtin_amdgcn_s_waitcnt(0);  // the loads past the last stage have landed

  const int mrow = wm * (BM / 2) + (lane & 15);
  if (whole) {
    gemm_epilogue<EPI, G::FM>(acc, m0 + mrow, n0 + wn * (PAIRED ? 32 : 64), g.M, g.N, g.bias, g.bias2, g.C, g.ldc,
                              g.vec_store);
    return;
  }
  float* dst = g.part + (int64_t)pos * (BM * BN) + 4 * (lane >> 4);  // pos == split * nsplit + st
#pragma unroll
  for (int j = 0; j < G::FM; ++j) {
    if (m0 + mrow + 16 * j >= g.M) continue;
#pragma unroll
    for (int i = 0; i < G::FN; ++i)
      *reinterpret_cast<f32x4*>(dst + (mrow + 16 * j) * BN + wrow(i)) = acc[i][j];
  }
}

// Adds the K ranges' partial sums of the split tiles in range order and
// applies the epilogue: four output columns per thread; grid (tile, rows).
template <int EPI, int BM, int BN>
__global__ __launch_bounds__(256) void gemm_bf16_reduce(MidArgs g) {
  constexpr bool PAIRED = (EPI == CATOPT_EPI_SILU_MUL || EPI == CATOPT_EPI_GLU);
  constexpr int COLS = PAIRED ? BN / 2 : BN, TPR = COLS / 4;  // threads per row
  const int nsplit = g.tiles_m * g.tiles_n - g.direct, st = blockIdx.x;
  const TileMap t = tile_of(g.direct + st, g.tiles_m, g.tiles_n);
  const int row = blockIdx.y * (256 / TPR) + threadIdx.x / TPR, col = 4 * (threadIdx.x % TPR);
  const int m = t.tm * BM + row, n = t.tn * COLS + col;
  if (m >= g.M || n >= g.N) return;
  const float* p = g.part + ((int64_t)st * BM + row) * BN + col;
  const int64_t step = (int64_t)nsplit * BM * BN;
  f32x4 a = f32x4{0.f, 0.f, 0.f, 0.f}, c = a;
  // batches of loads ahead of their (ordered) additions: a chain of one load
  // per range cost 10 us at 32 ranges
  constexpr int U = PAIRED ? 4 : 8;
  for (int s = 0; s < g.splits; s += U) {
    f32x4 av[U], cv[U];
#pragma unroll
    for (int i = 0; i < U; ++i)
      if (s + i < g.splits) {
        av[i] = *reinterpret_cast<const f32x4*>(p + (s + i) * step);
        if (PAIRED) cv[i] = *reinterpret_cast<const f32x4*>(p + (s + i) * step + COLS);
      }
#pragma unroll
    for (int i = 0; i < U; ++i)
      if (s + i < g.splits) {
        a += av[i];
        if (PAIRED) c += cv[i];
      }
  }
  float o[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int nn = min(n + r, g.N - 1);
    const float b1 = EPI == CATOPT_EPI_BIAS || EPI == CATOPT_EPI_BIAS_ADD2 ? bf16_to_f32(g.bias[nn]) : 0.f;
    const float b2 = EPI == CATOPT_EPI_BIAS_ADD2 ? bf16_to_f32(g.bias2[nn]) : 0.f;
    o[r] = epilogue_value<EPI>(a[r], c[r], b1, b2);
  }
  uint16_t* dst = g.C + (int64_t)m * g.ldc + n;
  if (g.vec_store && n + 3 < g.N) {
    *reinterpret_cast<u32x2*>(dst) = u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < g.N) dst[r] = f32_to_bf16(o[r]);
  }
}

template <int EPI, int BM, int BN, int STAGES>
int32_t run_mid(MidArgs a, hipStream_t s) {
  using G = Mid<BM, BN, STAGES>;
  constexpr int COLS = (EPI == CATOPT_EPI_SILU_MUL || EPI == CATOPT_EPI_GLU) ? BN / 2 : BN;
  static bool attr_done = false;  // idempotent; benign race (same value written)
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_bf16_mid<EPI, BM, BN, STAGES>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, G::BYTES);
    if (e != hipSuccess) return set_hip_error(e);
    attr_done = true;
  }
  a.tiles_m = (a.M + BM - 1) / BM;
  a.tiles_n = (a.N + COLS - 1) / COLS;
  const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
  if (tiles > 0x3fffffff) return CATOPT_E_UNSUPPORTED;
  if (a.splits <= 1) a.direct = (int)tiles;
  const int nsplit = (int)tiles - a.direct;
  gemm_bf16_mid<EPI, BM, BN, STAGES>
      <<<dim3((uint32_t)(a.direct + nsplit * a.splits)), dim3(G::NT), G::BYTES, s>>>(a);
  CATOPT_LAUNCH_CHECK();
  if (nsplit == 0) return CATOPT_OK;
  gemm_bf16_reduce<EPI, BM, BN><<<dim3((uint32_t)nsplit, BM * COLS / 1024), dim3(256), 0, s>>>(a);
  CATOPT_LAUNCH_CHECK();
  return CATOPT_OK;
}

template <int EPI>
int32_t run_shape(const MidArgs& a, int shape, hipStream_t s) {
  switch (shape) {
    case GEMM_MID_128x256: return run_mid<EPI, 128, 256, 3>(a, s);
    case GEMM_MID_64x128: return run_mid<EPI, 64, 128, 3>(a, s);
    default: return CATOPT_E_INVAL;
  }
}

}  // namespace

// Which kernel runs a bf16 NT product (or a batch of them), by the time each
// would take in us.  The constants are fits to 1242 single and 1765 batched
// sizes, plain and gated, 1 to 4096 rows, N from 32 to 131072, K from 64 to
// 11008, weights from memory (profiles/gemm_bf16_routes.md): the kernel chosen
// here is within 1.6% of the best one on average, 0.7% without a workspace and
// 0.3% in a batch, and at most 8% slower than the large tiles.  Before, few rows
// took the few-rows kernel whatever N and the batch were: 64 rows x 4096 ->
// 131072 630 us for 258 on the large tiles, a batch of 512 of 64 x 128 ->
// 2048 358 for 119.  The chip's clock moves all of the times together, so the
// choice does not depend on it.  Without a workspace no tile is split.
namespace {

struct TileCost {
  int shape, bm, bn, per_cu;
  double launch, lo, hi, edge, mb_per_us;   // one launch of whole tiles
  double fixed, split_edge, part_mb_per_us;  // with K ranges: both launches, partial sums
};
constexpr TileCost kLarge = {GEMM_MID_NONE, 256, 256, 1, 2.3, 1.08, 1.51, 3.0, 4.5e6, 0, 0, 0};
constexpr TileCost kMid[2] = {{GEMM_MID_64x128, 64, 128, 2, 1.8, 0.41, 0.68, 3.5, 5.2e6, 4.6, 3.8, 2.4e6},
                              {GEMM_MID_128x256, 128, 256, 1, 1.1, 0.67, 0.91, 4.5, 5.2e6, 4.5, 5.2, 2.6e6}};

// `units` workgroups in rounds of `slots`, in stage times: lo where one runs
// alone, hi where the chip is full (the clock falls and the L2s fill).
double rounds(double units, double slots, const TileCost& c) {
  const double full = (double)(int64_t)(units / slots), rest = units - full * slots;
  return full * c.hi + (rest > 0 ? c.lo + (c.hi - c.lo) * rest / slots : 0.0);
}

// The few-rows kernel: the latency of a wave's passes over K, the work of the
// workgroups that follow each other on a CU (a workgroup fills it; per
// projection and 16-row block, and per K chunk for W and each row of X), or
// the bytes at HBM's rate.
double rows_cost(double batch, int64_t M, int64_t N, int64_t K, int np, int n_cu, double bytes) {
  const double mb = (double)((M + 15) / 16), nch = (double)((K + BK - 1) / BK), w = np * mb;
  const int64_t per_pass = mb <= 2 ? (np == 2 ? 16 : 32) : 16;  // waves x chunks in flight
  const double passes = (double)(((int64_t)nch + per_pass - 1) / per_pass);
  const double work = 0.49 + 0.054 * w + nch * (0.066 * np + 0.0033 * (double)M);
  const double chip = (double)(((int64_t)batch * ((N + 15) / 16) + n_cu - 1) / n_cu) * work;
  const double latency = passes * 2.3, hbm = bytes / 6.2e6;
  return 2.15 + (latency > chip ? (latency > hbm ? latency : hbm) : (chip > hbm ? chip : hbm));
}

GemmMidPlan plan_for(int64_t batch, int64_t M, int64_t N, int64_t K, bool paired, int n_cu, bool ws) {
  GemmMidPlan best{GEMM_MID_NONE, 0, n_cu, 1};
  const int np = paired ? 2 : 1;
  const double nb = (double)batch, kst = (double)((K + BK - 1) / BK);
  const double wsize = nb * np * (double)N * (double)K;  // weight elements
  const double bytes = 2.0 * (wsize + nb * (double)M * (double)(K + N));
  const bool rows = gemm_bf16_rows_ok(M, N);
  // At most 16 rows of a long K over many weight bytes: the loads of W bound
  // every kernel and this one streams them best (8 rows x 4096 -> 131072 193 us
  // for 212, 1 row x 2048 -> 32768 23 for 33), which the fit underrates.
  if (rows && M <= 16 && K >= 2048 && wsize >= 1 << 25) {
    best.shape = GEMM_ROWS;
    return best;
  }
  auto tiles = [&](const TileCost& c) {
    const int64_t cols = paired ? c.bn / 2 : c.bn;
    return nb * (double)(((M + c.bm - 1) / c.bm) * ((N + cols - 1) / cols));
  };
  auto whole = [&](const TileCost& c) {
    const double t = (kst + c.edge) * rounds(tiles(c), (double)n_cu * c.per_cu, c), hbm = bytes / c.mb_per_us;
    return c.launch + (t > hbm ? t : hbm);
  };
  double cost = whole(kLarge);
  auto consider = [&](double c, const GemmMidPlan& p) {
    if (c < cost) {
      cost = c;
      best = p;
    }
  };
  // In a batch only where it is clearly cheaper: its fit is the looser one.  A
  // batch that fills the chip reads its X from memory too, which counts where
  // that is no smaller than W: 1024 of 64 x 2048 -> 64 257 us for 190.
  const double margin = batch == 1 ? 1.0 : 1.3;
  const bool x_counts = batch > 1 && M > 32 && M >= N && K >= 256 && nb * (double)((N + 15) / 16) >= 4.0 * n_cu;
  if (rows && !x_counts) consider(margin * rows_cost(nb, M, N, K, np, n_cu, bytes), GemmMidPlan{GEMM_ROWS, 0, n_cu, 1});
  // One row of large tiles on every CU reads W once where two rows of middle
  // ones read it twice: 256 rows x 512 -> 131072 44 us for 56.
  if (batch != 1 || (M > 128 && M <= 256 && tiles(kLarge) >= n_cu)) return best;
  for (const TileCost& c : kMid) {
    const double t = tiles(c), slots = (double)n_cu * c.per_cu;
    if (!grid_fits((int64_t)t + n_cu, 2 * c.bn)) continue;  // at most n_cu workgroups for split tiles
    consider(whole(c), GemmMidPlan{c.shape, (int)t, n_cu, 1});
    if (!ws) continue;
    // K ranges for the tiles past the last whole round, one workgroup per CU
    const int64_t direct = (int64_t)t / n_cu * n_cu, left = (int64_t)t - direct;
    if (left == 0 || (c.per_cu > 1 && direct > 0)) continue;
    int64_t splits = n_cu / left;
    if (splits > (int64_t)(kst / 2)) splits = (int64_t)(kst / 2);
    if (splits < 2) continue;
    const double units = (double)(left * splits), hbm = bytes / c.mb_per_us;
    const double loop = (kst + c.edge) * rounds((double)direct, slots, c) +
                        (kst / (double)splits + c.split_edge) * rounds(units, slots, c);
    // only rows below M are written: M of each column of tiles
    const double part = units * c.bn * 4.0 * (double)M / (double)((M + c.bm - 1) / c.bm);
    // taken where it is clearly cheaper, and for calls that the host's two
    // launches and the workspace (13 us) do not bound anyway: 128 rows x 1024
    // -> 1024 13.2 us for 8.4 whole
    const double t2 = 1.05 * (c.fixed + (loop > hbm ? loop : hbm) + part / c.part_mb_per_us);
    consider(t2 > 13.0 ? t2 : 13.0, GemmMidPlan{c.shape, (int)direct, n_cu, (int)splits});
  }
  return best;
}

}  // namespace

int64_t gemm_bf16_mid_workspace(const GemmMidPlan& p, int64_t M, int64_t N, bool paired) {
  if (p.shape < GEMM_MID_128x256 || p.splits <= 1) return 0;
  const int64_t bm = p.shape == GEMM_MID_128x256 ? 128 : 64, bn = p.shape == GEMM_MID_128x256 ? 256 : 128;
  const int64_t cols = paired ? bn / 2 : bn;
  const int64_t left = ((M + bm - 1) / bm) * ((N + cols - 1) / cols) - p.direct;
  return left * p.splits * bm * bn * (int64_t)sizeof(float);
}

GemmMidPlan gemm_bf16_plan(int64_t batch, int64_t M, int64_t N, int64_t K, bool paired, int n_cu, int64_t ws_bytes) {
  if (batch == 1 && ws_bytes > 0) {
    const GemmMidPlan p = plan_for(1, M, N, K, paired, n_cu, true);
    if (gemm_bf16_mid_workspace(p, M, N, paired) <= ws_bytes) return p;
  }
  return plan_for(batch, M, N, K, paired, n_cu, false);
}

int32_t gemm_bf16_mid_launch(const GemmMidPlan& plan, int32_t epi, int64_t M, int64_t N, int64_t K, const void* x,
                             int64_t ldx, const void* w, int64_t ldw, const void* bias, const void* bias2, void* y,
                             int64_t ldy, void* ws, hipStream_t s) {
  MidArgs a;
  a.X = static_cast<const uint16_t*>(x);
  a.W = static_cast<const uint16_t*>(w);
  a.bias = static_cast<const uint16_t*>(bias);
  a.bias2 = static_cast<const uint16_t*>(bias2);
  a.C = static_cast<uint16_t*>(y);
  a.part = static_cast<float*>(ws);
  a.ldx = ldx;
  a.ldw = ldw;
  a.ldc = ldy;
  a.M = (int)M;
  a.N = (int)N;
  a.K = (int)K;
  a.direct = plan.direct;
  a.round = plan.round;
  a.splits = plan.splits;
  a.vec_store = ldy % 8 == 0 && aligned16(y);
  switch (epi) {
    case CATOPT_EPI_NONE: return run_shape<CATOPT_EPI_NONE>(a, plan.shape, s);
    case CATOPT_EPI_BIAS: return run_shape<CATOPT_EPI_BIAS>(a, plan.shape, s);
    case CATOPT_EPI_BIAS_ADD2: return run_shape<CATOPT_EPI_BIAS_ADD2>(a, plan.shape, s);
    case CATOPT_EPI_SILU_MUL: return run_shape<CATOPT_EPI_SILU_MUL>(a, plan.shape, s);
    case CATOPT_EPI_GLU: return run_shape<CATOPT_EPI_GLU>(a, plan.shape, s);
    default: return CATOPT_E_INVAL;
  }
}

}  // namespace catopt
