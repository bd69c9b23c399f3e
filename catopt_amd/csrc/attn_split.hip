// Online-softmax attention for few queries (Tq <= 32) over many keys: a
// decode step, or a short block of queries against a long cache.
//
// K and V are read once and used by at most 32 queries, so HBM bounds it.
// The tile kernels of attention.hip give such a call one workgroup per
// (b, h), in which one wave's 32 (or 64) queries are real, and walk all keys
// there: 188 us a call for 128 heads x 8192 keys (2.9 TB/s, half the CUs idle),
// 106 us here (5.1 TB/s; a device copy moves 4.9, a read stream 6.8).
// Here a workgroup takes a range of the keys of one (b, h), its waves take
// 32 keys each of every stage, and the ranges' carriers are combined by a
// second launch (none when one range does).
//
// The products are those of attn_fwd_kernel: Sᵀ = K Qᵀ and Oᵀ += Vᵀ Pᵀ on
// the 32x32x16 MFMA, the accumulator column the query.  A wave's 32 keys of
// K and V go global->LDS directly, one stage ahead (two stages in LDS, two
// workgroups per CU: 128 KB per CU, half of it in flight).  Each wave keeps
// the running max, denominator and numerator of its own keys; they meet in
// LDS after the last stage.  The max moves eagerly, so it is the true row
// max and the combined (m, l, a) is the om_elem carrier.
#include "attention.hpp"

namespace catopt {
namespace {

constexpr float kNegInf = -__builtin_inff();

// Waves per workgroup: 64 KB of LDS for either head dim.
template <int D>
struct Split {
  static constexpr int WAVES = D == 128 ? 2 : 4, NT = 64 * WAVES;
  static constexpr int KEYS = 32 * WAVES;                   // per stage
  static constexpr int HALF = 32 * AttnRow<D>::BYTES;       // a wave's K (or V) rows of a stage
  static constexpr int WAVE_BYTES = 2 * HALF, STAGE = WAVES * WAVE_BYTES, BYTES = 2 * STAGE;
  static constexpr int LOADS = HALF / 1024;                 // 1 KB loads of K (and of V) per stage
  static constexpr int OLD = D + 4;                         // row of the merge buffer, floats
  static_assert(WAVES * 32 * OLD * 4 + WAVES * 64 * 4 <= BYTES, "the merge reuses the stages");
};

// exp2((from - to) c), 0 for an empty `from`.
__device__ __forceinline__ float move_factor(float from, float to, float c) {
  return from == kNegInf ? 0.f : __builtin_amdgcn_exp2f((from - to) * c);
}

// A row of the result: numerator piece x of a row with max m and sum l.
__device__ __forceinline__ float finish(float x, float l, int normalize) {
  if (!normalize) return x;
  if (l == 0.f) return normalize == 2 ? 0.f : __builtin_nanf("");
  return x * (1.0f / l);
}

template <int D, int MASK>
__global__ __launch_bounds__(Split<D>::NT, 2) void attn_split_kernel(AttnArgs a, int splits, float* part) {
  using L = Split<D>;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t bh = blockIdx.x / splits;
  const int split = blockIdx.x % splits;
  const int64_t b = bh / a.H, h = bh % a.H;
  const uint16_t* q = a.q + b * a.qs[0] + h * a.qs[1];
  const uint16_t* k = a.k + b * a.ks[0] + h * a.ks[1];
  const uint16_t* v = a.v + b * a.vs[0] + h * a.vs[1];
  const int Tq = (int)a.Tq, Tk = (int)a.Tk;
  // score units as in attn_fwd_kernel: raw q·k, or torch's scaled score where a bias is added
  constexpr bool kScaledScores = MASK == CATOPT_MASK_BIAS;
  const float c = (kScaledScores ? 1.f : a.scale) * 1.4426950408889634f;

  bf16x8 qf[D / 16];
#pragma unroll
  for (int j = 0; j < D / 16; ++j) {
    u32x4 t = u32x4{0, 0, 0, 0};
    if (l32 < Tq) t = *reinterpret_cast<const u32x4*>(q + (int64_t)l32 * a.qs[2] + 16 * j + 8 * g);
    qf[j] = __builtin_bit_cast(bf16x8, t);
  }

  int64_t kv_end = Tk;
  if (MASK == CATOPT_MASK_CAUSAL) {
    const int64_t lim = (int64_t)Tq + a.causal_off;  // past the last query's last key
    kv_end = lim < 0 ? 0 : (lim < Tk ? lim : Tk);
  }
  const int nst = (int)((kv_end + L::KEYS - 1) / L::KEYS);
  const int t0 = (int)((int64_t)nst * split / splits), t1 = (int)((int64_t)nst * (split + 1) / splits);

  // this wave's rows of a stage: 1 KB blocks, lane l slot 64 i + l
  // (literal array bounds: a bound that depends on D makes the host pass
  // drop the launch stub)
  static_assert(L::LOADS <= 8, "offset arrays hold 8 entries");
  uint32_t koff[8], voff[8];
#pragma unroll
  for (int i = 0; i < L::LOADS; ++i) {
    const int slot = 64 * i + lane, row = slot / AttnRow<D>::CH, cp = slot % AttnRow<D>::CH;
    koff[i] = (uint32_t)(row * (int)a.ks[2] + (cp ^ (row & (AttnRow<D>::CH - 1) & 15)) * 8) * 2u;
    voff[i] = (uint32_t)(row * (int)a.vs[2] + (cp ^ vswz<D>(row)) * 8) * 2u;
  }
  const uint32_t lds0 = lds_u32(lds) + wave * L::WAVE_BYTES;
  // rows past Tk lie outside the resources and read as zeros
  auto issue = [&](int t, int stage) {
    const int64_t key0 = (int64_t)t * L::KEYS + 32 * wave;
    const int64_t rows = Tk - key0 < 32 ? Tk - key0 : 32;
    const u32x4 kr = make_rsrc(k + key0 * a.ks[2], rows > 0 ? (uint32_t)(((rows - 1) * a.ks[2] + D) * 2) : 0u);
    const u32x4 vr = make_rsrc(v + key0 * a.vs[2], rows > 0 ? (uint32_t)(((rows - 1) * a.vs[2] + D) * 2) : 0u);
#pragma unroll
    for (int i = 0; i < L::LOADS; ++i) {
      dma_buf(kr, koff[i], lds0 + stage * L::STAGE + i * 1024);
      dma_buf(vr, voff[i], lds0 + stage * L::STAGE + L::HALF + i * 1024);
    }
  };

  f32x16 acc[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;
  float m = kNegInf, l = 0.f;

  if (t0 < t1) issue(t0, 0);
  for (int t = t0; t < t1; ++t) {
    const int stage = (t - t0) & 1;
    // stage t has landed (for every wave: an LDS-DMA write is read only past
    // a barrier), and every wave is done with the other half of the ring
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t + 1 < t1) issue(t + 1, stage ^ 1);
    const int key0 = t * L::KEYS + 32 * wave;
    if (key0 >= kv_end) continue;
    const char* Ks = lds + stage * L::STAGE + wave * L::WAVE_BYTES;
    const char* Vs = Ks + L::HALF;

    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int j = 0; j < D / 16; ++j)
      s = mfma32x32x16(*reinterpret_cast<const bf16x8*>(Ks + tile_off<D>(l32, 2 * j + g)), qf[j], s);
    bool need_mask = key0 + 32 > Tk || MASK == CATOPT_MASK_BOOL || MASK == CATOPT_MASK_BIAS;
    if (MASK == CATOPT_MASK_CAUSAL) need_mask = need_mask || (int64_t)key0 + 31 > a.causal_off;
    if (need_mask) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = key0 + acc_row(r, g);
        bool keep = key < Tk;
        if (MASK == CATOPT_MASK_CAUSAL) keep = keep & ((int64_t)key <= (int64_t)l32 + a.causal_off);
        float add = 0.f;
        if (MASK == CATOPT_MASK_BOOL || MASK == CATOPT_MASK_BIAS) {
          const int64_t mi = (int64_t)min(l32, Tq - 1) * a.mask_ld + min(key, Tk - 1);
          if (MASK == CATOPT_MASK_BOOL) keep = keep & (static_cast<const uint8_t*>(a.mask)[mi] != 0);
          if (MASK == CATOPT_MASK_BIAS) add = static_cast<const float*>(a.mask)[mi];
        }
        s[r] = keep ? (kScaledScores ? __builtin_fmaf(s[r], a.scale, add) : s[r]) : kNegInf;
      }
    }
    float mt = kNegInf;
#pragma unroll
    for (int r = 0; r < 16; ++r) mt = fmaxf(mt, s[r]);
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float m_new = fmaxf(m, mt);
    const float alpha = move_factor(m, m_new, c);
    m = m_new;
    const float mr = m == kNegInf ? 0.f : m;
    float lsum = 0.f;
    bf16x8 p[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      // the bias mode's scores may sit near -FLT_MAX, where s·c - m·c as one
      // fma leaves m·c's rounding error (or overflow); s - m is exact there
      const float e = kScaledScores ? __builtin_amdgcn_exp2f((s[r] - mr) * c)
                                    : __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], c, -mr * c));
      lsum += e;
      p[r >> 3][r & 7] = static_cast<__bf16>(e);
    }
    l = l * alpha + lsum;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] *= alpha;
    }
    // Vᵀ fragments.  Lane: group G = lane / 16, j = lane % 16 -> keys 4 (G / 2)
    // + j / 4 and 8 further, d block 16 (G % 2) + 4 (j % 4).
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int G = lane >> 4, jj = lane & 15;
        const int key = 16 * u + 4 * (G >> 1) + (jj >> 2);
        const int d = 32 * db + 16 * (G & 1) + 4 * (jj & 3);
        const s16x4 lo = ds_read_tr(Vs, vtile_off<D>(key, d >> 3) + (d & 7) * 2);
        const s16x4 hi = ds_read_tr(Vs, vtile_off<D>(key + 8, d >> 3) + (d & 7) * 2);
        const u32x2 lw = __builtin_bit_cast(u32x2, lo), hw = __builtin_bit_cast(u32x2, hi);
        acc[db] = mfma32x32x16(__builtin_bit_cast(bf16x8, u32x4{lw[0], lw[1], hw[0], hw[1]}), p[u], acc[db]);
      }
    }
  }

  // ---- the waves' carriers meet in LDS: [wave][query][d] numerators, then
  // [wave][query] (m, l)
  __syncthreads();  // every wave is done with the stages
  l += __shfl_xor(l, 32, 64);
  float* num = reinterpret_cast<float*>(lds);
  float* ml = num + L::WAVES * 32 * L::OLD;
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int rg = 0; rg < 4; ++rg)
      *reinterpret_cast<f32x4*>(num + (wave * 32 + l32) * L::OLD + 32 * db + 8 * rg + 4 * g) =
          f32x4{acc[db][4 * rg], acc[db][4 * rg + 1], acc[db][4 * rg + 2], acc[db][4 * rg + 3]};
  if (g == 0) {
    ml[(wave * 32 + l32) * 2] = m;
    ml[(wave * 32 + l32) * 2 + 1] = l;
  }
  __syncthreads();
  constexpr int TPQ = D / 4;  // threads per query, four numerators each
  const int d = 4 * (threadIdx.x % TPQ);
  for (int qr = threadIdx.x / TPQ; qr < Tq; qr += L::NT / TPQ) {
    float mw[L::WAVES], mx = kNegInf, lt = 0.f;
#pragma unroll
    for (int w = 0; w < L::WAVES; ++w) {
      mw[w] = ml[(w * 32 + qr) * 2];
      mx = fmaxf(mx, mw[w]);
    }
    f32x4 x = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < L::WAVES; ++w) {
      const float f = move_factor(mw[w], mx, c);
      lt += ml[(w * 32 + qr) * 2 + 1] * f;
      x += *reinterpret_cast<const f32x4*>(num + (w * 32 + qr) * L::OLD + d) * f;
    }
    if (splits > 1) {  // part: [row][split] (m, l, then D numerators at [row][split] of the second array)
      const int64_t i = (bh * Tq + qr) * splits + split, rows = (int64_t)gridDim.x * Tq;
      if (d == 0) {
        part[2 * i] = mx;
        part[2 * i + 1] = lt;
      }
      *reinterpret_cast<f32x4*>(part + ((2 * rows + 3) & ~(int64_t)3) + i * D + d) = x;
    } else {
      uint16_t* orow = a.o + b * a.os[0] + h * a.os[1] + (int64_t)qr * a.os[2];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = finish(x[e], lt, a.normalize);
      *reinterpret_cast<u32x2*>(orow + d) = u32x2{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])};
      if (d == 0) {
        if (a.m_out) a.m_out[bh * Tq + qr] = mx * (kScaledScores ? 1.f : a.scale);
        if (a.l_out) a.l_out[bh * Tq + qr] = lt;
      }
    }
  }
}

// The ranges' carriers of one row per wave: max, sum and numerator, in range order.
template <int D>
__global__ __launch_bounds__(256) void attn_split_combine(AttnArgs a, int splits, const float* part, float unit) {
  const int64_t rows = a.B * a.H * a.Tq, row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  constexpr int V = D / 64;  // numerators per lane
  const float c = unit * 1.4426950408889634f;
  const float* ml = part + 2 * row * splits;
  const float* num = part + ((2 * rows * splits + 3) & ~(int64_t)3) + row * splits * D + V * lane;
  float mx = kNegInf;
  for (int s = lane; s < splits; s += 64) mx = fmaxf(mx, ml[2 * s]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  float lt = 0.f, x[V];
#pragma unroll
  for (int e = 0; e < V; ++e) x[e] = 0.f;
  constexpr int U = 8;  // loads ahead of their additions
  for (int s0 = 0; s0 < splits; s0 += U) {
    float f[U], ls[U], xs[U][V];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const int s = min(s0 + i, splits - 1);
      f[i] = s0 + i < splits ? move_factor(ml[2 * s], mx, c) : 0.f;
      ls[i] = s0 + i < splits ? ml[2 * s + 1] : 0.f;
#pragma unroll
      for (int e = 0; e < V; ++e) xs[i][e] = s0 + i < splits ? num[(int64_t)s * D + e] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      lt += ls[i] * f[i];
#pragma unroll
      for (int e = 0; e < V; ++e) x[e] += xs[i][e] * f[i];
    }
  }
  const int64_t bh = row / a.Tq, t = row % a.Tq;
  uint16_t* orow = a.o + bh / a.H * a.os[0] + bh % a.H * a.os[1] + t * a.os[2];
#pragma unroll
  for (int e = 0; e < V; ++e) orow[V * lane + e] = f32_to_bf16(finish(x[e], lt, a.normalize));
  if (lane == 0) {
    if (a.m_out) a.m_out[row] = mx * unit;
    if (a.l_out) a.l_out[row] = lt;
  }
}

template <int D, int MASK>
int32_t launch_split(const AttnArgs& a, int splits, float* part, hipStream_t s) {
  static bool attr_done = false;  // idempotent; benign race (same value written)
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_split_kernel<D, MASK>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, Split<D>::BYTES);
    if (e != hipSuccess) return set_hip_error(e);
    attr_done = true;
  }
  const int64_t heads = a.B * a.H;
  if (heads * splits > 0x7fffffffLL) return CATOPT_E_UNSUPPORTED;
  attn_split_kernel<D, MASK><<<dim3((uint32_t)(heads * splits)), dim3(Split<D>::NT), Split<D>::BYTES, s>>>(a, splits, part);
  CATOPT_LAUNCH_CHECK();
  if (splits == 1) return CATOPT_OK;
  const int64_t blocks = (heads * a.Tq + 3) / 4;
  attn_split_combine<D><<<dim3((uint32_t)blocks), dim3(256), 0, s>>>(a, splits, part,
                                                                    MASK == CATOPT_MASK_BIAS ? 1.f : a.scale);
  CATOPT_LAUNCH_CHECK();
  return CATOPT_OK;
}

template <int D>
int32_t launch_mode(const AttnArgs& a, int32_t mode, int splits, float* part, hipStream_t s) {
  switch (mode) {
    case CATOPT_MASK_NONE: return launch_split<D, CATOPT_MASK_NONE>(a, splits, part, s);
    case CATOPT_MASK_CAUSAL: return launch_split<D, CATOPT_MASK_CAUSAL>(a, splits, part, s);
    case CATOPT_MASK_BOOL: return launch_split<D, CATOPT_MASK_BOOL>(a, splits, part, s);
    case CATOPT_MASK_BIAS: return launch_split<D, CATOPT_MASK_BIAS>(a, splits, part, s);
    default: return CATOPT_E_INVAL;
  }
}

}  // namespace

// Key ranges per (b, h): two workgroups per CU, at least two stages each.
int64_t attn_split_count(int64_t B, int64_t H, int64_t Tk, int64_t d) {
  constexpr int64_t kSlots = 512;
  const int64_t heads = B * H, keys = d == 128 ? Split<128>::KEYS : Split<64>::KEYS;
  int64_t n = heads > 0 ? kSlots / heads : 1;
  const int64_t stages = (Tk + keys - 1) / keys;
  if (n > stages / 2) n = stages / 2;
  return n < 1 ? 1 : n;
}

int64_t attn_split_workspace(int64_t B, int64_t H, int64_t Tq, int64_t Tk, int64_t d) {
  const int64_t n = attn_split_count(B, H, Tk, d), rows = B * H * Tq * n;
  return n <= 1 ? 0 : (((2 * rows + 3) & ~(int64_t)3) + rows * d) * (int64_t)sizeof(float);
}

int32_t attn_split_launch(const AttnArgs& a, int64_t d, int32_t mask_mode, void* ws, int64_t ws_bytes,
                          hipStream_t s) {
  int64_t n = attn_split_count(a.B, a.H, a.Tk, d);
  if (!ws || !aligned16(ws) || ws_bytes < attn_split_workspace(a.B, a.H, a.Tq, a.Tk, d)) n = 1;
  float* part = static_cast<float*>(ws);
  return d == 128 ? launch_mode<128>(a, mask_mode, (int)n, part, s) : launch_mode<64>(a, mask_mode, (int)n, part, s);
}

}  // namespace catopt
