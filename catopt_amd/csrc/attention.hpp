// What the bf16 attention kernels share: the swizzled K and V tile layouts,
// the transposing LDS read, and the launchers' declarations.
#pragma once
#include "common.hpp"

namespace catopt {

typedef __attribute__((ext_vector_type(4))) short s16x4;

// A K or V row of head dim D.
template <int D>
struct AttnRow {
  static constexpr int BYTES = D * 2;
  static constexpr int CH = D / 8;  // 16-byte chunks
};

// Byte offset of (key, 16-byte chunk) inside a swizzled tile.
template <int D>
__device__ __forceinline__ int tile_off(int key, int chunk) {
  return key * AttnRow<D>::BYTES + ((chunk ^ (key & (AttnRow<D>::CH - 1) & 15)) << 4);
}

// V tiles use their own swizzle.  A transposing read of Vᵀ covers, per
// 32-lane pass, 4 consecutive keys x 4 adjacent 16-byte chunks; XOR-ing the
// chunk index with 4 * (the key's position among those 4, per 256-byte bank
// window) puts the 16 pieces in 16 different bank groups (the key-row
// swizzle above would put all 4 keys on the same 4 groups).
template <int D>
__device__ __forceinline__ int vswz(int key) {
  constexpr int R = 256 / AttnRow<D>::BYTES;  // tile rows per 256-byte bank window
  return 4 * ((key / R) & (4 / R - 1));
}
template <int D>
__device__ __forceinline__ int vtile_off(int key, int chunk) {
  return key * AttnRow<D>::BYTES + ((chunk ^ vswz<D>(key)) << 4);
}

__device__ __forceinline__ s16x4 ds_read_tr(const char* lds_base, int byte_off) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)(lds_base + byte_off));
}

// Few queries over split keys (attn_split.hip).
struct AttnArgs {
  const uint16_t *q, *k, *v;
  uint16_t* o;
  int64_t qs[3], ks[3], vs[3], os[3];
  float *m_out, *l_out;
  int64_t B, H, Tq, Tk, causal_off;
  const void* mask;
  int64_t mask_ld;
  float scale;
  int normalize;
};
constexpr int64_t kAttnSplitQueries = 32;  // the largest Tq it takes
int64_t attn_split_count(int64_t B, int64_t H, int64_t Tk, int64_t d);
int64_t attn_split_workspace(int64_t B, int64_t H, int64_t Tq, int64_t Tk, int64_t d);
int32_t attn_split_launch(const AttnArgs& a, int64_t d, int32_t mask_mode, void* ws, int64_t ws_bytes, hipStream_t s);

}  // namespace catopt
