// attn_tq3_lut.h -- the centroid-pair table of the TQ3 attention kernels, the
// operand lookups built on it, and the wave-level pieces they share.
#pragma once
#include "attn_common.h"
#include "qkv_device.h"

namespace qkv {

// Centroid-pair table, one copy per lane: entry E of lane L at byte
// E * 256 + 4 * L, so every lane reads its own bank and a wave's 64 lookups
// never conflict.  An address is 4 * L in byte 0 and an 8-bit index in byte 1,
// written by one SDWA shift (sdwa_index): the low 6 bits of the index are two
// 3-bit codes, the top 2 bits are whatever follows them in the code stream,
// so entry E holds the pair of E & 63.  The table sits at LDS offset 0 so
// that no base has to be added (256 x 64 x 4 B = 64 KiB).
constexpr int kLdsLut = 0;
constexpr int kLdsLutBytes = 256 * 64 * 4;

__device__ __forceinline__ uint32_t lut_read(const uint8_t* lds, uint32_t addr) {
  return *reinterpret_cast<const uint32_t*>(lds + kLdsLut + addr);
}

// Table address of the 6-bit field at bit BIT of a 3-dword code stream
// (a field that crosses a dword boundary is first funnel-shifted to bit 0).
template <int BIT>
__device__ __forceinline__ uint32_t pair_addr3(uint32_t& chain, const uint32_t (&q)[3]) {
  constexpr int w = BIT >> 5, sh = BIT & 31;
  if constexpr (sh + 6 <= 32)
    chain = sdwa_index<sh>(chain, q[w]);
  else
    chain = sdwa_index<0>(chain, __builtin_amdgcn_alignbit(q[w + 1], q[w], sh));
  return chain;
}

// B operand for code group U (8 codes, bits 24U..24U+23) of a 3-dword stream.
template <int U>
__device__ __forceinline__ h8_t group_operand(const uint8_t* lds, uint32_t (&ac)[4],
                                              const uint32_t (&q)[3]) {
  u4_t v;
  v[0] = lut_read(lds, pair_addr3<24 * U + 0>(ac[0], q));
  v[1] = lut_read(lds, pair_addr3<24 * U + 6>(ac[1], q));
  v[2] = lut_read(lds, pair_addr3<24 * U + 12>(ac[2], q));
  v[3] = lut_read(lds, pair_addr3<24 * U + 18>(ac[3], q));
  return __builtin_bit_cast(h8_t, v);
}

// Dims 0, 2, 4, 6 of a 24-bit code group (bits 6d .. 6d + 2).
constexpr uint32_t kEvenDims = 0x1C71C7u;

// (a & m) | (b & ~m) in one v_bfi_b32 (the compiler splits some constant
// masks into an and plus an and-or)
__device__ __forceinline__ uint32_t bit_select(uint32_t m, uint32_t a, uint32_t b) {
  uint32_t d;
  asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(d) : "s"(m), "v"(a), "v"(b));
  return d;
}

// Key pairs (i, i + 1) = (2k, 2k + 1) of a pass's codes as loaded (x[i]: key
// i's code group): the second key's codes moved up by one code, merged with
// the first key's by bit select.  Done in place at the pass's first table
// reads, two steps after its staging loads were issued.
__device__ __forceinline__ void interleave_pairs(uint32_t (&x)[8]) {
  uint32_t z[8];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t hi = x[2 * k + 1] << 3;
    z[k] = bit_select(kEvenDims, x[2 * k], hi);
    z[4 + k] = bit_select(kEvenDims << 3, x[2 * k], hi);
  }
#pragma unroll
  for (int i = 0; i < 8; i++) x[i] = z[i];
}

// Key visibility of one query (attention.cuh:1923-1929, 2101-2105): the
// sink/window rule on 32-key tiles, then the tree bits for keys of the block.
// Branch-free: every key of a tile is tested with the same instructions.
struct KeyRule {
  int start_pos, sink, window;
  bool sw, has_tree;
  uint32_t tree_bits;   // bit j: key start_pos + j is visible
  __device__ KeyRule(int start_pos_, int t_idx, int sink_, int window_, const uint32_t* tree)
      : start_pos(start_pos_), sink(sink_), window(window_), sw(sink_ > 0 || window_ > 0),
        has_tree(tree != nullptr), tree_bits(tree ? tree[t_idx] : 0u) {}
  // every key of [a, b) is visible (no rule applies there)
  __device__ __forceinline__ bool all_visible(int b) const {
    return !sw && (!has_tree || b <= start_pos);
  }
  __device__ __forceinline__ bool visible(int key, int active_end) const {
    const int ts = key & ~31;
    const int te = min(ts + 32, active_end);
    const bool sw_ok = !sw | (ts < sink) | (te > active_end - window);
    const bool tree_ok = !has_tree | (key < start_pos) |
                         (((tree_bits >> ((key - start_pos) & 31)) & 1u) != 0u);
    return sw_ok & tree_ok;
  }
};

// Max / sum over the 4 rows of the wave (lanes l, l^16, l^32, l^48); every
// lane receives the result.  Each gfx950 row swap leaves a lane holding its
// own value and its partner row's value in the two registers.
__device__ __forceinline__ float xrow_max(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float xrow_sum(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

}  // namespace qkv
