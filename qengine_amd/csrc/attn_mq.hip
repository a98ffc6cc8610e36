// attn_mq.hip -- decode of multi-query calls (verify blocks):
// every cache tile is read once for up to 64 (query, head) columns (gfx950).
//
// Reference semantics: the split kernels with sub_n > 1 and their merge
// (attention.cuh:1905-2177, 2633-2801, 1837-1891), over TQ3 caches, Q8_0
// caches, or Q8_0 keys with TQ3 values.  TQ3 blocks are consumed in rotated
// coordinates as in attn_tq3.hip.  Column c = qi * gqa + hh of a workgroup is q head h * gqa + hh
// of query t0 + qi.
//
// Workgroup: 8 waves on one kv head, one block of queries (up to 64 columns)
// and one key chunk, walked in 64-key tiles:
//   staging  the tile's key and value rows arrive with 16-byte loads (12-byte
//            ones for TQ3 pieces), a tile ahead, and are stored to LDS as
//            packed: the codes are decoded by the wave that feeds them to an
//            MFMA, straight into the operand registers, so no decoded tile
//            passes through the LDS.
//   scores   wave w = (key group kg = w & 3, column half ch = w >> 2): 16 keys
//            x 32 columns, v_mfma_f32_16x16x32_f16 with A = keys decoded in
//            registers and B = the queries (held for the whole kernel).
//   softmax  per column against a reference maximum, base 2; the
//            probabilities go to LDS as fp16 in the operand order of the value
//            product.  A score above the reference by more than kSlack (the
//            first tile, rarely later) raises it: only then do the key groups
//            exchange maxima and the sums and accumulators get rescaled.  The
//            largest weight is therefore not 1 and exact, but rounded like the
//            others: with Q8_0 values (whose weights carry no norm to round) what
//            the rounding leaves out is kept as a second fp16 number, with a
//            product of its own, so that the rows are no further from the exact
//            ones than with a running maximum in every wave (2-norm, 16 queries
//            over 4,096 keys: 6.30e-4 there, 6.48e-4 with one product).
//   values   wave w owns dims 32 w .. 32 w + 31 of all columns: A = the
//            probabilities (one 16-byte read per 16 columns and 32 keys), B =
//            its own dims of 32 keys, decoded in registers.  32 accumulators
//            per lane and no merge of waves at the end: every wave stores its
//            dims of the records itself.
// One barrier per tile: the scores of tile t + 1 follow the value product of
// tile t in the same interval (three staging buffers, two of probabilities).
// The records are merged by a launch of their own (attn_merge.hip): no workgroup
// waits for another, so a call completes on whatever part of the GPU is free.
#include <type_traits>

#include "attn_common.h"
#include "attn_fastmerge.h"
#include "attn_tq3_lut.h"
#include "qkv_device.h"
#include "tq3_encode.h"

namespace qkv {
namespace {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h4_t __attribute__((ext_vector_type(4)));

constexpr int kTile = 64;
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kHD = 256;
constexpr int kQ8Row = 288, kTq3Row = 104;   // bytes of one kv head of one token

// Staged Q8_0 rows: 18 16-byte pieces at a pitch of 76 dwords, so that the
// 8-byte reads of 16 key rows (12-dword steps modulo the 64 banks) and the
// dword reads of the value rows hit different banks.
constexpr int kQ8Pitch = 304;
// Staged TQ3 value codes: [32 groups of 8 dims][64 keys], one dword per group
// and key, rows 68 dwords apart.
constexpr int kVgPitch = 68;
// How far (log2 units) a score may exceed its column's reference before the
// reference is raised to the running maximum minus kHead: the reference settles
// within the first tiles, so that a tile normally needs no exchange of maxima
// between the waves.  Weights stay below 2^kSlack, and kHead keeps small ones
// clear of fp16's denormals (TQ3 values: the weights carry the block norm).
template <bool VT>
constexpr float kSlack = VT ? 8.0f : 14.0f;
template <bool VT>
constexpr float kHead = VT ? 0.0f : 6.0f;
constexpr float kNoRef = -1e30f;

// Centroid-pair table: entry e (two 3-bit codes) of lane L at byte e * 256 + 4 * L
// (64 entries, so indexes are clean 6-bit values).
constexpr int kLutBytes = 64 * 64 * 4;

// KT / VT: TQ3 keys / values (TQ3 keys come with TQ3 values).
template <bool KT, bool VT>
struct MqLds {
  // TQ3 keys: [64 keys][8 pieces] of 16 bytes, one byte per code pair, key r's
  // piece c at c ^ ((r >> 1) & 7) (16 rows at one logical piece: 16 bank groups)
  static constexpr int kKBuf = KT ? kTile * 128 : kTile * kQ8Pitch;
  static constexpr int kVBuf = VT ? 32 * kVgPitch * 4 : kTile * kQ8Pitch;
  // [64 columns][64 keys] fp16: TQ3 values one per 128-block, Q8_0 values the weights and their rests
  static constexpr int kPBuf = 2 * 64 * 128;
  static constexpr int kK = VT ? kLutBytes : 0;           // three buffers each
  static constexpr int kV = kK + 3 * kKBuf;
  // TQ3 norms [3 buffers][keys block 0, 1 (x the softmax scale), values block 0, 1][64] f32
  static constexpr int kNorm = kV + 3 * kVBuf;
  static constexpr int kP = kNorm + (VT ? 3 * 4 * kTile * 4 : 0);   // probabilities, two buffers
  static constexpr int kMx = kP + 2 * kPBuf;              // [64 columns][4 key groups] f32
  static constexpr int kCorr = kMx + 64 * 4 * 4;          // [64] rescale factors, then 4 flags
  static constexpr int kSc = kCorr + 64 * 4 + 16;         // Q8 values: per wave [64 keys] fp16 scales of its block
  static constexpr int kEnc = kSc + (VT ? 0 : kWaves * kTile * 2);   // fused append: [64 new keys][K, V x 2 blocks][13 dwords]
  static constexpr int kEnd = kEnc + (KT ? 64 * 4 * 13 * 4 : 0);
  // setup (TQ3 keys): rotated queries, fp16 rounding and remainder [64 columns][512 B] each
  static constexpr int kQhi = kK, kQlo = kK + 64 * 512;
  // after the tile loop
  static constexpr int kSum = 0;                          // [4][64] sums, [64] maxima, [64] record indices
  static constexpr int kRowPitch = kHD + 4;               // SPLIT: rows to rotate back, kSum's maxima in between
  static constexpr int kRows = kSum + 10 * 64 * 4;
  static_assert(kRows + 32 * kRowPitch * 4 <= kEnd, "rows to rotate back (NG = 2)");
  static_assert(kSum + 6 * 64 * 4 <= kP, "end-of-kernel scalars must not reach the probabilities");
  static_assert(!KT || kQlo + 64 * 512 <= kMx, "query scratch must not reach the flags");
  static_assert(kEnd <= 160 * 1024, "LDS");
};

// One tile's rows in flight.  Q8_0 rows: 16-byte pieces c = tid + 512 i of the
// 1,152 key pieces (then, for Q8_0 values, the 1,152 value pieces), piece c of
// row c / 18.  TQ3 rows: thread (row tid / 8, pc = tid % 8) takes the 12 bytes
// of code groups 4 pc .. 4 pc + 3; waves 0..3 one norm per lane (lane = key):
// keys block 0, 1 (TQ3 keys), values block 0, 1.
template <bool KT, bool VT>
struct MqRegs {
  u4_t q[KT ? 1 : VT ? 3 : 5];
  u3_t k, v;
  float nm;
};

// The rows of a thread's 16-byte Q8_0 pieces, 6 bits each: one register through
// the tile loop, from which a piece's offsets are formed where they are used
// (opaque, so that they are not hoisted into registers of their own).
template <bool KT, bool VT>
__device__ __forceinline__ uint32_t mq_rows(int tid) {
  uint32_t v = 0u;
  if constexpr (KT) return v;
#pragma unroll
  for (int i = 0; i < (VT ? 3 : 5); i++) {
    const int c = tid + kThreads * i;
    v |= (uint32_t)((c >= 1152 ? c - 1152 : c) / 18) << (6 * i);
  }
  return v;
}
struct MqPiece {
  uint32_t row, byte;   // its row, and 16 x its index in the tensor's piece list
  __device__ __forceinline__ uint32_t cache(int nkv, int h) const {
    return byte + row * (uint32_t)(kQ8Row * (nkv - 1)) + (uint32_t)(kQ8Row * h);
  }
  __device__ __forceinline__ uint32_t lds() const { return byte + 16u * row; }   // pitch kQ8Pitch = 19 pieces
};
// piece i of thread tid; val: it is one of the value pieces
__device__ __forceinline__ MqPiece mq_piece(uint32_t rows, int tid, int i, bool val) {
  return {(rows >> (6 * i)) & 63u, 16u * (uint32_t)(tid + kThreads * i - (val ? 1152 : 0))};
}

template <bool KT, bool VT>
__device__ __forceinline__ void mq_load(const AttnArgs& p, int ts, int h, int tid, int wave, int lane, uint32_t rows,
                                        MqRegs<KT, VT>& r) {
  const uint64_t row0 = (uint64_t)(uint32_t)ts * (uint32_t)p.num_kv;
  const __amdgpu_buffer_rsrc_t rk = cache_rsrc(p.k, row0 * (KT ? kTq3Row : kQ8Row), p.kv_bytes);
  const __amdgpu_buffer_rsrc_t rv =
      cache_rsrc(p.v, row0 * (VT ? kTq3Row : kQ8Row), VT && !KT ? p.v_bytes : p.kv_bytes);
  asm volatile("" : "+v"(rows));
  auto piece = [&](int i, const __amdgpu_buffer_rsrc_t& rs, bool val) {
    return __builtin_amdgcn_raw_buffer_load_b128(rs, mq_piece(rows, tid, i, val).cache(p.num_kv, h), 0, 0);
  };
  const int row = tid >> 3, pc = tid & 7;
  const uint32_t toff =
      (uint32_t)(row * p.num_kv + h) * (uint32_t)kTq3Row + 52u * (uint32_t)(pc >> 2) + 4u + 12u * (uint32_t)(pc & 3);
  const uint32_t noff = (uint32_t)(lane * p.num_kv + h) * (uint32_t)kTq3Row + 52u * (uint32_t)(wave & 1);
  if constexpr (KT) {
    r.k = __builtin_amdgcn_raw_buffer_load_b96(rk, toff, 0, 0);
  } else {
    r.q[0] = piece(0, rk, false);
    r.q[1] = piece(1, rk, false);
  }
  if constexpr (VT) {
    if constexpr (!KT) {
      if (wave < 2) r.q[2] = piece(2, rk, false);   // pieces 1024 .. 1151
    }
    if (KT && wave < 2)
      r.nm = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rk, noff, 0, 0));
    else if (wave < 4 && wave >= 2)
      r.nm = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rv, noff, 0, 0));
    r.v = __builtin_amdgcn_raw_buffer_load_b96(rv, toff, 0, 0);
  } else {
    r.q[2] = wave < 2 ? piece(2, rk, false) : piece(2, rv, true);   // pieces 1024 .. 1535
    r.q[3] = piece(3, rv, true);
    if (wave < 4) r.q[4] = piece(4, rv, true);                      // pieces 2048 .. 2303
  }
}

// Four 6-bit fields (bits 0, 6, 12, 18 of w) as the four bytes of a dword.
__device__ __forceinline__ uint32_t spread6(uint32_t w) {
  const uint32_t y = ((w & 0xfff000u) << 4) | (w & 0xfffu);
  return ((y & 0x0fc00fc0u) << 2) | (y & 0x003f003fu);
}

// r's rows to staging buffer `buf`.  Rows [new_r, new_r + n_new) of the tile (fused
// append; n_new 0: none) come from their encoded blocks at enc instead.
template <bool KT, bool VT>
__device__ __forceinline__ void mq_stage(uint8_t* lds, int buf, int tid, int wave, int lane, uint32_t rows,
                                         MqRegs<KT, VT>& r, float scale2, const uint32_t* enc, int new_r, int n_new) {
  using L = MqLds<KT, VT>;
  uint8_t* kd = lds + L::kK + buf * L::kKBuf;
  uint8_t* vd = lds + L::kV + buf * L::kVBuf;
  asm volatile("" : "+v"(rows));
  auto put = [&](int i, uint8_t* d, bool val) {
    *reinterpret_cast<u4_t*>(d + mq_piece(rows, tid, i, val).lds()) = r.q[i];
  };
  const int row = tid >> 3, pc = tid & 7;
  if constexpr (KT) {
    if (n_new > 0) {   // (uniform)
      const int e = row - new_r, en = lane - new_r;
      if (e >= 0 && e < n_new) {
        const uint32_t* b = enc + (4 * e + (pc >> 2)) * 13 + 1 + 3 * (pc & 3);
        r.k = u3_t{b[0], b[1], b[2]};
        r.v = u3_t{b[26], b[27], b[28]};
      }
      if (wave < 4 && en >= 0 && en < n_new) r.nm = __uint_as_float(enc[(4 * en + wave) * 13]);
    }
    const u4_t w = {spread6(r.k[0]), spread6(__builtin_amdgcn_alignbyte(r.k[1], r.k[0], 3)),
                    spread6(__builtin_amdgcn_alignbyte(r.k[2], r.k[1], 2)), spread6(r.k[2] >> 8)};
    *reinterpret_cast<u4_t*>(kd + row * 128 + 16 * (pc ^ ((row >> 1) & 7))) = w;
  } else {
    put(0, kd, false);
    put(1, kd, false);
  }
  if constexpr (VT) {
    if constexpr (!KT) {
      if (wave < 2) put(2, kd, false);
    }
    if (wave < 4 && (KT || wave >= 2))
      *reinterpret_cast<float*>(lds + L::kNorm + ((buf * 4 + wave) * kTile + lane) * 4) = wave < 2 ? r.nm * scale2 : r.nm;
    // weights p * norm must stay inside fp16 with p up to 2^kSlack: a larger value
    // norm anywhere in the chunk ends the slack (p <= 1 from there on)
    if (wave == 2 || wave == 3) {
      if (__builtin_amdgcn_ballot_w64(r.nm > 128.0f) != 0 && lane == 0)
        *reinterpret_cast<int*>(lds + L::kCorr + 256 + 12) = 1;
    }
    uint32_t* d = reinterpret_cast<uint32_t*>(vd) + 4 * pc * kVgPitch + row;
    d[0] = r.v[0];
    d[kVgPitch] = __builtin_amdgcn_alignbyte(r.v[1], r.v[0], 3);
    d[2 * kVgPitch] = __builtin_amdgcn_alignbyte(r.v[2], r.v[1], 2);
    d[3 * kVgPitch] = r.v[2] >> 8;
  } else {
    put(2, wave < 2 ? kd : vd, wave >= 2);
    put(3, vd, true);
    if (wave < 4) put(4, vd, true);
  }
}

// Two int8 codes as fp16, times their scales.  x: the codes (biased to 0..255
// by flipping their sign bits) under the exponent byte 0x64, i.e. the fp16
// values 1024 + code + 128; the subtraction is exact and the product is the
// single rounding half(q * d) of the reference.
__device__ __forceinline__ uint32_t q8_pair(uint32_t x, h2_t d) {
  h2_t v = __builtin_bit_cast(h2_t, x) - h2_t{(_Float16)1152.0f, (_Float16)1152.0f};
  v = v * d;
  return __builtin_bit_cast(uint32_t, v);
}

// A operand of score slice S: block S >> 2 of the lane's two (18 dwords: 8 code
// dwords and pad|scale each), elements 8 (S & 3) .. + 7
template <int S>
__device__ __forceinline__ h8_t q8_key_operand(const uint32_t (&k)[18]) {
  constexpr int base = 9 * (S >> 2) + 2 * (S & 3);
  const _Float16 d1 = __builtin_bit_cast(h2_t, k[9 * (S >> 2) + 8])[1];
  const h2_t d = {d1, d1};
  const uint32_t w0 = k[base] ^ 0x80808080u, w1 = k[base + 1] ^ 0x80808080u;
  const u4_t v = {q8_pair(__builtin_amdgcn_perm(0x64646464u, w0, 0x04010400u), d),
                  q8_pair(__builtin_amdgcn_perm(0x64646464u, w0, 0x04030402u), d),
                  q8_pair(__builtin_amdgcn_perm(0x64646464u, w1, 0x04010400u), d),
                  q8_pair(__builtin_amdgcn_perm(0x64646464u, w1, 0x04030402u), d)};
  return __builtin_bit_cast(h8_t, v);
}

// Two centroids of code pair byte B of w (bytes of pair indexes) from the table.
template <int B>
__device__ __forceinline__ uint32_t pair_read(const uint8_t* lds, uint32_t w, uint32_t lane4) {
  return *reinterpret_cast<const uint32_t*>(lds + __builtin_amdgcn_perm(w, lane4, 0x0c0c0000u | (4u + B) << 8));
}

// NG: 16-column groups of a workgroup, 2 or 4.
// SPLIT: the split API.  The chunk is a reference split, whose partials (true maximum
// in natural-log units, sum, unnormalised row in the caller's coordinates) go to
// part_m / part_l / part_o.
// SW: a sink or a window (TQ3 caches).
template <bool KT, bool VT, int NG, bool SPLIT, bool SW = false>
__global__ __launch_bounds__(kThreads, 1) void mq_attn_kernel(QKV_ATTN_LEAD_PARAMS, AttnArgs pin) {
  QKV_ATTN_LEAD_APPLY(p, pin);
  static_assert((!KT || VT) && (KT || !SW), "TQ3 keys come with TQ3 values, sinks and windows with TQ3 keys");
  using L = MqLds<KT, VT>;
  __shared__ __attribute__((aligned(16))) uint8_t lds[L::kEnd];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int gqa = __builtin_amdgcn_readfirstlane(p.num_q / p.num_kv);
  // work id, XCD-aware: the num_kv workgroups of one (query block, chunk) share an XCD
  int h, t0, chunk;
  {
    const int Lid = blockIdx.x;
    const int xcd = Lid & 7, r = Lid >> 3;
    h = r % p.num_kv;
    const int g = (r / p.num_kv) * 8 + xcd;
    const int groups = (p.sub_n + p.qpw - 1) / p.qpw;
    if (g >= groups * p.n_chunks) return;
    const int tq = g / p.n_chunks;
    chunk = g - tq * p.n_chunks;
    t0 = tq * p.qpw;
  }
  const int nq = min(p.qpw, p.sub_n - t0);
  const int cols = __builtin_amdgcn_readfirstlane(nq * gqa);   // <= 64
  const int n = lane & 15, kb = lane >> 4;
  // scores: 16 keys 16 kg .. of a tile, kCg column groups from kCg * ch on
  constexpr int kCg = NG / 2;
  const int kg = wave & 3, ch = wave >> 2;
  // ---- queries.  Q8_0 keys: slice s of column c0 + 16 cg straight into
  // the operand registers, dims 32 (2 kb + (s >> 2)) + 8 (s & 3) .. + 7 (the
  // lane's two Q8_0 blocks).  TQ3 keys: 32 NG WHTs of 128 (columns x
  // 2 blocks), 16 lanes each, NG per thread, rotated below.
  u4_t qa[kCg][8];
  u4_t q_raw[NG];
  const int c0 = 16 * kCg * ch + n;   // this lane's score columns: c0 (+ 16)
  const int q_part = tid & 15;
  {
    const uint32_t q_extent = (uint32_t)(p.sub_n * p.num_q * kHD * 2);
    const __amdgpu_buffer_rsrc_t rq =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.q), 0, q_extent, kBufferRsrcWord3);
    auto q_row = [&](int c) {   // (columns past `cols`: zero queries, never stored)
      return c < cols ? (uint32_t)(((t0 + c / gqa) * p.num_q + h * gqa + c % gqa) * kHD * 2) : q_extent;
    };
    if constexpr (KT) {
#pragma unroll
      for (int i = 0; i < NG; i++) {
        const int wi = (tid >> 4) + 32 * i;
        q_raw[i] = __builtin_amdgcn_raw_buffer_load_b128(rq, q_row(wi >> 1) + 256 * (wi & 1) + 16 * q_part, 0, 0);
      }
    } else {
#pragma unroll
      for (int cg = 0; cg < kCg; cg++) {
        const uint32_t off = q_row(c0 + 16 * cg) + 128 * kb;
#pragma unroll
        for (int s = 0; s < 8; s++) qa[cg][s] = __builtin_amdgcn_raw_buffer_load_b128(rq, off + 16 * s, 0, 0);
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- key range of the workgroup
  const int active_last = p.start_pos + t0 + nq;
  int lo = chunk * p.chunk_keys;
  const int c_end = !SPLIT && chunk == p.n_chunks - 1 ? active_last : lo + p.chunk_keys;
  int hi = min(c_end, active_last), hi_first = min(c_end, p.start_pos + t0 + 1);
  lo = __builtin_amdgcn_readfirstlane(lo);
  hi = __builtin_amdgcn_readfirstlane(hi);
  hi_first = __builtin_amdgcn_readfirstlane(hi_first);
  int n_tiles = hi > lo ? (hi - lo + kTile - 1) / kTile : 0;
  // ---- the sink / window rule (KeyRule), by tile where all columns agree: the tiles
  // that none sees (past the sink, before the first query's window) are one range, left
  // out of the walk; of the others, those that every column sees need no rule.  (An
  // instance of its own: even this much costs other calls 1%, a branch in the loop 3.5%:
  // 16 queries over 131,072 keys 83.4, 84.1 and 87.0 us.)
  int skip_from = 0, skip_keys = 0;
  if constexpr (SW) {
    const int seen_from = p.start_pos + t0 + 1 - p.window_tok;
    const int first = p.sink_tok > lo ? (p.sink_tok - lo - 1) / kTile + 1 : 0;
    const int past = seen_from > lo ? min(n_tiles, (seen_from - lo) / kTile) : 0;
    const int out = __builtin_amdgcn_readfirstlane(max(past - first, 0));
    skip_from = __builtin_amdgcn_readfirstlane(first);
    skip_keys = out * kTile;
    n_tiles -= out;
  }
  auto tile_key = [&](int t) { return lo + t * kTile + (SW && t >= skip_from ? skip_keys : 0); };
  auto sw_all = [&](int t32) { return t32 < p.sink_tok || t32 + 32 > active_last - p.window_tok; };
  // ---- fused append (qkv_decode_attn_tq3_append): the new keys start_pos ..
  // that this workgroup reads, [new_lo, new_lo + n_new), are encoded here
  // (tq3_encode_row16, the small append's arithmetic), 32 blocks per round, and
  // take the place of their (stale) cache rows when their tile is staged; the
  // last query group's workgroups also store them to the caches.
  int new_lo = 0, n_new = 0;
  if constexpr (KT) {
    if (p.k_new != nullptr && hi > max(lo, p.start_pos)) {
      new_lo = max(lo, p.start_pos);
      n_new = hi - new_lo;   // <= sub_n <= 64 (the host takes this path only then)
    }
    new_lo = __builtin_amdgcn_readfirstlane(new_lo);
    n_new = __builtin_amdgcn_readfirstlane(n_new);
  }
  auto enc_input = [&](int round) {
    const int j = 32 * round + (tid >> 4), t = tid & 15;
    uint4 raw = make_uint4(0u, 0u, 0u, 0u);
    if (j < 4 * n_new) {
      const int tv = (j >> 1) & 1, blk = j & 1;
      const uint16_t* src = (tv ? p.v_new : p.k_new) +
                            ((long)(new_lo + (j >> 2) - p.start_pos) * p.num_kv + h) * kHD + blk * 128 + 8 * t;
      raw = *reinterpret_cast<const uint4*>(src);
    }
    return raw;
  };
  uint4 enc_raw0 = make_uint4(0u, 0u, 0u, 0u), enc_raw1 = make_uint4(0u, 0u, 0u, 0u);
  if (KT && n_new > 0) enc_raw0 = enc_input(0);
  if (KT && n_new > 8) enc_raw1 = enc_input(1);
  uint32_t* enc = reinterpret_cast<uint32_t*>(lds + L::kEnc);

  const uint32_t rows = mq_rows<KT, VT>(tid);
  MqRegs<KT, VT> ra, rb;
  if (n_tiles > 0) mq_load<KT, VT>(p, tile_key(0), h, tid, wave, lane, rows, ra);
  if (n_tiles > 1) mq_load<KT, VT>(p, tile_key(1), h, tid, wave, lane, rows, rb);
  const uint32_t lane4 = 4u * (uint32_t)lane;
  if constexpr (VT) {
    // table: wave w writes every lane's copy of entries 8 w .. 8 w + 7
    const uint32_t hi16 = centroid_scaled_h((uint32_t)wave) << 16;
#pragma unroll
    for (int e = 0; e < 8; e++)
      *reinterpret_cast<uint32_t*>(lds + (8 * wave + e) * 256 + lane4) = centroid_scaled_h((uint32_t)e) | hi16;
  }
  int* flag_s = reinterpret_cast<int*>(lds + L::kCorr + 256);
  if (tid < 4) flag_s[tid] = 0;   // tiles' raise flags, and the sticky large-norm flag
  if constexpr (VT) __syncthreads();
  // the key norms carry the softmax scale and undo the table's
  const float scale2 = __uint_as_float(__builtin_amdgcn_readfirstlane(
      __float_as_uint(KT ? p.scale_log2 * kCenScaleInv : p.scale_log2)));   // (scalar register)
  u4_t ql[kCg][8];   // TQ3 keys: remainders of the rotated queries
  if constexpr (KT) {
    const uint32_t sbits = sign_word_sel(q_part >> 2) >> (8 * (q_part & 3));   // elements part*8..+7
    const float rs = wht_scale();
#pragma unroll
    for (int i = 0; i < NG; i++) {
      const int wi = (tid >> 4) + 32 * i, c = wi >> 1, jb = wi & 1;
      float x[8];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        x[2 * e] = h2f(q_raw[i][e] & 0xffffu);
        x[2 * e + 1] = h2f(q_raw[i][e] >> 16);
      }
#pragma unroll
      for (int e = 0; e < 8; e++) x[e] = ((sbits >> e) & 1u) ? x[e] : -x[e];
      wht8_inreg(x);
      wht_xor_lanes16(x, lane);
      uint32_t pk[4], pl[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float a = x[2 * e] * rs, b = x[2 * e + 1] * rs;
        const uint32_t ha = f2h(a), hb = f2h(b);
        pk[e] = ha | (hb << 16);
        pl[e] = f2h(a - h2f(ha)) | (f2h(b - h2f(hb)) << 16);
      }
      const int qb = c * 512 + 256 * jb + 16 * (q_part ^ (c & 15));
      *reinterpret_cast<uint4*>(lds + L::kQhi + qb) = make_uint4(pk[0], pk[1], pk[2], pk[3]);
      *reinterpret_cast<uint4*>(lds + L::kQlo + qb) = make_uint4(pl[0], pl[1], pl[2], pl[3]);
    }
    if (n_new > 0) {
      const bool store = t0 + nq == p.sub_n;   // the last query group stores the rows
      for (int round = 0; 32 * round < 4 * n_new; round++) {
        const uint4 raw = round == 0 ? enc_raw0 : round == 1 ? enc_raw1 : enc_input(round);
        const uint32_t word = tq3_encode_row16(raw, lane);
        const int j = 32 * round + (tid >> 4), t = tid & 15;
        if (j < 4 * n_new && t <= 12) {
          const int w = t == 12 ? 0 : 1 + t;
          enc[j * 13 + w] = word;
          if (store) {
            const int tv = (j >> 1) & 1, blk = j & 1;
            uint32_t* dst = reinterpret_cast<uint32_t*>(tv ? p.v_w : p.k_w) +
                            ((long)(new_lo + (j >> 2)) * p.num_kv + h) * 26 + blk * 13 + w;
            *dst = word;
          }
        }
      }
    }
    __syncthreads();
    // slice s = 4 j + u of column c0 + 16 cg: dims 128 j + 8 (4 kb + u) .. + 7
    // (the lane's 12-byte piece kb of key block j)
#pragma unroll
    for (int cg = 0; cg < kCg; cg++)
#pragma unroll
      for (int s = 0; s < 8; s++) {
        const int c = c0 + 16 * cg;
        const int qb = c * 512 + 256 * (s >> 2) + 16 * ((4 * kb + (s & 3)) ^ n);
        qa[cg][s] = *reinterpret_cast<const u4_t*>(lds + L::kQhi + qb);
        ql[cg][s] = *reinterpret_cast<const u4_t*>(lds + L::kQlo + qb);
      }
    __syncthreads();   // the query scratch is read: the staging buffers are free
  }
  // tiles before this key are seen whole by every column, as far as the end of its keys
  // and the tree bits (keys past start_pos) go
  const int dense_end = KT && p.tree_mask != nullptr ? min(hi_first, p.start_pos) : hi_first;
  // (opaque thread indexes: the offsets of staging and loads are formed at each
  // use instead of being held in registers through the loop)
  auto stage = [&](int ts, int buf, MqRegs<KT, VT>& r) {
    const int n_in = KT && n_new > 0 && ts + kTile > new_lo ? n_new : 0;
    int ti = tid;
    asm volatile("" : "+v"(ti));
    mq_stage<KT, VT>(lds, buf, ti, wave, ti & 63, rows, r, scale2, enc, new_lo - ts, n_in);
  };
  auto load = [&](int ts, MqRegs<KT, VT>& r) {
    int ti = tid;
    asm volatile("" : "+v"(ti));
    mq_load<KT, VT>(p, ts, h, ti, wave, ti & 63, rows, r);
  };
  // tiles 0 and 1 staged, tile 2 on its way
  if (n_tiles > 0) stage(tile_key(0), 0, ra);
  if (n_tiles > 1) stage(tile_key(1), 1, rb);
  if (n_tiles > 2) load(tile_key(2), ra);
  __syncthreads();

  // (a reference that no visible score has touched yet is kNoRef, not -inf: the
  // weights of masked keys are then 0 without a test)
  float m2[kCg], lsum[kCg];
  float mt[kCg];   // SPLIT: this lane's part of the columns' maxima
#pragma unroll
  for (int cg = 0; cg < kCg; cg++) {
    m2[cg] = kNoRef;
    mt[cg] = -INFINITY;
    lsum[cg] = 0.0f;
  }
  f4_t acc[NG][2];
#pragma unroll
  for (int g = 0; g < NG; g++) acc[g][0] = acc[g][1] = f4_t{0.f, 0.f, 0.f, 0.f};
  float* mx = reinterpret_cast<float*>(lds + L::kMx);
  float* corr_s = reinterpret_cast<float*>(lds + L::kCorr);
  // this lane's dims of the value product: 32 wave + 2 n and + 1.
  // TQ3: the 6-bit field of the dim, rotated to bits 8..13 of a table address
  const uint32_t vrot0 = (6u * (uint32_t)(n & 3) + 24u) & 31u, vrot1 = (6u * (uint32_t)(n & 3) + 27u) & 31u;
  // Q8_0: bytes 2 (n & 1) (and + 1) of the lane's dim quad in two keys' dwords
  const uint32_t vsel0 = 0x0c000c00u + 0x00040000u + 0x00010001u * (uint32_t)(2 * (n & 1));
  const uint32_t vsel1 = vsel0 + 0x00010001u;

  // unit kb of row n (16-byte units swizzled with the row), unit 4 + kb at ^ 64:
  // this lane's probabilities, and in row 16 kg + n its key piece
  const uint32_t p_at = (uint32_t)(n * 128 + 16 * (kb ^ ((n >> 1) & 7)));
  const uint32_t k_at = p_at + (uint32_t)(16 * kg * 128);
  // tile t's staging buffer and flag, those of t + 1 and of t + 2
  int b0 = 0, b1 = 1, b2 = 2;
  float slack = kSlack<VT>;
  for (int t = 0; t < n_tiles; t++) {
    const int ts = tile_key(t);
    const uint8_t* kbuf = lds + L::kK + b0 * L::kKBuf;
    const uint8_t* vbuf = lds + L::kV + b0 * L::kVBuf;
    const float* knorm = reinterpret_cast<const float*>(lds + L::kNorm) + b0 * 4 * kTile;
    uint8_t* pbuf = lds + L::kP + (t & 1) * L::kPBuf;
    bool dense = ts + kTile <= dense_end;
    if constexpr (SW) dense = dense && sw_all(ts) && sw_all(ts + 32);
    bool v_nonfinite = false;
    if constexpr (!VT) {
      // the scales of this wave's value block, one key per lane, to the wave's own area
      const uint32_t d = *reinterpret_cast<const uint16_t*>(vbuf + lane * kQ8Pitch + 36 * wave + 34);
      *reinterpret_cast<uint16_t*>(lds + L::kSc + (wave * kTile + lane) * 2) = (uint16_t)d;
      v_nonfinite = __builtin_amdgcn_ballot_w64((d & 0x7c00u) == 0x7c00u) != 0;
    }
    // ---- scores: D rows = keys 16 kg + 4 kb + r, D column = c0 + 16 cg
    // norms of the lane's keys 16 kg + 4 kb ..: key blocks (x scale), value blocks
    struct Norms {
      f4_t n[2];
    };
    auto norms = [&](int first) {
      Norms nm;
#pragma unroll
      for (int j = 0; j < 2; j++) nm.n[j] = *reinterpret_cast<const f4_t*>(knorm + (first + j) * kTile + 16 * kg + 4 * kb);
      return nm;
    };
    f4_t sa[kCg][KT ? 2 : 1];   // [column group][128-block]
#pragma unroll
    for (int cg = 0; cg < kCg; cg++)
#pragma unroll
      for (int j = 0; j < (KT ? 2 : 1); j++) sa[cg][j] = f4_t{0.f, 0.f, 0.f, 0.f};
    if constexpr (KT) {
      u4_t w[2];
#pragma unroll
      for (int j = 0; j < 2; j++) w[j] = *reinterpret_cast<const u4_t*>(kbuf + (k_at ^ (64 * j)));
      // table reads one step (u, j) ahead of their products
      auto operand = [&](int st) {
        const uint32_t x = w[st & 1][st >> 1];
        return __builtin_bit_cast(h8_t, u4_t{pair_read<0>(lds, x, lane4), pair_read<1>(lds, x, lane4),
                                             pair_read<2>(lds, x, lane4), pair_read<3>(lds, x, lane4)});
      };
      h8_t a[2] = {operand(0), operand(1)};
#pragma unroll
      for (int st = 0; st < 8; st++) {   // u = st >> 1, j = st & 1
        const h8_t cur = a[st & 1];
        if (st + 2 < 8) a[st & 1] = operand(st + 2);
        const int j = st & 1, sl = 4 * j + (st >> 1);
#pragma unroll
        for (int cg = 0; cg < kCg; cg++)
          sa[cg][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cur, __builtin_bit_cast(h8_t, qa[cg][sl]), sa[cg][j], 0, 0, 0);
#pragma unroll
        for (int cg = 0; cg < kCg; cg++)
          sa[cg][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(cur, __builtin_bit_cast(h8_t, ql[cg][sl]), sa[cg][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      uint32_t k[18];
      const u2_t* kr = reinterpret_cast<const u2_t*>(kbuf + (16 * kg + n) * kQ8Pitch + 72 * kb);
#pragma unroll
      for (int i = 0; i < 9; i++) {
        const u2_t c = kr[i];
        k[2 * i] = c[0];
        k[2 * i + 1] = c[1];
      }
      auto slice = [&](auto S) {
        constexpr int si = decltype(S)::value;
        const h8_t a = q8_key_operand<si>(k);
#pragma unroll
        for (int cg = 0; cg < kCg; cg++)
          sa[cg][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, __builtin_bit_cast(h8_t, qa[cg][si]), sa[cg][0], 0, 0, 0);
      };
      slice(std::integral_constant<int, 0>{});
      slice(std::integral_constant<int, 1>{});
      slice(std::integral_constant<int, 2>{});
      slice(std::integral_constant<int, 3>{});
      slice(std::integral_constant<int, 4>{});
      slice(std::integral_constant<int, 5>{});
      slice(std::integral_constant<int, 6>{});
      slice(std::integral_constant<int, 7>{});
    }
    // score of key 16 kg + 4 kb + r minus x (log2 units)
    auto score = [&](const Norms& kn, int cg, int r, float x) {
      if constexpr (KT) return __builtin_fmaf(kn.n[1][r], sa[cg][1][r], __builtin_fmaf(kn.n[0][r], sa[cg][0][r], -x));
      else return __builtin_fmaf(sa[cg][0][r], scale2, -x);
    };
    // Whether the wave's keys are visible to column c0 + 16 cg, bit r.  (Formed
    // from opaque values, so that no part of it moves into the common path.)
    auto visible = [&](int cg) {
      int c = c0 + 16 * cg, k0 = ts;
      asm volatile("" : "+v"(c), "+s"(k0));
      const int tq = t0 + min(c / gqa, nq - 1), end = p.start_pos + tq + 1;
      const KeyRule rule(p.start_pos, tq, SW ? p.sink_tok : 0, SW ? p.window_tok : 0, KT ? p.tree_mask : nullptr);
      uint32_t bits = 0u;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int key = k0 + 16 * kg + 4 * kb + r;
        const bool vis = key < min(c_end, end) && (!KT || rule.visible(key, end));
        bits |= vis ? 1u << r : 0u;
      }
      return bits;
    };
    // probabilities of the wave's 16 keys to LDS: column c's 16-byte unit
    // (half kg >> 1, kb), stored at unit ^ ((c >> 1) & 7), holds keys
    // 32 (kg >> 1) + 4 kb + 0..3 and + 16..19 (the k order of the value product).
    // Returns the largest score above the reference.
    float ps[kCg], tl[kCg];   // (tl, SPLIT: the columns' maxima above the reference)
    uint8_t* pd = pbuf + c0 * 128 + 16 * (((kg >> 1) * 4 + kb) ^ ((c0 >> 1) & 7)) + 8 * (kg & 1);
    auto put_p = [&](auto DENSE) {
      constexpr bool all = decltype(DENSE)::value;
      uint32_t vis[kCg];
      if constexpr (!all) {
#pragma unroll
        for (int cg = 0; cg < kCg; cg++) {
          vis[cg] = visible(cg);
          __builtin_amdgcn_sched_barrier(0);   // (one column's rule in registers at a time)
        }
      }
      Norms kn, vn;
      if constexpr (KT) kn = norms(0);
      if constexpr (VT) vn = norms(2);
      float top = -INFINITY;
#pragma unroll
      for (int cg = 0; cg < kCg; cg++) {
        float d[4], pr[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          d[r] = score(kn, cg, r, m2[cg]);
          if constexpr (!all) d[r] = (vis[cg] >> r & 1u) ? d[r] : -INFINITY;
        }
        tl[cg] = fmaxf(fmaxf(d[0], d[1]), fmaxf(d[2], d[3]));
        top = fmaxf(top, tl[cg]);
#pragma unroll
        for (int r = 0; r < 4; r++) pr[r] = __builtin_amdgcn_exp2f(d[r]);
        ps[cg] = (pr[0] + pr[1]) + (pr[2] + pr[3]);
        if constexpr (VT) {
#pragma unroll
          for (int j = 0; j < 2; j++) {
            h4_t w;
#pragma unroll
            for (int r = 0; r < 4; r++) {
              float x = pr[r] * vn.n[j][r];
              // (a masked key's norm may be inf or NaN: its weight is 0)
              if constexpr (!all) x = d[r] == -INFINITY ? 0.0f : x;
              w[r] = (_Float16)x;
            }
            *reinterpret_cast<h4_t*>(pd + 2048 * cg + j * 64 * 128) = w;
          }
        } else {
          h4_t w, rest;
#pragma unroll
          for (int r = 0; r < 4; r++) {
            w[r] = (_Float16)pr[r];
            rest[r] = (_Float16)(pr[r] - (float)w[r]);
          }
          *reinterpret_cast<h4_t*>(pd + 2048 * cg) = w;
          *reinterpret_cast<h4_t*>(pd + 64 * 128 + 2048 * cg) = rest;
        }
      }
      return top;
    };
    bool raised = false;
    for (;;) {
      const float top = dense ? put_p(std::true_type{}) : put_p(std::false_type{});
      if (!raised && __builtin_amdgcn_ballot_w64(top > slack) != 0 && lane == 0) flag_s[b0] = 1;
      __syncthreads();   // probabilities and flag are in; buffer b2 is free
      if (raised || !__builtin_amdgcn_readfirstlane(flag_s[b0])) break;
      // some column's maximum rose past the slack: every column's reference
      // becomes its running maximum (rounded up, minus kHead), the sums (and, below, the accumulators) are
      // rescaled, and the tile's probabilities are formed again
      raised = true;
      uint32_t vis[kCg];
#pragma unroll
      for (int cg = 0; cg < kCg; cg++) {
        vis[cg] = visible(cg);
        __builtin_amdgcn_sched_barrier(0);
      }
      Norms kn;
      if constexpr (KT) kn = norms(0);
      int c1 = c0;
      asm volatile("" : "+v"(c1));   // (the addresses of this path are not held through the loop)
#pragma unroll
      for (int cg = 0; cg < kCg; cg++) {
        float mt = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; r++) mt = fmaxf(mt, (vis[cg] >> r & 1u) ? score(kn, cg, r, 0.0f) : -INFINITY);
        mt = xrow_max(mt);
        if (kb == 0) mx[(c1 + 16 * cg) * 4 + kg] = mt;
      }
      __syncthreads();
#pragma unroll
      for (int cg = 0; cg < kCg; cg++) {
        const f4_t mk = *reinterpret_cast<const f4_t*>(mx + 4 * (c1 + 16 * cg));
        // (a whole number: every rescale is by an exact power of two)
        const float mm = fmaxf(fmaxf(mk[0], mk[1]), fmaxf(mk[2], mk[3]));
        const float mn = fmaxf(m2[cg], __builtin_ceilf(mm) - kHead<VT>);
        if constexpr (SPLIT) mt[cg] = fmaxf(mt[cg], mm);   // (an infinite one shows only here)
        const float corr = __builtin_amdgcn_exp2f(m2[cg] - mn);
        lsum[cg] *= corr;
        m2[cg] = mn;
        if (kg == 0 && kb == 0) corr_s[c1 + 16 * cg] = corr;
      }
    }
    if (raised) {
      int kb4 = 4 * kb;
      asm volatile("" : "+v"(kb4));
#pragma unroll
      for (int g = 0; g < NG; g++) {
        const f4_t cr = *reinterpret_cast<const f4_t*>(corr_s + 16 * g + kb4);
#pragma unroll
        for (int e = 0; e < 2; e++)
#pragma unroll
          for (int r = 0; r < 4; r++) acc[g][e][r] *= cr[r];
      }
    }
    if constexpr (VT) slack = __builtin_amdgcn_readfirstlane(flag_s[3]) ? 0.0f : kSlack<VT>;
    if (t + 2 < n_tiles) {
      stage(tile_key(t + 2), b2, ra);
      if (t + 3 < n_tiles) load(tile_key(t + 3), ra);
    }
    if (tid == 0) flag_s[b2] = 0;   // (set by tile t + 2, after the next barrier)
#pragma unroll
    for (int cg = 0; cg < kCg; cg++) {
      lsum[cg] += ps[cg];
      if constexpr (SPLIT) mt[cg] = fmaxf(mt[cg], tl[cg] + m2[cg]);
    }
    // ---- values: acc[g][e] += P(16 columns x 32 keys) V(32 keys x 16 dims)
    const uint8_t* pbase = pbuf + (VT ? (wave >> 2) * 64 * 128 : 0);
    auto p_operand = [&](int g, int c2, int rest = 0) {   // columns 16 g + n, keys of half c2
      return *reinterpret_cast<const h8_t*>(pbase + rest * 64 * 128 + 16 * g * 128 + (p_at ^ (64 * c2)));
    };
    // B operands of half c2: dims 32 wave + 2 n (bv[0]) and + 1 (bv[1])
    auto v_operands = [&](int c2, u4_t (&bv)[2]) {
      if constexpr (VT) {
        const uint32_t* vr = reinterpret_cast<const uint32_t*>(vbuf) + (4 * wave + (n >> 2)) * kVgPitch + 32 * c2 + 4 * kb;
        const u4_t xa = *reinterpret_cast<const u4_t*>(vr), xb = *reinterpret_cast<const u4_t*>(vr + 16);
        uint32_t x[8] = {xa[0], xa[1], xa[2], xa[3], xb[0], xb[1], xb[2], xb[3]};
        interleave_pairs(x);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          bv[0][i] = *reinterpret_cast<const uint32_t*>(lds + ((__builtin_amdgcn_alignbit(x[i], x[i], vrot0) & 0x3f00u) | lane4));
          bv[1][i] = *reinterpret_cast<const uint32_t*>(lds + ((__builtin_amdgcn_alignbit(x[4 + i], x[4 + i], vrot1) & 0x3f00u) | lane4));
        }
      } else {
        uint32_t x[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const int key = 32 * c2 + 4 * kb + (i & 3) + 16 * (i >> 2);
          x[i] = *reinterpret_cast<const uint32_t*>(vbuf + key * kQ8Pitch + 36 * wave + 4 * (n >> 1));
        }
        const uint8_t* sc = lds + L::kSc + (wave * kTile + 32 * c2 + 4 * kb) * 2;
        const u2_t da = *reinterpret_cast<const u2_t*>(sc), db = *reinterpret_cast<const u2_t*>(sc + 32);
        const uint32_t d[4] = {da[0], da[1], db[0], db[1]};
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const h2_t dd = __builtin_bit_cast(h2_t, d[i]);
          bv[0][i] = q8_pair(__builtin_amdgcn_perm(x[2 * i + 1], x[2 * i], vsel0) ^ 0x64806480u, dd);
          bv[1][i] = q8_pair(__builtin_amdgcn_perm(x[2 * i + 1], x[2 * i], vsel1) ^ 0x64806480u, dd);
        }
      }
    };
    if (!VT && v_nonfinite) {
      // a key with an inf or NaN scale: 0 * inf must not reach the rows of a query
      // that does not see it, nor 0 be the rest of a weight there, so every query
      // takes products of its own, of the weights alone, with the keys that it does
      // not see zeroed
#pragma unroll 1
      for (int it = 0; it < 2 * nq; it++) {
        const int c2 = it & 1, qi = it >> 1;
        const int q_end = min(hi, p.start_pos + t0 + qi + 1);
        u4_t bv[2];
        v_operands(c2, bv);
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int key = ts + 32 * c2 + 4 * kb + 2 * (i & 1) + 16 * (i >> 1);
          const uint32_t keep = (key < q_end ? 0xffffu : 0u) | (key + 1 < q_end ? 0xffff0000u : 0u);
          bv[0][i] &= keep;
          bv[1][i] &= keep;
        }
#pragma unroll
        for (int g = 0; g < NG; g++) {
            const h8_t pa = p_operand(g, c2);
#pragma unroll
            for (int e = 0; e < 2; e++) {
              const f4_t o = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa, __builtin_bit_cast(h8_t, bv[e]),
                                                                    f4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
              for (int r = 0; r < 4; r++)
                if ((16 * g + 4 * kb + r) / gqa == qi) acc[g][e][r] += o[r];
            }
          }
      }
    } else {
#pragma unroll
      for (int c2 = 0; c2 < 2; c2++) {
        u4_t bv[2];
        v_operands(c2, bv);
#pragma unroll
        for (int part = 0; part < (VT ? 1 : 2); part++) {   // Q8_0 values: the weights, then their rests
          h8_t pa[NG];
#pragma unroll
          for (int g = 0; g < NG; g++) pa[g] = p_operand(g, c2, part);
#pragma unroll
          for (int g = 0; g < NG; g++)
#pragma unroll
            for (int e = 0; e < 2; e++)
              acc[g][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa[g], __builtin_bit_cast(h8_t, bv[e]), acc[g][e], 0, 0, 0);
        }
      }
    }
    const int b = b0;
    b0 = b1;
    b1 = b2;
    b2 = b;
  }

  // (indexes of the rest of the kernel formed here, not held through the loop)
  int tid_e = tid;
  asm volatile("" : "+v"(tid_e));
  const int n_e = tid_e & 15, kb_e = (tid_e & 63) >> 4;
  // ---- records (SPLIT: partials): the waves of a column half hold its sums per key group, every
  // wave its dims of every column
  __syncthreads();
  float* sums = reinterpret_cast<float*>(lds + L::kSum);
  uint32_t* recs = reinterpret_cast<uint32_t*>(lds + L::kSum + 5 * 64 * 4);   // (byte offsets up to 4 GiB)
  const __amdgpu_buffer_rsrc_t rml = __builtin_amdgcn_make_buffer_rsrc(p.ws_ml, 0, p.ws_ml_bytes, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(p.ws_o, 0, p.ws_o_bytes, kBufferRsrcWord3);
  int gqa_m = gqa;
  asm volatile("" : "+s"(gqa_m));   // (its reciprocal is formed here, not held through the loop)
#pragma unroll
  for (int cg = 0; cg < kCg; cg++) {
    const float l = xrow_sum(lsum[cg]);
    const int c = 16 * (kCg * ch + cg) + n_e;
    if (kb_e == 0) {
      sums[kg * 64 + c] = l;
      if (kg == 0) sums[4 * 64 + c] = m2[cg];
    }
    if constexpr (SPLIT) {
      const float m = xrow_max(mt[cg]);
      if (kb_e == 0) sums[(6 + kg) * 64 + c] = m;
    }
  }
  if constexpr (SPLIT) {
    __syncthreads();
    // rows scaled from the reference to the maximum, and rotated back (TQ3 values)
    auto column_max = [&](int c) {
      return fmaxf(fmaxf(sums[6 * 64 + c], sums[7 * 64 + c]), fmaxf(sums[8 * 64 + c], sums[9 * 64 + c]));
    };
    auto factor = [&](int c) {
      const float m = column_max(c);
      return m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(sums[4 * 64 + c] - m);
    };
    auto row_index = [&](int c) {
      return ((long)(h * gqa_m + c % gqa_m) * p.sub_n_max + t0 + c / gqa_m) * p.k_splits + chunk;
    };
    if (tid_e < cols) {
      const float m = column_max(tid_e), f = factor(tid_e);
      const long at = row_index(tid_e);
      p.part_m[at] = m == -INFINITY ? -INFINITY : m * kLn2;
      p.part_l[at] = f * ((sums[tid_e] + sums[64 + tid_e]) + (sums[128 + tid_e] + sums[192 + tid_e]));
    }
    typedef float f2a4_t __attribute__((ext_vector_type(2), aligned(4)));
    float* rows_s = reinterpret_cast<float*>(lds + L::kRows);
#pragma unroll
    for (int g = 0; g < NG; g++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int R = 16 * g + 4 * kb_e + r;
        if (R >= cols) continue;
        const float f = factor(R);
        if constexpr (VT)
          *reinterpret_cast<f2_t*>(rows_s + R * L::kRowPitch + 32 * wave + 2 * n_e) = f2_t{acc[g][0][r], acc[g][1][r]} * f;
        else
          *reinterpret_cast<f2a4_t*>(p.part_o + row_index(R) * kHD + 32 * wave + 2 * n_e) =
              f2a4_t{acc[g][0][r] * f, acc[g][1][r] * f};
      }
    if constexpr (VT) {
      __syncthreads();
      const int part = tid_e & 15;
      const uint32_t sbits = sign_word_sel(part >> 2) >> (8 * (part & 3));   // elements part*8..+7
      const float rs = wht_scale();
      for (int u0 = 0; u0 < 2 * cols; u0 += kThreads / 16) {
        const int u = u0 + (tid_e >> 4), R = u >> 1, blk = u & 1;
        const bool live = u < 2 * cols;
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; e++)   // the centroid table is scaled by kCenScale: undo it here
          x[e] = live ? rows_s[R * L::kRowPitch + blk * 128 + part * 8 + e] * kCenScaleInv : 0.0f;
        wht8_inreg(x);
        wht_xor_lanes16(x, tid_e & 63);
        if (!live) continue;
        float* o = p.part_o + row_index(R) * kHD + blk * 128 + part * 8;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float v = x[e] * rs;
          o[e] = ((sbits >> e) & 1u) ? v : -v;
        }
      }
    }
    return;
  }
  if (tid_e < 64) recs[tid_e] = (uint32_t)rec_index(p, h * gqa_m + tid_e % gqa_m, t0 + min(tid_e, cols - 1) / gqa_m, chunk);
  __syncthreads();
#pragma unroll
  for (int g = 0; g < NG; g++) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int R = 16 * g + 4 * kb_e + r;
      if (R < cols)
        __builtin_amdgcn_raw_buffer_store_b64(f2_t{acc[g][0][r], acc[g][1][r]}, ro,
                                              (recs[R] * kHD + (uint32_t)(32 * wave + 2 * n_e)) * 4u, 0, kCoherent);
    }
  }
  if (tid_e < cols) {
    const float l = (sums[tid_e] + sums[64 + tid_e]) + (sums[128 + tid_e] + sums[192 + tid_e]);
    __builtin_amdgcn_raw_buffer_store_b128(
        u4_t{__float_as_uint(sums[4 * 64 + tid_e]), __float_as_uint(l), kTagValid, kTagValid}, rml,
        recs[tid_e] * kRecMlBytes, 0, kCoherent);
  }
}

}  // namespace

template <bool KT, bool VT, bool SW = false>
static void launch_mq(const AttnArgs& a, int n_wg, hipStream_t stream) {
  if (a.qpw * (a.num_q / a.num_kv) > 32)
    hipLaunchKernelGGL((mq_attn_kernel<KT, VT, 4, false, SW>), dim3(n_wg), dim3(kThreads), 0, stream, QKV_ATTN_LEAD_ARGS(a), a);
  else
    hipLaunchKernelGGL((mq_attn_kernel<KT, VT, 2, false, SW>), dim3(n_wg), dim3(kThreads), 0, stream, QKV_ATTN_LEAD_ARGS(a), a);
}
static bool has_sink_or_window(const AttnArgs& a) { return a.sink_tok > 0 || a.window_tok > 0; }

hipError_t launch_mq_attn(const AttnArgs& a, bool k_tq3, bool v_tq3, uint16_t* out, hipStream_t stream) {
  const int groups = (a.sub_n + a.qpw - 1) / a.qpw * a.n_chunks;
  const int n_wg = (groups + 7) / 8 * 8 * a.num_kv;
  if (k_tq3 && has_sink_or_window(a))
    launch_mq<true, true, true>(a, n_wg, stream);
  else if (k_tq3)
    launch_mq<true, true>(a, n_wg, stream);
  else if (v_tq3)
    launch_mq<false, true>(a, n_wg, stream);
  else
    launch_mq<false, false>(a, n_wg, stream);
  const hipError_t e = hipGetLastError();
  return e != hipSuccess ? e : launch_record_merge(a, v_tq3, out, stream);
}

// The split API's partials (TQ3 caches: at most 32 columns per workgroup).
hipError_t launch_mq_split(const AttnArgs& a, bool tq3, hipStream_t stream) {
  const int groups = (a.sub_n + a.qpw - 1) / a.qpw * a.n_chunks;
  const dim3 grid((groups + 7) / 8 * 8 * a.num_kv), block(kThreads);
  const bool wide = a.qpw * (a.num_q / a.num_kv) > 32;
  if (tq3 && wide) return hipErrorInvalidValue;
  if (tq3 && has_sink_or_window(a))
    hipLaunchKernelGGL((mq_attn_kernel<true, true, 2, true, true>), grid, block, 0, stream, QKV_ATTN_LEAD_ARGS(a), a);
  else if (tq3)
    hipLaunchKernelGGL((mq_attn_kernel<true, true, 2, true>), grid, block, 0, stream, QKV_ATTN_LEAD_ARGS(a), a);
  else if (wide)
    hipLaunchKernelGGL((mq_attn_kernel<false, false, 4, true>), grid, block, 0, stream, QKV_ATTN_LEAD_ARGS(a), a);
  else
    hipLaunchKernelGGL((mq_attn_kernel<false, false, 2, true>), grid, block, 0, stream, QKV_ATTN_LEAD_ARGS(a), a);
  return hipGetLastError();
}

}  // namespace qkv
