// attn_tq3.hip -- split-K flash decode over the packed TQ3 cache (gfx950).
//
// Reference semantics: flash_attn_chunk_fused_split_tq3 (attention.cuh:1905-2177)
// and flash_attn_split_merge (attention.cuh:1837-1891).
//
// Design (not the reference's): attention runs in the rotated domain.  With
// R = rs*H*D (orthogonal, D = signs, H = Sylvester Hadamard), a stored block
// decodes to k = norm * R^T c[idx], so q.k = norm * (R q).c[idx]: the query is
// rotated once per workgroup and keys are never inverse-transformed.  Values
// accumulate sum_t p_t norm_t c[idx_t] in rotated coordinates and each output
// row is rotated back once.
//
// Workgroup: 8 waves (two per SIMD) on one kv head and one key chunk; each
// wave takes 64-key tiles.  The first wave of each SIMD issues its first
// tile's loads before the second, so that its tile arrives first and is
// computed while the second one streams.  Per tile:
//   scores  v_mfma_f32_16x16x32_f16, A = key codes of 16 keys x 32 dims, B =
//           rotated query (columns = heads, held in 32 VGPRs for the whole
//           kernel; the fp16 rounding and the remainder of the query either
//           share the 16 columns, or, for calls with more than 8 / GQA
//           queries, fill them with 16 / GQA queries each, the remainders
//           read from LDS into a second product chained onto the first):
//           lane (key, octet o) takes the 12 bytes holding code groups
//           4o..4o+3 of each 128-block and decodes centroid pairs through a
//           per-lane LDS table.  The fast path loads a tile in 16-byte units,
//           four lanes to a block, and passes the keys through LDS (TileRegs);
//           the split forms load each lane's own 12 bytes (TileRows).  One accumulator per 128-block, each
//           scaled by its block norm (which carries the softmax scale).
//   softmax online, per head, base 2.
//   values  v_mfma_f32_16x16x32_f16, A = p*norm (fp16, the lane's own
//           probabilities), B = codes of 32 keys x 16 dims.  The value codes
//           are staged in LDS, a dword per dim group and key; lane (n, o) gathers dim group n of both blocks for 8 keys
//           and interleaves the codes of key pairs (bit select), so that each
//           table entry read is a B dword (two keys, one dim); the table
//           reads run two steps ahead.
// Merging: the 8 waves merge in LDS and each merged piece goes straight to
// its record {m, l, tags} + o[256] (rotated); the tags are set once the
// workgroup's data stores are complete.  The last workgroups of the grid are
// designated mergers, one per (q head, query, 128-block) unit: each polls its
// unit's tags (bounded), clears them, reads the rows in one round of 16-byte
// loads, merges, rotates back and stores fp16 (attn_fastmerge.h); calls with
// many units leave that to a second launch (merges_apart).  Paged (ragged) launches split each kv head's record shares over the slots in
// proportion to their key counts.  Split API: one workgroup per reference
// split, written in the reference partial layout.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "qkv_device.h"
#include "attn_common.h"
#include "attn_fastmerge.h"
#include "attn_tq3_lut.h"
#include "qkv_launch.h"
#include "tq3_encode.h"

namespace qkv {

typedef uint32_t u32_a1 __attribute__((aligned(1)));

constexpr int kTile = 64;
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kHD = 256;

// Phase stamps of the fast path (a diagnostic build, compiled with
// -DQKV_PHASE_TRACE; the product build has none of this).  Every wave keeps
// s_memrealtime values (100 MHz, one clock for the whole GPU) at the phase
// boundaries below in registers and stores them once, at the end of the
// kernel, to qkv_phase_stamps[workgroup][wave][16]; slot 15 holds the XCD
// the workgroup ran on.  Workgroups past kTraceMaxWgs are not recorded.
enum TracePhase {
  kPhEntry = 0,      // kernel entry
  kPhQuery = 1,      // the query has arrived
  kPhSetup = 2,      // table and rotated query ready (setup barrier passed)
  kPhScores = 3,     // the wave's first tile: scores done
  kPhSoftmax = 4,    // the wave's first tile: staging and softmax done
  kPhTiles = 5,      // every tile of the wave done
  kPhMerged = 6,     // in-workgroup merge done (records stored)
  kPhPublished = 7,  // tags stored
  kPhPolled = 8,     // mergers: every record of the unit seen
  kPhEnd = 9,        // the workgroup is done (mergers: output stored)
  kPhMergeBar = 10,  // in-workgroup merge: every wave's rows are in LDS (barrier passed)
  kPhRowsIn = 11,    // mergers: the unit's record rows have arrived
  kPhFolded = 12,    // mergers: the waves' partials are folded (before normalise/rotate/store)
  kPhSetupWork = 13, // the wave's setup work done (before the setup barrier)
  kPhTileBar = 14,   // every wave's tiles done (the barrier before the in-workgroup merge)
  kPhXcd = 15
};
#ifdef QKV_PHASE_TRACE
constexpr int kTraceMaxWgs = 4096;
__device__ uint64_t qkv_phase_stamps[kTraceMaxWgs * kWaves * 16];
#define QKV_STAMP(k) (trace_st[k] = __builtin_amdgcn_s_memrealtime())
#else
#define QKV_STAMP(k) ((void)0)
#endif

// Per-wave staging of one 64-key tile, in dwords; every row holds 64 keys
// (key = position in the tile) at a pitch of 68, so 16 lanes reading 16-byte
// pieces of 16 different rows hit 16 disjoint bank quads.
constexpr int kKeyPitch = 68;
constexpr int kStCodes = 0;                  // [block j][group g] rows: value code group g (3 bytes, dword-expanded)
constexpr int kStVn = 32 * kKeyPitch;        // [block j] rows: value block norms
constexpr int kStKn = 34 * kKeyPitch;        // [block j] rows: key block norms
constexpr int kStCorr = 36 * kKeyPitch;      // 16 floats: per-head rescale of the accumulators
constexpr int kStageBytes = (36 * kKeyPitch + 16) * 4;   // 9856

// LDS layout (bytes).  The merge area aliases the staging areas (used after the loop).
constexpr int kLdsStage = kLdsLut + kLdsLutBytes;            // per wave, kStageBytes
constexpr int kLdsQ = kLdsStage + kWaves * kStageBytes;      // rotated query, 512 x 16 B (q_unit)
constexpr int kLdsTileEnd = kLdsQ + 16 * 256 * 2;
// After the tile loop the table and the staging areas are free: the merge
// area starts at 0.
constexpr int kLdsMergeO = 0;                                // [waves][16 rows][256] f32
constexpr int kLdsMergeML = kLdsMergeO + kWaves * 16 * kHD * 4;
constexpr int kLdsMergeEnd = kLdsMergeML + 512 * 4;
// one-query step with its token appended in the launch: the new key's
// encoded K and V blocks (4 x 13 dwords)
constexpr int kLdsNewRow = kLdsTileEnd;
constexpr int kLdsTotal = kLdsNewRow + 256;
static_assert(kLdsMergeEnd <= kLdsQ, "merge area must not reach the query scratch");
static_assert(kTracePolledByte >= kWaves * 128 * 4 && kTracePolledByte + 24 <= kLdsMergeML - kLdsMergeO,
              "the merger's trace slot lies in the merge area, past the reduction area");

// merge-area float offsets (ML): m[w][16], l[w][16], M[16], L[16]
constexpr int kMlW0 = 0, kMlLw0 = 16 * kWaves, kMlM = 32 * kWaves, kMlL = 32 * kWaves + 16;
static_assert(kMlL + 16 <= 512, "merge scalars must fit the ML area");

// 16-byte unit of the rotated-query scratch holding elements 8(4o+u)..+7 of
// 128-block j of column c, s = 4j + u.  The column is swizzled with (u, o) so
// that the 16 lanes of one WHT writing (fixed c, j) and the 16 lanes of one
// MFMA row reading (fixed s, o) each touch 16 distinct 16-byte bank groups.
__device__ __forceinline__ int q_unit(int c, int s, int o) {
  return (s * 4 + o) * 16 + (c ^ (4 * (s & 3) + o));
}

// Score MFMAs for one 16-key group: 4 slices per block, one accumulator per
// block.  Slice U+1's table reads are issued before slice U's MFMAs.
// CHAIN: the query remainders (lo) have MFMA columns of their own in a second
// product chained onto the same accumulator; slice s of this lane's lo
// operand is at LDS byte qlo + 1024 s.
template <int U, bool CHAIN>
__device__ __forceinline__ void score_group(const uint8_t* lds, uint32_t (&ac)[4], const uint32_t (&k0)[3],
                                            const uint32_t (&k1)[3], const h8_t (&qa)[8],
                                            uint32_t qlo,
                                            const h8_t& b0, const h8_t& b1, f4_t& a0, f4_t& a1) {
  if constexpr (U < 4) {
    h8_t n0, n1, l0, l1;
    if constexpr (CHAIN) {
      l0 = *reinterpret_cast<const h8_t*>(lds + qlo + 1024 * U);
      l1 = *reinterpret_cast<const h8_t*>(lds + qlo + 1024 * (4 + U));
    }
    if constexpr (U < 3) {
      n0 = group_operand<U + 1>(lds, ac, k0);
      n1 = group_operand<U + 1>(lds, ac, k1);
    }
    a0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(b0, qa[U], a0, 0, 0, 0);
    a1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(b1, qa[4 + U], a1, 0, 0, 0);
    if constexpr (CHAIN) {
      a0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(b0, l0, a0, 0, 0, 0);
      a1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(b1, l1, a1, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (U < 3) score_group<U + 1, CHAIN>(lds, ac, k0, k1, qa, qlo, n0, n1, a0, a1);
  }
}

// One value pass: a (32-key chunk c2, 128-block j) pair.  MFMA k index i of
// the pass is key 32*c2 + 4*row + i (i < 4) or 32*c2 + 16 + 4*row + i - 4.
// x: the code group `col` (8 dims, 24 bits) of key i as loaded; from the
// pass's first table reads on (interleave_pairs), the codes of keys 2k and
// 2k + 1 interleaved per dim, so that one 6-bit field is a table index whose
// entry is already the B dword (key 2k in the low half, key 2k + 1 in the
// high half): x[k] holds dims 0, 2, 4, 6 (field 6d: codes of dim 2d),
// x[4 + k] dims 1, 3, 5, 7 (field 6d + 3: codes of dim 2d + 1).
// a: A operand (p * value norm of those keys, head `col`).
struct ValuePass {
  uint32_t x[8];
  h8_t a;
};

// Codes and A operand of pass c = 2*c2 + j from the tile's staging area.
__device__ __forceinline__ void value_pass_load(const float* st, const uint32_t* stu, int c, int row,
                                                int col, const float (&s)[4][4], ValuePass& vp) {
  const int c2 = c >> 1, j = c & 1;
  const f4_t va = *reinterpret_cast<const f4_t*>(st + kStVn + j * kKeyPitch + 32 * c2 + 4 * row);
  const f4_t vb = *reinterpret_cast<const f4_t*>(st + kStVn + j * kKeyPitch + 32 * c2 + 16 + 4 * row);
  const u4_t xa = *reinterpret_cast<const u4_t*>(stu + kStCodes + (16 * j + col) * kKeyPitch + 32 * c2 + 4 * row);
  const u4_t xb =
      *reinterpret_cast<const u4_t*>(stu + kStCodes + (16 * j + col) * kKeyPitch + 32 * c2 + 16 + 4 * row);
#pragma unroll
  for (int r = 0; r < 4; r++) {
    vp.a[r] = (_Float16)(s[2 * c2][r] * va[r]);
    vp.a[4 + r] = (_Float16)(s[2 * c2 + 1][r] * vb[r]);
    vp.x[r] = xa[r];
    vp.x[4 + r] = xb[r];
  }
}

// Table reads of dims 2PP (cp[0..3]) and 2PP+1 (cp[4..7]) of the 4 key pairs:
// each entry is a B dword (two keys, one dim).
template <int PP>
__device__ __forceinline__ void value_pairs(const uint8_t* lds, uint32_t (&ac)[4], uint32_t (&x)[8],
                                            uint32_t (&cp)[8]) {
  if constexpr (PP == 0) interleave_pairs(x);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    ac[k] = sdwa_index<6 * PP>(ac[k], x[k]);
    cp[k] = lut_read(lds, ac[k]);
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
    ac[k] = sdwa_index<6 * PP + 3>(ac[k], x[4 + k]);
    cp[4 + k] = lut_read(lds, ac[k]);
  }
}

// Step K of the value phase (pass c = K / 4, centroid pair PP = K % 4): tiles
// 8j + 2PP (low dim) and 8j + 2PP + 1 (high dim).  Software-pipelined two
// steps deep: the table reads of step K+2 are issued before the perms and
// MFMAs of step K (cp: step K's pairs, cq: step K+1's), and the codes and A
// operand of pass c+1 are read during the first step of pass c.
// FIRST: the workgroup's first tile, whose passes 0 and 1 write every
// accumulator tile for the first time (zero C operand).
template <int K, bool FIRST>
__device__ __forceinline__ void value_steps(const uint8_t* lds, uint32_t (&ac)[4], ValuePass (&vp)[2],
                                            const uint32_t (&cp)[8], const uint32_t (&cq)[8],
                                            f4_t (&acc)[16], const float* st, const uint32_t* stu, int row,
                                            int col, const float (&s)[4][4]) {
  if constexpr (K < 16) {
    constexpr int c = K >> 2, PP = K & 3;
    if constexpr (PP == 0 && c < 3) value_pass_load(st, stu, c + 1, row, col, s, vp[(c + 1) & 1]);
    uint32_t cn[8];
    if constexpr (K + 2 < 16) value_pairs<(K + 2) & 3>(lds, ac, vp[((K + 2) >> 2) & 1].x, cn);
#pragma unroll
    for (int e = 0; e < 2; e++) {
      u4_t bv;
#pragma unroll
      for (int k2 = 0; k2 < 4; k2++) bv[k2] = cp[4 * e + k2];
      constexpr int t0 = 8 * (c & 1) + 2 * PP;
      const f4_t cin = (FIRST && c < 2) ? f4_t{0.f, 0.f, 0.f, 0.f} : acc[t0 + e];
      acc[t0 + e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vp[c & 1].a, __builtin_bit_cast(h8_t, bv),
                                                           cin, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (K < 15) value_steps<K + 1, FIRST>(lds, ac, vp, cq, cn, acc, st, stu, row, col, s);
  }
}

// Registers of one 64-key tile, as loaded: unit i of the lane is piece lane & 3 of
// block lane >> 5 of the row of key 8 i + ((lane >> 2) & 7) -- the 16 bytes from byte
// 12 (lane & 3) of the 52-byte block on, i.e. the code groups 4 (lane & 3) .. + 3 in
// dwords 1..3 and, in piece 0, the block's norm in dword 0.  Four lanes read one
// block's 52 bytes: the cache looks up a third of the lines it does with a row or a
// strided piece per lane (1.7 million lookups of a cycle each and CU for 18,016 keys in
// 8 splits bound that launch: 27 us).  Buffer loads: offsets are 32-bit and reads
// past the cache extent (num_records) return zero, so partial tiles need no
// branches; keys in [hi, extent) are read and masked out of the softmax.
struct TileRegs {
  u4_t k[8], v[8];
};
__device__ __forceinline__ int unit_key8(int lane) { return (lane >> 2) & 7; }

// prow: cache row of the tile's first key (64 consecutive rows, wave-uniform);
// the buffer resources are rebased at that row (64-bit byte offset)
template <int FROM, int TO>   // units FROM .. TO - 1
__device__ __forceinline__ void load_tile_part(const uint32_t* base, uint64_t bytes, int prow, int nkv, int h,
                                               int lane, u4_t (&r)[8]) {
  const uint64_t off0 = (uint64_t)(uint32_t)prow * (uint32_t)nkv * 104u;
  const __amdgpu_buffer_rsrc_t rs = cache_rsrc(base, off0, bytes);
  asm volatile("" : "+v"(lane));   // (the offsets are formed per tile, not held in registers)
  const uint32_t unit = (uint32_t)(unit_key8(lane) * nkv + h) * 104u + 52u * (uint32_t)(lane >> 5) +
                        12u * (uint32_t)(lane & 3);
#pragma unroll
  for (int i = FROM; i < TO; i++)
    r[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, unit + (uint32_t)(i * 8 * nkv) * 104u, 0, 0);
}
template <int FROM = 0, int TO = 8>
__device__ __forceinline__ void load_tile_keys(const AttnArgs& p, int prow, int nkv, int h, int lane, TileRegs& tr) {
  load_tile_part<FROM, TO>(p.k, p.kv_bytes, prow, nkv, h, lane, tr.k);
}
__device__ __forceinline__ void load_tile_values(const AttnArgs& p, int prow, int nkv, int h, int lane, TileRegs& tr) {
  load_tile_part<0, 8>(p.v, p.kv_bytes, prow, nkv, h, lane, tr.v);
}
// keys first: values arrive while the scores are computed
__device__ __forceinline__ void load_tile(const AttnArgs& p, int prow, int nkv, int h, int lane, TileRegs& tr) {
  load_tile_keys(p, prow, nkv, h, lane, tr);
  load_tile_values(p, prow, nkv, h, lane, tr);
}

// The same tile with a lane's own operands: strided 12-byte key pieces and whole value
// rows, which need no pass through the LDS before the scores.  For the split forms
// (MODE >= 1): their few workgroups walk many tiles in a row, where that pass is part
// of every round and the cache lookups are not the bound (one query in 8 splits,
// 64,533 keys: 81.6 us, 89.7 in units; 18,016: 29.4, 30.7).
struct TileRows {
  u4_t vr[6];            // value row of key ts+lane (dwords 0..23)
  u2_t vr6;              // dwords 24..25
  uint32_t kq[4][2][3];  // key code groups 4*row..4*row+3, group g, block j
  float kn[4][2];        // key block norms, group g, block j
};
template <int FROM = 0, int TO = 8>
__device__ __forceinline__ void load_tile_keys(const AttnArgs& p, int prow, int nkv, int h, int lane, TileRows& tr) {
  if constexpr (FROM < TO) {
    const int row = lane >> 4, col = lane & 15;
    const __amdgpu_buffer_rsrc_t rk = cache_rsrc(p.k, (uint64_t)(uint32_t)prow * (uint32_t)nkv * 104u, p.kv_bytes);
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const uint32_t krow = (uint32_t)((16 * g + col) * nkv + h) * 104u;
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const u3_t c = __builtin_amdgcn_raw_buffer_load_b96(rk, krow + 52 * j + 4 + 12 * row, 0, 0);
        tr.kq[g][j][0] = c[0];
        tr.kq[g][j][1] = c[1];
        tr.kq[g][j][2] = c[2];
        tr.kn[g][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rk, krow + 52 * j, 0, 0));
      }
    }
  }
}
__device__ __forceinline__ void load_tile_values(const AttnArgs& p, int prow, int nkv, int h, int lane, TileRows& tr) {
  const __amdgpu_buffer_rsrc_t rv = cache_rsrc(p.v, (uint64_t)(uint32_t)prow * (uint32_t)nkv * 104u, p.kv_bytes);
  const uint32_t vrow = (uint32_t)(lane * nkv + h) * 104u;
#pragma unroll
  for (int i = 0; i < 6; i++) tr.vr[i] = __builtin_amdgcn_raw_buffer_load_b128(rv, vrow + 16 * i, 0, 0);
  tr.vr6 = __builtin_amdgcn_raw_buffer_load_b64(rv, vrow + 96, 0, 0);
}
__device__ __forceinline__ void load_tile(const AttnArgs& p, int prow, int nkv, int h, int lane, TileRows& tr) {
  load_tile_keys(p, prow, nkv, h, lane, tr);
  load_tile_values(p, prow, nkv, h, lane, tr);
}
// Staging of a tile in rows: key norms, value codes and norms.
__device__ __forceinline__ void stage_rows(float* st, int lane, const TileRows& tr, float scale2) {
  const int row = lane >> 4, col = lane & 15;
  uint32_t* stu = reinterpret_cast<uint32_t*>(st);
  if (row == 0) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
      st[kStKn + 16 * g + col] = tr.kn[g][0] * scale2;
      st[kStKn + kKeyPitch + 16 * g + col] = tr.kn[g][1] * scale2;
    }
  }
  uint32_t d[27];
#pragma unroll
  for (int i = 0; i < 6; i++)
#pragma unroll
    for (int e = 0; e < 4; e++) d[4 * i + e] = tr.vr[i][e];
  d[24] = tr.vr6[0];
  d[25] = tr.vr6[1];
  d[26] = 0u;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    stu[kStVn + j * kKeyPitch + lane] = d[13 * j];
#pragma unroll
    for (int g = 0; g < 16; g++) {
      // code group g of block j: bytes 3g..3g+2 of the codes (dword 13j+1 on)
      const int w = 13 * j + 1 + ((3 * g) >> 2), sh = (3 * g) & 3;
      stu[kStCodes + (16 * j + g) * kKeyPitch + lane] = sh ? __builtin_amdgcn_alignbyte(d[w + 1], d[w], sh) : d[w];
    }
  }
}

// The encoded new key (4 x 13 dwords at nr) written over the registers of
// the tile that holds it, r = its index in the tile (constant register indices).
__device__ __forceinline__ void patch_new_key(TileRegs& tr, const uint32_t* nr, int r, int lane) {
  if (unit_key8(lane) == (r & 7)) {
    const uint32_t* k = nr + 13 * (lane >> 5) + 3 * (lane & 3);
    const u4_t nk = {k[0], k[1], k[2], k[3]}, nv = {k[26], k[27], k[28], k[29]};
#pragma unroll
    for (int i = 0; i < 8; i++) {
      tr.k[i] = i == r >> 3 ? nk : tr.k[i];
      tr.v[i] = i == r >> 3 ? nv : tr.v[i];
    }
  }
}

// A tile's key units pass through the wave's staging area (before its value codes
// take it) to the lanes whose score operands they are: key r's piece c of 16 bytes
// (c = 4 block + piece) at 128 r + 16 (c ^ f(r)), where f(r) = 4 ((r >> 1) & 1) +
// ((r >> 2) & 3) gives both the 16 lanes of a store (4 keys, 4 pieces) and those of a
// read (16 keys, one piece) 16 different bank groups.
__device__ __forceinline__ void stage_keys(uint8_t* st, int lane, const u4_t (&k)[8], float scale2) {
  const int key8 = unit_key8(lane), c = 4 * (lane >> 5) + (lane & 3);
  const int at = 128 * key8 + 16 * (c ^ (4 * ((key8 >> 1) & 1) + (key8 >> 2)));
#pragma unroll
  for (int i = 0; i < 8; i++) *reinterpret_cast<u4_t*>(st + (at ^ (32 * (i & 1))) + 1024 * i) = k[i];
  if ((lane & 3) == 0) {
    // key norms carry the softmax scale and undo the table scale
    float* kn = reinterpret_cast<float*>(st) + kStKn + (lane >> 5) * kKeyPitch + key8;
#pragma unroll
    for (int i = 0; i < 8; i++) kn[8 * i] = __uint_as_float(k[i][0]) * scale2;
  }
}
// Byte of piece `row` of block 0 of key `col` (block 1: ^ 64; key 16 g + col: + 2048 g).
__device__ __forceinline__ int staged_key(int row, int col) {
  return 128 * col + 16 * (row ^ (4 * ((col >> 1) & 1) + (col >> 2)));
}
// Value codes, one dword per 8-dim group and key, and norms.
__device__ __forceinline__ void stage_values(float* st, int lane, const u4_t (&v)[8]) {
  const int key8 = unit_key8(lane), j = lane >> 5, pc = lane & 3;
  uint32_t* d = reinterpret_cast<uint32_t*>(st) + kStCodes + (16 * j + 4 * pc) * kKeyPitch + key8;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    d[8 * i] = v[i][1];
    d[8 * i + kKeyPitch] = __builtin_amdgcn_alignbyte(v[i][2], v[i][1], 3);
    d[8 * i + 2 * kKeyPitch] = __builtin_amdgcn_alignbyte(v[i][3], v[i][2], 2);
    d[8 * i + 3 * kKeyPitch] = v[i][3] >> 8;
  }
  if (pc == 0) {
    float* vn = st + kStVn + j * kKeyPitch + key8;
#pragma unroll
    for (int i = 0; i < 8; i++) vn[8 * i] = __uint_as_float(v[i][0]);
  }
}

// max / sum inside each 16-lane row (all lanes of the row receive the result)
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, dpp_f<0xB1>(v));
  v = fmaxf(v, dpp_f<0x4E>(v));
  v = fmaxf(v, dpp_f<0x124>(v));
  v = fmaxf(v, dpp_f<0x128>(v));
  return v;
}
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_f<0xB1>(v);
  v += dpp_f<0x4E>(v);
  v += dpp_f<0x124>(v);
  v += dpp_f<0x128>(v);
  return v;
}

// Rotate the merged rows back (o = rs*D*H*o_rot per 128-block) and store the
// unnormalised f32 partials of the reference splits split0 .. split0 + n - 1 (m in
// natural-log units): row r of split0 + i is merge row i slot + r, its scalars at
// i rows + r.
__device__ void finish_rows(const uint8_t* lds, const AttnArgs& p, int h, int t, int rows, int split0, int n,
                            int slot) {
  const float* mo = reinterpret_cast<const float*>(lds + kLdsMergeO);
  const float* ml = reinterpret_cast<const float*>(lds + kLdsMergeML);
  const int gqa = p.num_q / p.num_kv;
  const int lane = threadIdx.x & 63;
  n = min(n, p.k_splits - split0);
  for (int w0 = 0; w0 < n * rows * 2; w0 += kThreads / 16) {
    const int wht = w0 + (threadIdx.x >> 4);
    const int part = threadIdx.x & 15;
    const int ri = wht >> 1, blk = wht & 1, i = ri / rows, r = ri - i * rows;
    const bool live = wht < n * rows * 2;
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; e++)   // the centroid table is scaled by kCenScale: undo it here (fp32)
      x[e] = live ? mo[(i * slot + r) * kHD + blk * 128 + part * 8 + e] * kCenScaleInv : 0.f;
    wht8_inreg(x);
    wht_xor_lanes16(x, lane);
    if (!live) continue;
    const float rs = wht_scale();
    const int qh = h * gqa + r % gqa, tq = t + r / gqa;
    const uint32_t sbits = sign_word_sel(part >> 2) >> (8 * (part & 3));  // elements part*8..+7
    const long mlx = ((long)qh * p.sub_n_max + tq) * p.k_splits + split0 + i;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const bool pos = (sbits >> e) & 1u;
      const float v = x[e] * rs;
      p.part_o[mlx * kHD + blk * 128 + part * 8 + e] = pos ? v : -v;
    }
    if (blk == 0 && part == 0) {
      const float M = ml[kMlM + ri];
      p.part_m[mlx] = (M == -INFINITY) ? -INFINITY : M * kLn2;
      p.part_l[mlx] = ml[kMlL + ri];
    }
  }
}

// MODE 0: fast path (final fp16 rows).  MODE 1: reference split partials.
// MODE 2: block-sparse split partials (attention.cuh:2193-2433): one query
// per workgroup (qpw = 1), wg_splits splits of its selected 64-key blocks.
// CHAIN (fast path, several queries): 16 / GQA queries per workgroup, every
// MFMA column a real (query, head); the remainders ride in a chained second
// score product (see score_group).
// APPEND (MODE 0, one query): the step's new token is encoded in the launch
// (qkv_decode_attn_tq3_append), a separate instance so that the plain decode
// compiles without it.
template <int MODE, bool CHAIN = false, bool APPEND = false>
__global__ __launch_bounds__(kThreads, 1) void tq3_attn_kernel(QKV_ATTN_LEAD_PARAMS, AttnArgs pin,
                                                                uint16_t* out) {
  QKV_ATTN_LEAD_APPLY(p, pin);
  const bool paged = (lead_flags & (1u << 8)) != 0, ragged = (lead_flags & (1u << 9)) != 0;
  // static LDS: table and tile offsets fold into the instructions' offset field
  __shared__ __attribute__((aligned(16))) uint8_t lds[kLdsTotal];
#ifdef QKV_PHASE_TRACE
  uint64_t trace_st[15] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#endif
  QKV_STAMP(kPhEntry);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int gqa = __builtin_amdgcn_readfirstlane(p.num_q / p.num_kv);   // scalar register

  // ---- work id (XCD-aware: the num_kv workgroups of one (query group, chunk)
  // share an XCD).  A workgroup serves queries t0 .. t0+nq-1 (nq <= qpw) of
  // one kv head: MFMA column c = qi * gqa + hh is q head h*gqa + hh of query
  // t0 + qi (columns past nq * gqa carry nothing).
  int h, t0, chunk;
  int rec_t0, rec_chunk;      // record coordinates of this workgroup's rows
  int chunk_keys = p.chunk_keys;
  bool has_work;
  {
    const int L = blockIdx.x;
    const int xcd = L & 7, r = L >> 3;
    h = r % p.num_kv;
    const int g = (r / p.num_kv) * 8 + xcd;
    const int groups = (p.sub_n + p.qpw - 1) / p.qpw;
    has_work = g < groups * p.n_chunks;
    if (MODE == 0 && ragged) {
      // ragged slots (one query each): share g of the length-proportional split
      int first, count;
      const int s = has_work ? share_slot(p, g, first, count) : -1;
      has_work = s >= 0;
      t0 = has_work ? s : 0;
      chunk = has_work ? g - first : 0;
      if (has_work) {   // the slot's keys in count chunks of whole 512-key steps
        const int per = (slot_keys(p, s) + count - 1) / count;
        chunk_keys = max(1, (per + kWaves * kTile - 1) / (kWaves * kTile)) * (kWaves * kTile);
      }
      rec_t0 = 0;
      rec_chunk = g;
    } else {
      const int tq = has_work ? g / p.n_chunks : 0;
      chunk = has_work ? g - tq * p.n_chunks : 0;
      t0 = tq * p.qpw;
      rec_t0 = t0;
      rec_chunk = chunk;
    }
  }
  if (MODE >= 1 && !has_work) return;
  const int nq = min(p.qpw, p.sub_n - t0);
  // accumulator rows (columns) that hold heads (uniform: kept in a scalar register)
  const int rows_used = __builtin_amdgcn_readfirstlane(nq * gqa);
  const int row = lane >> 4;        // 16-lane row of the MFMA D layout
  const int col = lane & 15;
  const int t_col = t0 + min(col / gqa, nq - 1);   // this lane's query (clamped for dead columns)
  // ---- the query load goes out first: its address depends only on the
  // preloaded arguments
  // 32 WHTs of 128 (16 columns x 2 blocks), 16 lanes each
  const int q_wht = threadIdx.x >> 4;
  const int q_part = threadIdx.x & 15;
  const int q_col = q_wht >> 1, q_blk = q_wht & 1;   // column, 128-block
  u4_t q_raw;
  {
    // unconditional (rows past the buffer's extent read as zero): a load
    // under a branch makes the compiler wait for every load at the join
    const uint32_t q_extent = (uint32_t)(p.sub_n * p.num_q * kHD * 2);
    const __amdgpu_buffer_rsrc_t rq =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.q), 0, q_extent, kBufferRsrcWord3);
    const uint32_t qoff =
        q_col < rows_used ? (uint32_t)((((t0 + q_col / gqa) * p.num_q + h * gqa + q_col % gqa) * kHD +
                                        q_blk * 128 + q_part * 8) * 2)
                          : q_extent;
    q_raw = __builtin_amdgcn_raw_buffer_load_b128(rq, qoff, 0, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
  // key counts: the lane's own query, and the first / last query of the group
  // (a paged group has one query)
  const int active_end = ragged ? min(max(p.ctx_lens[t_col], 0), p.ctx_max)
                                    : p.start_pos + t_col + 1;
  const int active_first = ragged ? active_end : p.start_pos + t0 + 1;
  const int active_last = ragged ? active_end : p.start_pos + t0 + nq;
  int lo = 0, hi = 0, hi_col = 0, hi_first = 0;
  if (MODE == 0) {
    if (has_work) {
      lo = chunk * chunk_keys;
      // the last chunk of a contiguous launch runs to the end of the keys: the
      // host may have joined a remainder of at most one tile to it
      const int c_end = (!ragged && chunk == p.n_chunks - 1) ? active_last : lo + chunk_keys;
      hi = min(c_end, active_last);
      hi_col = min(c_end, active_end);
      hi_first = min(c_end, active_first);
    }
  } else if (MODE == 2) {
    // the selected blocks bound the keys; the query's causal end masks them
    lo = 0;
    hi = active_end;
    hi_col = active_end;
    hi_first = active_end;
  } else {
    // reference split range (attention.cuh:1944-1951)
    const int total_tiles = (p.active_end_max + 31) / 32;
    const int tps = (total_tiles + p.k_splits - 1) / p.k_splits;
    lo = chunk * tps * 32;
    hi = min((chunk + 1) * tps * 32, active_last);
    hi_col = min((chunk + 1) * tps * 32, active_end);
    hi_first = min((chunk + 1) * tps * 32, active_first);
  }
  lo = __builtin_amdgcn_readfirstlane(lo);
  hi = __builtin_amdgcn_readfirstlane(hi);
  hi_first = __builtin_amdgcn_readfirstlane(hi_first);
  // appended token (one-query launches of qkv_decode_attn_tq3_append): the
  // wave whose tiles hold key start_pos (tile k of wave w starts at lo + 64w
  // + k * 512), and its input, lane l: 16-byte piece l & 15 of block l >> 4
  // (K block 0, K block 1, V block 0, V block 1 of kv head h)
  int fa_wave = -1;
  uint4 fa_raw = make_uint4(0u, 0u, 0u, 0u);
  if constexpr (APPEND) {
    if (p.k_new != nullptr && has_work && lo <= p.start_pos && p.start_pos < hi)
      fa_wave = ((p.start_pos - lo) >> 6) & (kWaves - 1);
    fa_wave = __builtin_amdgcn_readfirstlane(fa_wave);
    if (fa_wave == wave) {
      const int blk = lane >> 4;
      fa_raw = *reinterpret_cast<const uint4*>((blk < 2 ? p.k_new : p.v_new) + h * kHD + (blk & 1) * 128 +
                                               8 * (lane & 15));
    }
  }
  // A dead column has a zero query: its scores are 0 and its accumulator rows
  // are never stored, so it needs no mask of its own.

  // ---- setup: centroid-pair table, rotated query --------------------------
  // The query is loaded and rotated before any tile load is issued: a query
  // load issued after the tile loads of the whole chip would wait behind
  // them in the memory queues.
  // paged caches: the block-table entries of this wave's first 64 tiles (lane
  // k: tile k, key lo + wave*64 + k*kStep), loaded now so that no tile load
  // waits for a table read (rows past the table's extent read as 0)
  constexpr int kStep = kWaves * kTile;
  // block-sparse: lane k holds entry k of this split's block list; the list
  // ends at its first -1 (n_sel entries).  A workgroup serves wg_splits
  // consecutive splits of its query, kWaves / wg_splits (spw) waves each: wave
  // sw of a split takes entries sw, sw + spw, ...  (a split past the last has
  // an empty list)
  const int spw = MODE == 2 ? kWaves / p.wg_splits : kWaves, sw = wave % spw;
  int sel = -1, n_sel = 0;
  if constexpr (MODE == 2) {
    const int per = (p.top_k + p.k_splits - 1) / p.k_splits;
    const int tk_lo = (chunk * p.wg_splits + wave / spw) * per, tk_n = max(0, min(per, p.top_k - tk_lo));
    const __amdgpu_buffer_rsrc_t rbi = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int32_t*>(p.block_index), 0, (uint32_t)(p.num_kv * p.sub_n_max * p.top_k * 4),
        kBufferRsrcWord3);
    // unconditional load (an out-of-range offset reads 0), masked after
    const uint32_t off = lane < tk_n
        ? (uint32_t)((((h * p.sub_n_max + t0) * p.top_k) + tk_lo + lane) * 4) : 0xffffffffu;
    const int ld = (int)__builtin_amdgcn_raw_buffer_load_b32(rbi, off, 0, 0);
    const int e = lane < tk_n ? ld : -1;
    const uint64_t ends = __builtin_amdgcn_ballot_w64(e < 0);
    n_sel = ends ? (int)__builtin_ctzll(ends) : 64;
    sel = e;
  }
  const int ts0 = MODE == 2 ? (sw < n_sel ? __builtin_amdgcn_readlane(sel, sw) * kTile : 0)
                            : lo + wave * kTile;
  const __amdgpu_buffer_rsrc_t rbt = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int32_t*>(p.block_tables), 0,
      p.block_tables ? (uint32_t)(p.sub_n * p.bt_stride * 4) : 0u, kBufferRsrcWord3);
  auto bt_batch = [&](int k0) -> int {   // entries of tiles k0 .. k0+63 (one per lane)
    const int ts = ts0 + (k0 + lane) * kStep;
    int bt = __builtin_amdgcn_readfirstlane(max(p.block_tokens, 1));
    asm volatile("" : "+s"(bt));   // (divisor re-read per batch, not held through the loop)
    const uint32_t off = ts < hi ? (uint32_t)((t0 * p.bt_stride + ts / bt) * 4) : 0xffffffffu;
    return (int)__builtin_amdgcn_raw_buffer_load_b32(rbt, off, 0, 0);
  };
  int bt_entry = paged ? bt_batch(0) : 0, bt_k0 = 0;
  // cache row of this wave's tile starting at key ts: ts itself for a
  // contiguous cache; through the query's block table for a paged one (block
  // sizes are multiples of 64, so a 64-key tile never straddles two blocks);
  // rows outside the cache extent read as zero (buffer range checks)
  auto wave_tile_row = [&](int ts) -> int {
    if (!paged) return ts;
    if (ts >= hi) return 0;
    const int k = (ts - ts0) / kStep;
    if (k - bt_k0 >= 64) {
      bt_k0 = k & ~63;
      bt_entry = bt_batch(bt_k0);
    }
    const int e = __builtin_amdgcn_readlane(bt_entry, k - bt_k0);
    // (the divisor re-read per tile instead of held through the loop)
    int bt = __builtin_amdgcn_readfirstlane(p.block_tokens);
    asm volatile("" : "+s"(bt));
    const int b = ts / bt;
    return e * bt + (ts - b * bt);
  };
  // waves 0..3 issue their first tile's loads as soon as the query has
  // arrived (so it does not queue behind them), ahead of the table build
  // and the rotation; waves 4..7 issue theirs after the setup barrier.
  __builtin_amdgcn_s_waitcnt(0);
  QKV_STAMP(kPhQuery);
  constexpr bool kUnits = MODE == 0;   // tiles in units, or in rows (TileRows)
  std::conditional_t<kUnits, TileRegs, TileRows> tr;
  if (wave < 4) load_tile(p, wave_tile_row(ts0), p.num_kv, h, lane, tr);
  // centroid-pair table: entry e = (centroid[e & 7], centroid[(e >> 3) & 7])
  // as fp16, from immediates (wave-uniform values); wave w writes every lane's
  // copy of entries 32w .. 32w+31
  static_assert(kWaves == 8, "8 waves x 32 entries");
  const uint32_t lane4 = 4u * (uint32_t)lane;
  {
    const uint32_t w = (uint32_t)wave;
#pragma unroll
    for (int hk = 0; hk < 4; hk++) {
      const uint32_t hi = centroid_scaled_h((4u * w + hk) & 7u) << 16;
#pragma unroll
      for (int k = 0; k < 8; k++)
        *reinterpret_cast<uint32_t*>(lds + kLdsLut + (w * 32 + hk * 8 + k) * 256 + lane4) =
            centroid_scaled_h(k) | hi;
    }
  }
  uint32_t ac[4] = {lane4, lane4, lane4, lane4};   // table address chains
  uint32_t q_lo[4] = {0u, 0u, 0u, 0u};              // CHAIN: this thread's query remainders
  {
    // rotated query: fp16 in LDS scratch (q_unit), so that each lane's A
    // operand slice is one 16-byte read
    // Column c < 8 holds the fp16 rounding of the rotated query (hi) and
    // column c + 8 the fp16 rounding of its remainder (lo): the score MFMA
    // computes both against the same decoded keys and the two halves are added
    // in fp32, so the rotated query is carried to ~2^-22 (real columns <= 8).
    uint16_t* qs = reinterpret_cast<uint16_t*>(lds + kLdsQ);
    const int o = q_part >> 2, u = q_part & 3;   // elements part*8..+7 = code group 4*o + u
    if (CHAIN) {
      // every column is a (query, head) of its own; the remainders stay in
      // registers until the rounded query has been read (then they replace it)
      uint32_t pk[4] = {0u, 0u, 0u, 0u};
      if (q_col < rows_used) {
        float x[8];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          x[2 * i] = h2f(q_raw[i] & 0xffffu);
          x[2 * i + 1] = h2f(q_raw[i] >> 16);
        }
        const uint32_t sbits = sign_word_sel(q_part >> 2) >> (8 * (q_part & 3));
#pragma unroll
        for (int i = 0; i < 8; i++) {
          const bool pos = (sbits >> i) & 1u;
          x[i] = pos ? x[i] : -x[i];
        }
        wht8_inreg(x);
        wht_xor_lanes16(x, lane);
        const float rs = wht_scale();
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float a = x[2 * i] * rs, b = x[2 * i + 1] * rs;
          const uint32_t ha = f2h(a), hb = f2h(b);
          pk[i] = ha | (hb << 16);
          q_lo[i] = f2h(a - h2f(ha)) | (f2h(b - h2f(hb)) << 16);
        }
      }
      *reinterpret_cast<uint4*>(qs + q_unit(q_col, 4 * q_blk + u, o) * 8) =
          make_uint4(pk[0], pk[1], pk[2], pk[3]);
    } else if (q_col >= 8) {
      // columns 8..15 are written by the waves of columns 0..7
    } else if (2 * wave >= rows_used) {
      // a wave whose two columns are both dead writes zeros (hi and lo)
      *reinterpret_cast<uint4*>(qs + q_unit(q_col, 4 * q_blk + u, o) * 8) = make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(qs + q_unit(q_col + 8, 4 * q_blk + u, o) * 8) = make_uint4(0, 0, 0, 0);
    } else {
      float x[8];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        x[2 * i] = h2f(q_raw[i] & 0xffffu);
        x[2 * i + 1] = h2f(q_raw[i] >> 16);
      }
      const uint32_t sbits = sign_word_sel(q_part >> 2) >> (8 * (q_part & 3));   // elements part*8..+7
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const bool pos = (sbits >> i) & 1u;
        x[i] = pos ? x[i] : -x[i];
      }
      wht8_inreg(x);
      wht_xor_lanes16(x, lane);
      const float rs = wht_scale();
      uint32_t pk[4], pl[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float a = x[2 * i] * rs, b = x[2 * i + 1] * rs;
        const uint32_t ha = f2h(a), hb = f2h(b);
        pk[i] = ha | (hb << 16);
        pl[i] = f2h(a - h2f(ha)) | (f2h(b - h2f(hb)) << 16);
      }
      *reinterpret_cast<uint4*>(qs + q_unit(q_col, 4 * q_blk + u, o) * 8) =
          make_uint4(pk[0], pk[1], pk[2], pk[3]);
      *reinterpret_cast<uint4*>(qs + q_unit(q_col + 8, 4 * q_blk + u, o) * 8) =
          make_uint4(pl[0], pl[1], pl[2], pl[3]);
    }
  }
  if constexpr (APPEND) {
    // the step's new token appended in this launch (qkv_decode_attn_tq3_append
    // with one query): the wave whose tile holds key start_pos encodes its
    // K and V blocks (one 16-lane row each, tq3_encode_row16), stores them
    // to the caches and keeps them in LDS for its tile registers
    if (fa_wave == wave) {
      const uint32_t word = tq3_encode_row16(fa_raw, lane);
      const int blk = lane >> 4, t = lane & 15;
      if (t <= 12) {
        const int w = t == 12 ? 0 : 1 + t;
        reinterpret_cast<uint32_t*>(lds + kLdsNewRow)[blk * 13 + w] = word;
        uint32_t* dst = reinterpret_cast<uint32_t*>(blk < 2 ? p.k_w : p.v_w) +
                        ((long)p.start_pos * p.num_kv + h) * 26 + (blk & 1) * 13 + w;
        *dst = word;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
  QKV_STAMP(kPhSetupWork);
  __syncthreads();
  QKV_STAMP(kPhSetup);
  // (built after the setup: its tree word is a load the first loads must not wait for)
  const KeyRule rule(p.start_pos, t_col, p.sink_tok, p.window_tok, p.tree_mask);
  // ---- first tile: the first wave of each SIMD (waves 0..3) issues its loads
  // before the second (waves 4..7), so that across the chip the first waves'
  // tiles arrive in the first half of the stream and are computed while the
  // second waves' tiles are still in flight.
  if (wave >= 4) load_tile(p, wave_tile_row(ts0), p.num_kv, h, lane, tr);
  // qa[s], slice s = 4j+u: column `col`, element i = dim 128j + 8(4*row+u) + i
  h8_t qa[8];
  {
    const uint16_t* qs = reinterpret_cast<const uint16_t*>(lds + kLdsQ);
#pragma unroll
    for (int s = 0; s < 8; s++)   // dead columns were written as zeros
      qa[s] = *reinterpret_cast<const h8_t*>(qs + q_unit(col, s, row) * 8);
  }
  // CHAIN: the remainders replace the rounded query in the scratch, unswizzled
  // (written once): 16-byte unit (s * 4 + o) * 16 + c holds elements
  // 8(4o+u)..+7 of 128-block j of column c, s = 4j + u
  const uint32_t qlo = (uint32_t)(kLdsQ + row * 256 + col * 16);
  if constexpr (CHAIN) {
    __syncthreads();
    {
      const int o = q_part >> 2, u = q_part & 3;
      *reinterpret_cast<uint4*>(lds + kLdsQ + (((4 * q_blk + u) * 4 + o) * 16 + q_col) * 16) =
          make_uint4(q_lo[0], q_lo[1], q_lo[2], q_lo[3]);
    }
    __syncthreads();
  }

  const float scale2 = p.scale_log2 * kCenScaleInv;
  float m2 = -INFINITY;   // running max of head `col` (base-2 units)
  float lsum = 0.0f;      // this lane's part of the running sum of head `col`
  f4_t acc[16];

  float* st = reinterpret_cast<float*>(lds + kLdsStage + wave * kStageBytes);
  const uint32_t* stu = reinterpret_cast<const uint32_t*>(st);

  // Key units of the next tile that are loaded ahead, during the softmax and the
  // values: all (131,072 keys: 31.6 -> 31.0 us, 65,000: 20.6 -> 20.1), or the half
  // that the chained form has registers for (all: 35 spills, 35.7 -> 41.7 us).
  constexpr int kAhead = CHAIN ? 4 : 8;
  int next_row = 0;   // cache row of the wave's next tile, whose keys are on their way
  // One 64-key tile.  The wave's first tile is a separate instance: its loads
  // were issued with the setup, and its accumulators start at zero.
  // next: first key of the wave's next tile, < 0 if this is its last.
  auto tile_body = [&](auto first_tag, int ts, int next) {
    constexpr bool first = decltype(first_tag)::value;
    // (opaque lane index: the staging addresses are formed here, not held in
    // registers through the tile)
    int lane_o = lane;
    asm volatile("" : "+v"(lane_o));
    if constexpr (kUnits) {
      stage_keys(reinterpret_cast<uint8_t*>(st), lane_o, tr.k, scale2);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    // ---------------- scores: D rows = keys 16g + 4*row + r, D col = head `col` ----------------
    f4_t sa[4][2];
    if constexpr (kUnits) {
      const uint8_t* ks = reinterpret_cast<const uint8_t*>(st) + staged_key(lane_o >> 4, lane_o & 15);
      const uint8_t* ks1 = reinterpret_cast<const uint8_t*>(st) + (staged_key(lane_o >> 4, lane_o & 15) ^ 64);
      u4_t n0 = *reinterpret_cast<const u4_t*>(ks), n1 = *reinterpret_cast<const u4_t*>(ks1);
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const uint32_t k0[3] = {n0[1], n0[2], n0[3]}, k1[3] = {n1[1], n1[2], n1[3]};
        if (g < 3) {   // the next group's codes ahead of this group's products
          n0 = *reinterpret_cast<const u4_t*>(ks + 2048 * (g + 1));
          n1 = *reinterpret_cast<const u4_t*>(ks1 + 2048 * (g + 1));
        }
        sa[g][0] = f4_t{0.f, 0.f, 0.f, 0.f};
        sa[g][1] = f4_t{0.f, 0.f, 0.f, 0.f};
        score_group<0, CHAIN>(lds, ac, k0, k1, qa, qlo, group_operand<0>(lds, ac, k0), group_operand<0>(lds, ac, k1),
                              sa[g][0], sa[g][1]);
      }
    } else {
#pragma unroll
      for (int g = 0; g < 4; g++) {
        sa[g][0] = f4_t{0.f, 0.f, 0.f, 0.f};
        sa[g][1] = f4_t{0.f, 0.f, 0.f, 0.f};
        score_group<0, CHAIN>(lds, ac, tr.kq[g][0], tr.kq[g][1], qa, qlo, group_operand<0>(lds, ac, tr.kq[g][0]),
                              group_operand<0>(lds, ac, tr.kq[g][1]), sa[g][0], sa[g][1]);
      }
    }

    if constexpr (first) QKV_STAMP(kPhScores);
    // ---------------- staging: value codes and norms ----------------
    if constexpr (kUnits) {
      // (they take the place of the key units, which other lanes have read)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      stage_values(st, lane_o, tr.v);
    } else {
      stage_rows(st, lane_o, tr, scale2);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // the key registers are free: the next tile's keys fly during the softmax and the
    // value products (its values, during its scores: there are no registers for both)
    if (next >= 0) {
      next_row = wave_tile_row(next);
      load_tile_keys<0, kAhead>(p, next_row, p.num_kv, h, lane, tr);
    }

    // dense is wave-uniform: the common full tile (every key visible to every
    // query of the group) skips the per-key rule
    const bool dense = ts + kTile <= hi_first && rule.all_visible(ts + kTile);
    float s[4][4];
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const f4_t k0 = *reinterpret_cast<const f4_t*>(st + kStKn + 16 * g + 4 * row);
      const f4_t k1 = *reinterpret_cast<const f4_t*>(st + kStKn + kKeyPitch + 16 * g + 4 * row);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s[g][r] = k0[r] * sa[g][0][r] + k1[r] * sa[g][1][r];
        if constexpr (!CHAIN)
          s[g][r] += dpp_f<0x128>(s[g][r]);   // + the lo half of the query (column + 8, row_ror:8)
      }
    }
    if (!dense) {
#pragma unroll
      for (int g = 0; g < 4; g++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int key = ts + 16 * g + 4 * row + r;
          const bool vis = (key < hi_col) & rule.visible(key, active_end);   // padded keys too
          s[g][r] = vis ? s[g][r] : -INFINITY;
        }
    }

    // ---------------- online softmax of head `col` (its 64 keys sit in 4 rows) ----------------
    float mt = s[0][0];
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
      for (int r = 0; r < 4; r++) mt = fmaxf(mt, s[g][r]);
    mt = xrow_max(mt);
    const float mn = fmaxf(m2, mt);
    const float msafe = (mn == -INFINITY) ? 0.0f : mn;   // all keys so far masked: p = 0
    const float corr = __builtin_amdgcn_exp2f(m2 - msafe);
    float ps = 0.0f;
#pragma unroll
    for (int g = 0; g < 4; g++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s[g][r] = __builtin_amdgcn_exp2f(s[g][r] - msafe);
        ps += s[g][r];
      }
    lsum = lsum * corr + ps;
    m2 = mn;
    if constexpr (!first) {   // accumulators are still zero on the first tile
      // accumulator rows are heads 4*row + r: their factors come from lanes 4*row + r
      if (row == 0) st[kStCorr + col] = corr;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const f4_t cr = *reinterpret_cast<const f4_t*>(st + kStCorr + 4 * row);
#pragma unroll
      for (int t = 0; t < 16; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[t][r] *= cr[r];
    }

    if constexpr (first) QKV_STAMP(kPhSoftmax);
    // ---------------- values ----------------
    // 32-key chunk c2: MFMA k index i <-> key 32*c2 + 4*row + i (i < 4) and
    // 32*c2 + 16 + 4*row + (i - 4) (i >= 4), in both operands.  A = p * value
    // norm (head `col`, this lane's own probabilities), B = codes of 8 keys
    // in dim group `col`.
    {
      ValuePass vp[2];
      uint32_t cp[8], cq[8];
      value_pass_load(st, stu, 0, row, col, s, vp[0]);
      value_pairs<0>(lds, ac, vp[0].x, cp);
      value_pairs<1>(lds, ac, vp[0].x, cq);
      value_steps<0, first>(lds, ac, vp, cp, cq, acc, st, stu, row, col, s);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // lo and hi are wave-uniform (a paged workgroup serves one query): the tile
  // loop is a scalar loop
  if constexpr (MODE == 2) {
    auto tile = [&](int k) { return k < n_sel ? __builtin_amdgcn_readlane(sel, k) * kTile : -1; };
    if (sw < n_sel) {
      int ts = tile(sw + spw);
      tile_body(std::true_type{}, ts0, ts);
      for (int k = sw + spw; k < n_sel; k += spw) {
        const int next = tile(k + spw);
        load_tile_values(p, next_row, p.num_kv, h, lane, tr);
        tile_body(std::false_type{}, ts, next);
        ts = next;
      }
    } else {
#pragma unroll
      for (int t = 0; t < 16; t++) acc[t] = f4_t{0.f, 0.f, 0.f, 0.f};
    }
  } else if (ts0 < hi) {
    auto following = [&](int ts) { return ts + kStep < hi ? ts + kStep : -1; };
    if constexpr (APPEND)
      if (fa_wave == wave && ts0 <= p.start_pos && p.start_pos < ts0 + kTile)
        patch_new_key(tr, reinterpret_cast<const uint32_t*>(lds + kLdsNewRow), p.start_pos - ts0, lane);
    tile_body(std::true_type{}, ts0, following(ts0));
    for (int ts = ts0 + kStep; ts < hi; ts += kStep) {
      load_tile_keys<kAhead, 8>(p, next_row, p.num_kv, h, lane, tr);
      load_tile_values(p, next_row, p.num_kv, h, lane, tr);
      if constexpr (APPEND)
        if (fa_wave == wave && ts <= p.start_pos && p.start_pos < ts + kTile)
          patch_new_key(tr, reinterpret_cast<const uint32_t*>(lds + kLdsNewRow), p.start_pos - ts, lane);
      tile_body(std::false_type{}, ts, following(ts));
    }
  } else {
#pragma unroll
    for (int t = 0; t < 16; t++) acc[t] = f4_t{0.f, 0.f, 0.f, 0.f};
  }
  lsum = xrow_sum(lsum);
  QKV_STAMP(kPhTiles);

  // ---------------- merge the waves in LDS ----------------
  __syncthreads();
  QKV_STAMP(kPhTileBar);
  float* mo = reinterpret_cast<float*>(lds + kLdsMergeO);    // [wave][8][256]
  float* ml = reinterpret_cast<float*>(lds + kLdsMergeML);
  // (row offset recomputed from the thread index rather than held through the loop)
  int row4 = ((int)threadIdx.x & 63) >> 4 << 2;
  asm volatile("" : "+v"(row4));
  if (row4 < rows_used) {   // accumulator rows 4*row + r; rows >= rows_used are unused
    // acc tile t: rows 4*row+r, dim 128*(t>>3) + 8*col + (t&7): 16-byte stores
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int q4 = 0; q4 < 4; q4++) {
        const int t = 4 * q4;   // tiles t..t+3: dims 128*(q4>>1) + 8*col + 4*(q4&1) + 0..3
        *reinterpret_cast<f4_t*>(mo + (wave * 16 + row4 + r) * kHD + 128 * (q4 >> 1) + 8 * col +
                                 4 * (q4 & 1)) = f4_t{acc[t][r], acc[t + 1][r], acc[t + 2][r], acc[t + 3][r]};
      }
  }
  if (row == 0) {
    ml[kMlW0 + wave * 16 + col] = m2;
    ml[kMlLw0 + wave * 16 + col] = lsum;
  }
  __syncthreads();
  QKV_STAMP(kPhMergeBar);
  const int rows = rows_used;
  // fast path: every merged piece goes straight to its record
  const __amdgpu_buffer_rsrc_t rml =
      __builtin_amdgcn_make_buffer_rsrc(p.ws_ml, 0, MODE == 0 ? p.ws_ml_bytes : 0u, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t ro =
      __builtin_amdgcn_make_buffer_rsrc(p.ws_o, 0, MODE == 0 ? p.ws_o_bytes : 0u, kBufferRsrcWord3);
  // (an opaque copy of gqa: its division reciprocal is formed here, not held
  // in a register through the tile loop)
  int gqa_m = gqa;
  asm volatile("" : "+s"(gqa_m));
  if constexpr (MODE == 2) {
    // rows of split i, waves i spw ..: merged into slot (i spw, row), scalars at i rows + row
    for (int idx = threadIdx.x; idx < p.wg_splits * rows * 64; idx += kThreads) {
      const int ri = idx >> 6, d4 = (idx & 63) * 4, r = ri % rows, w0 = ri / rows * spw;
      float M = -INFINITY;
      for (int w = w0; w < w0 + spw; w++) M = fmaxf(M, ml[kMlW0 + w * 16 + r]);
      float L = 0.f;
      f4_t o = {0.f, 0.f, 0.f, 0.f};
      for (int w = w0; w < w0 + spw; w++) {
        const float mw = ml[kMlW0 + w * 16 + r];
        const float wt = (mw == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(mw - M);
        L += wt * ml[kMlLw0 + w * 16 + r];
        o += wt * *reinterpret_cast<const f4_t*>(mo + (w * 16 + r) * kHD + d4);
      }
      *reinterpret_cast<f4_t*>(mo + (w0 * 16 + r) * kHD + d4) = o;   // own elements only
      if (d4 == 0) {
        ml[kMlM + ri] = M;
        ml[kMlL + ri] = L;
      }
    }
    __syncthreads();
    finish_rows(lds, p, h, t0, rows, chunk * p.wg_splits, p.wg_splits, 16 * spw);
    return;
  }
  for (int idx = threadIdx.x; idx < rows * 64; idx += kThreads) {
    const int r = idx >> 6, d4 = (idx & 63) * 4;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; w++) M = fmaxf(M, ml[kMlW0 + w * 16 + r]);
    float L = 0.f;
    f4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; w++) {
      const float mw = ml[kMlW0 + w * 16 + r];
      const float wt = (mw == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(mw - M);
      L += wt * ml[kMlLw0 + w * 16 + r];
      o += wt * *reinterpret_cast<const f4_t*>(mo + (w * 16 + r) * kHD + d4);
    }
    if constexpr (MODE == 1) {
      *reinterpret_cast<f4_t*>(mo + r * kHD + d4) = o;   // wave-0 slot, own elements only
      if (d4 == 0) {
        ml[kMlM + r] = M;
        ml[kMlL + r] = L;
      }
    } else if (has_work) {
      store_record_piece(p, rml, ro, h * gqa_m + r % gqa_m, rec_t0 + r / gqa_m, rec_chunk, d4, o, M, L);
    }
  }

  if constexpr (MODE == 1) {
    __syncthreads();
    finish_rows(lds, p, h, t0, rows, chunk, 1, 0);
    return;
  }

  // ---------------- fast path: tagged records, designated mergers ----------------
  QKV_STAMP(kPhMerged);
  if (has_work) publish_records(p, rml, h, gqa_m, rec_t0, rows, rec_chunk, out == nullptr);
  QKV_STAMP(kPhPublished);
  if (out == nullptr) return;   // (merged by a launch of its own)
#ifdef QKV_PHASE_TRACE
  if (threadIdx.x < 3) *reinterpret_cast<uint64_t*>(lds + kLdsMergeO + kTracePolledByte + 8 * threadIdx.x) = 0;
#endif
  using ML = MergeLayout<kThreads>;
  static_assert(kLdsMergeO + ML::kRedFloats * 4 <= kLdsMergeML, "merge reduction must fit");
  merge_phase<kThreads, true>(reinterpret_cast<float*>(lds + kLdsMergeO),
                              reinterpret_cast<f2_t*>(lds + kLdsMergeML), p, rml, ro, out);
#ifdef QKV_PHASE_TRACE
  __syncthreads();
  trace_st[kPhPolled] = *reinterpret_cast<const uint64_t*>(lds + kLdsMergeO + kTracePolledByte);
  trace_st[kPhRowsIn] = *reinterpret_cast<const uint64_t*>(lds + kLdsMergeO + kTracePolledByte + 8);
  trace_st[kPhFolded] = *reinterpret_cast<const uint64_t*>(lds + kLdsMergeO + kTracePolledByte + 16);
  QKV_STAMP(kPhEnd);
  if (lane < 15 && blockIdx.x < kTraceMaxWgs) {
    uint64_t v = 0;
#pragma unroll
    for (int i = 0; i < 15; i++) v = lane == i ? trace_st[i] : v;
    qkv_phase_stamps[(blockIdx.x * kWaves + wave) * 16 + lane] = v;
  }
  if (lane == 0 && blockIdx.x < kTraceMaxWgs)
    qkv_phase_stamps[(blockIdx.x * kWaves + wave) * 16 + kPhXcd] =
        __builtin_amdgcn_s_getreg((3 << 11) | 20) & 15u;   // HW_REG_XCC_ID bits 3:0
#endif
}

size_t tq3_attn_lds_bytes() { return kLdsTotal; }

#ifdef QKV_PHASE_TRACE
}  // namespace qkv
// Diagnostic build only: copies the phase stamps of the last fast-path
// launch (n <= kTraceMaxWgs * 8 * 16 values) to host memory.
extern "C" int qkv_debug_phase_stamps(uint64_t* host, size_t n) {
  if (host == nullptr || n > sizeof(qkv::qkv_phase_stamps) / 8) return -1;
  return hipMemcpyFromSymbol(host, HIP_SYMBOL(qkv::qkv_phase_stamps), n * 8, 0, hipMemcpyDeviceToHost) ==
                 hipSuccess ? 0 : -6;
}
extern "C" int qkv_debug_phase_clear() {
  void* p = nullptr;
  if (hipGetSymbolAddress(&p, HIP_SYMBOL(qkv::qkv_phase_stamps)) != hipSuccess) return -6;
  return qkv::launch_fill_zero(p, sizeof(qkv::qkv_phase_stamps), nullptr) == hipSuccess ? 0 : -6;
}
namespace qkv {
#endif

// ---- the allocation-free decode's scratch ----------------------------------
// One fixed-size array per GPU, holding the fast path's workspace layout
// (header, record scalars, record rows).  In host code `scratch` names a
// host-side stand-in, not a device address: kernels only ever receive the
// address hipGetSymbolAddress returns for the current device, kept per device.
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

namespace {
std::mutex g_scratch_mu;
void* g_scratch_ptr[64];
}  // namespace

hipError_t noalloc_scratch(int device, bool clear, hipStream_t stream, void** ptr) {
  if (device < 0 || device >= 64) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  bool fresh = false;
  if (g_scratch_ptr[device] == nullptr) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (p == nullptr) return hipErrorInvalidSymbol;
    g_scratch_ptr[device] = p;
    fresh = true;
  }
  *ptr = g_scratch_ptr[device];
  if (clear || fresh) return launch_fill_zero(*ptr, kNoAllocScratchBytes, stream);
  return hipSuccess;
}

constexpr int kResident = 256;   // workgroups that the GPU holds at once: one per CU
hipError_t launch_tq3_attn(const AttnArgs& a, int mode, uint16_t* out, hipStream_t stream) {
  const int groups = (a.sub_n + a.qpw - 1) / a.qpw * a.n_chunks;
  const int per = 8 * a.num_kv;
  int n_wg = (groups + 7) / 8 * per;
  const bool apart = mode == 0 && merges_apart(a, kResident);
  // Fast path: one workgroup per merge unit -- a short context with several queries
  // has more units than chunks, and a merger takes its units one after the other
  // (4 queries over 301 keys: 128 units on 32 workgroups 22.7 us, on 128 15.3).
  if (mode == 0 && !apart) n_wg = std::max(n_wg, (2 * a.num_q * a.sub_n + per - 1) / per * per);
  uint16_t* merged = apart ? nullptr : out;
  dim3 grid(n_wg), block(kThreads);
  if (mode == 0 && a.qpw * (a.num_q / a.num_kv) > 8)
    hipLaunchKernelGGL((tq3_attn_kernel<0, true>), grid, block, 0, stream, QKV_ATTN_LEAD_ARGS(a), a, merged);
  else if (mode == 0 && a.k_new != nullptr)
    hipLaunchKernelGGL((tq3_attn_kernel<0, false, true>), grid, block, 0, stream, QKV_ATTN_LEAD_ARGS(a), a, merged);
  else if (mode == 0)
    hipLaunchKernelGGL((tq3_attn_kernel<0>), grid, block, 0, stream, QKV_ATTN_LEAD_ARGS(a), a, merged);
  else if (mode == 1)
    hipLaunchKernelGGL((tq3_attn_kernel<1>), grid, block, 0, stream, QKV_ATTN_LEAD_ARGS(a), a, out);
  else
    hipLaunchKernelGGL((tq3_attn_kernel<2>), grid, block, 0, stream, QKV_ATTN_LEAD_ARGS(a), a, out);
  const hipError_t e = hipGetLastError();
  return e != hipSuccess || !apart ? e : launch_record_merge(a, true, out, stream);
}

}  // namespace qkv
