// attn_mq.hip -- single-launch decode of multi-query calls (verify blocks):
// every cache tile is read once for up to 64 (query, head) columns (gfx950).
//
// Reference semantics: the split kernels with sub_n > 1 and their merge
// (attention.cuh:1905-2177, 2633-2801, 1837-1891), over Q8_0 keys with Q8_0 or
// TQ3 values.  Column c = qi * gqa + hh of a workgroup is q head h * gqa + hh
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
//            exchange maxima and the sums and accumulators get rescaled.
//   values   wave w owns dims 32 w .. 32 w + 31 of all columns: A = the
//            probabilities (one 16-byte read per 16 columns and 32 keys), B =
//            its own dims of 32 keys, decoded in registers.  32 accumulators
//            per lane and no merge of waves at the end: every wave stores its
//            dims of the records itself.
// One barrier per tile: the scores of tile t + 1 follow the value product of
// tile t in the same interval (three staging buffers, two of probabilities).
// Records are merged across workgroups as in the
// other fast paths (attn_fastmerge.h).
#include <algorithm>
#include <type_traits>

#include "attn_common.h"
#include "attn_fastmerge.h"
#include "attn_tq3_lut.h"
#include "qkv_device.h"

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
// How far (log2 units) a score may exceed its column's reference maximum
// before the reference is raised: weights stay below 2^8, and the reference
// settles within the first tiles, so that a tile normally needs no exchange of
// maxima between the waves.
constexpr float kSlack = 8.0f;
constexpr int kMaxWgs = 256;   // one workgroup per CU

// Centroid-pair table of the value codes: entry e (two 3-bit codes) of lane L
// at byte e * 256 + 4 * L (64 entries, so indexes are masked to 6 bits).
constexpr int kLutBytes = 64 * 64 * 4;

template <bool VT>
struct MqLds {
  static constexpr int kKBuf = kTile * kQ8Pitch;
  static constexpr int kVBuf = VT ? 32 * kVgPitch * 4 : kTile * kQ8Pitch;
  static constexpr int kPBuf = (VT ? 2 : 1) * 64 * 128;   // [64 columns][64 keys] fp16 (TQ3: per 128-block)
  static constexpr int kK = VT ? kLutBytes : 0;           // three buffers each
  static constexpr int kV = kK + 3 * kKBuf;
  static constexpr int kVn = kV + 3 * kVBuf;              // TQ3 value norms [3 buffers][2 blocks][64] f32
  static constexpr int kP = kVn + (VT ? 3 * 2 * kTile * 4 : 0);   // probabilities, two buffers
  static constexpr int kMx = kP + 2 * kPBuf;              // [64 columns][4 key groups] f32
  static constexpr int kCorr = kMx + 64 * 4 * 4;          // [64] rescale factors, then 4 flags
  static constexpr int kSc = kCorr + 64 * 4 + 16;         // Q8 values: per wave [64 keys] fp16 scales of its block
  static constexpr int kEnd = kSc + (VT ? 0 : kWaves * kTile * 2);
  // after the tile loop
  static constexpr int kRed = 0;                          // mergers
  static constexpr int kMls = kRed + kWaves * 128 * 4;
  static constexpr int kSum = kMls + 256 * 8;             // [4][64] sums, [64] maxima, [64] record indices
  static_assert(kSum + 6 * 64 * 4 <= kP, "end-of-kernel scalars must not reach the probabilities");
  static_assert(kEnd <= 160 * 1024, "LDS");
};

// One tile's rows in flight.  Q8_0 rows: 16-byte pieces c = tid + 512 i of the
// 1,152 key pieces (then, for Q8_0 values, the 1,152 value pieces), piece c of
// row c / 18.  TQ3 values: thread (row tid / 8, pc = tid % 8) takes the 12
// bytes of code groups 4 pc .. 4 pc + 3, waves 0 and 1 the norms of block 0
// and 1 (lane = key).
template <bool VT>
struct MqRegs {
  u4_t q[VT ? 3 : 5];
  u3_t v;
  float vn;
};

// The rows of a thread's 16-byte Q8_0 pieces, 6 bits each: one register through
// the tile loop, from which a piece's offsets are formed where they are used
// (opaque, so that they are not hoisted into registers of their own).
template <bool VT>
__device__ __forceinline__ uint32_t mq_rows(int tid) {
  uint32_t v = 0u;
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

template <bool VT>
__device__ __forceinline__ void mq_load(const AttnArgs& p, int ts, int h, int tid, int wave, int lane, uint32_t rows,
                                        MqRegs<VT>& r) {
  const uint64_t row0 = (uint64_t)(uint32_t)ts * (uint32_t)p.num_kv;
  const __amdgpu_buffer_rsrc_t rk = cache_rsrc(p.k, row0 * kQ8Row, p.kv_bytes);
  asm volatile("" : "+v"(rows));
  auto piece = [&](int i, const __amdgpu_buffer_rsrc_t& rs, bool val) {
    return __builtin_amdgcn_raw_buffer_load_b128(rs, mq_piece(rows, tid, i, val).cache(p.num_kv, h), 0, 0);
  };
  r.q[0] = piece(0, rk, false);
  r.q[1] = piece(1, rk, false);
  if constexpr (VT) {
    const __amdgpu_buffer_rsrc_t rv = cache_rsrc(p.v, row0 * kTq3Row, p.v_bytes);
    if (wave < 2) {   // pieces 1024 .. 1151
      r.q[2] = piece(2, rk, false);
      r.vn = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
          rv, (uint32_t)(lane * p.num_kv + h) * (uint32_t)kTq3Row + 52u * (uint32_t)wave, 0, 0));
    }
    const int row = tid >> 3, pc = tid & 7;
    r.v = __builtin_amdgcn_raw_buffer_load_b96(
        rv, (uint32_t)(row * p.num_kv + h) * (uint32_t)kTq3Row + 52u * (uint32_t)(pc >> 2) + 4u + 12u * (uint32_t)(pc & 3),
        0, 0);
  } else {
    const __amdgpu_buffer_rsrc_t rv = cache_rsrc(p.v, row0 * kQ8Row, p.kv_bytes);
    r.q[2] = wave < 2 ? piece(2, rk, false) : piece(2, rv, true);   // pieces 1024 .. 1535
    r.q[3] = piece(3, rv, true);
    if (wave < 4) r.q[4] = piece(4, rv, true);                      // pieces 2048 .. 2303
  }
}

template <bool VT>
__device__ __forceinline__ void mq_stage(uint8_t* lds, int buf, int tid, int wave, int lane, uint32_t rows,
                                         const MqRegs<VT>& r) {
  using L = MqLds<VT>;
  uint8_t* kd = lds + L::kK + buf * L::kKBuf;
  uint8_t* vd = lds + L::kV + buf * L::kVBuf;
  asm volatile("" : "+v"(rows));
  auto put = [&](int i, uint8_t* d, bool val) {
    *reinterpret_cast<u4_t*>(d + mq_piece(rows, tid, i, val).lds()) = r.q[i];
  };
  put(0, kd, false);
  put(1, kd, false);
  if constexpr (VT) {
    if (wave < 2) {
      put(2, kd, false);
      *reinterpret_cast<float*>(lds + L::kVn + ((buf * 2 + wave) * kTile + lane) * 4) = r.vn;
    }
    const int row = tid >> 3, pc = tid & 7;
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

template <bool VT>
__global__ __launch_bounds__(kThreads, 1) void mq_attn_kernel(QKV_ATTN_LEAD_PARAMS, AttnArgs pin, uint16_t* out) {
  QKV_ATTN_LEAD_APPLY(p, pin);
  using L = MqLds<VT>;
  __shared__ __attribute__((aligned(16))) uint8_t lds[L::kEnd];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int gqa = __builtin_amdgcn_readfirstlane(p.num_q / p.num_kv);
  // work id, XCD-aware: the num_kv workgroups of one (query block, chunk) share an XCD
  int h, t0, chunk;
  bool has_work;
  {
    const int Lid = blockIdx.x;
    const int xcd = Lid & 7, r = Lid >> 3;
    h = r % p.num_kv;
    const int g = (r / p.num_kv) * 8 + xcd;
    const int groups = (p.sub_n + p.qpw - 1) / p.qpw;
    has_work = g < groups * p.n_chunks;
    const int tq = has_work ? g / p.n_chunks : 0;
    chunk = has_work ? g - tq * p.n_chunks : 0;
    t0 = tq * p.qpw;
  }
  const int nq = min(p.qpw, p.sub_n - t0);
  const int cols = __builtin_amdgcn_readfirstlane(nq * gqa);   // <= 64
  const int n = lane & 15, kb = lane >> 4;
  const int kg = wave & 3, ch = wave >> 2;
  // ---- queries: slice s of column 32 ch + 16 cg + n, dims
  // 32 (2 kb + (s >> 2)) + 8 (s & 3) .. + 7 (the lane's two Q8_0 blocks)
  u4_t qa[2][8];
  int t_col[2];
  {
    const uint32_t q_extent = (uint32_t)(p.sub_n * p.num_q * kHD * 2);
    const __amdgpu_buffer_rsrc_t rq =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.q), 0, q_extent, kBufferRsrcWord3);
#pragma unroll
    for (int cg = 0; cg < 2; cg++) {
      const int c = 32 * ch + 16 * cg + n;
      t_col[cg] = t0 + min(c / gqa, nq - 1);
      const uint32_t off = c < cols ? (uint32_t)(((t0 + c / gqa) * p.num_q + h * gqa + c % gqa) * kHD * 2 + 128 * kb)
                                    : q_extent;   // (columns past `cols`: zero queries, never stored)
#pragma unroll
      for (int s = 0; s < 8; s++) qa[cg][s] = __builtin_amdgcn_raw_buffer_load_b128(rq, off + 16 * s, 0, 0);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- key range of the workgroup and of this lane's columns
  const int active_last = p.start_pos + t0 + nq;
  int lo = 0, hi = 0, hi_first = 0, hi_col[2] = {0, 0};
  if (has_work) {
    lo = chunk * p.chunk_keys;
    const int c_end = chunk == p.n_chunks - 1 ? active_last : lo + p.chunk_keys;
    hi = min(c_end, active_last);
    hi_first = min(c_end, p.start_pos + t0 + 1);
#pragma unroll
    for (int cg = 0; cg < 2; cg++) hi_col[cg] = min(c_end, p.start_pos + t_col[cg] + 1);
  }
  lo = __builtin_amdgcn_readfirstlane(lo);
  hi = __builtin_amdgcn_readfirstlane(hi);
  hi_first = __builtin_amdgcn_readfirstlane(hi_first);
  const int n_tiles = hi > lo ? (hi - lo + kTile - 1) / kTile : 0;
  const uint32_t rows = mq_rows<VT>(tid);
  MqRegs<VT> ra, rb;
  if (n_tiles > 0) mq_load<VT>(p, lo, h, tid, wave, lane, rows, ra);
  if (n_tiles > 1) mq_load<VT>(p, lo + kTile, h, tid, wave, lane, rows, rb);
  const uint32_t lane4 = 4u * (uint32_t)lane;
  if constexpr (VT) {
    // table: wave w writes every lane's copy of entries 8 w .. 8 w + 7
    const uint32_t hi16 = centroid_scaled_h((uint32_t)wave) << 16;
#pragma unroll
    for (int e = 0; e < 8; e++)
      *reinterpret_cast<uint32_t*>(lds + (8 * wave + e) * 256 + lane4) = centroid_scaled_h((uint32_t)e) | hi16;
  }
  int* flag_s = reinterpret_cast<int*>(lds + L::kCorr + 256);
  if (tid < 3) flag_s[tid] = 0;
  // tiles 0 and 1 staged, tile 2 on its way
  if (n_tiles > 0) mq_stage<VT>(lds, 0, tid, wave, lane, rows, ra);
  if (n_tiles > 1) mq_stage<VT>(lds, 1, tid, wave, lane, rows, rb);
  if (n_tiles > 2) mq_load<VT>(p, lo + 2 * kTile, h, tid, wave, lane, rows, ra);
  __syncthreads();

  const bool score_live = 32 * ch < cols;            // wave-uniform: the column half holds columns
  const int groups_live = (cols + 15) >> 4;          // 16-column groups that hold columns
  const float scale2 = p.scale_log2;
  float m2[2] = {-INFINITY, -INFINITY}, lsum[2] = {0.0f, 0.0f};
  f4_t acc[4][2];
#pragma unroll
  for (int g = 0; g < 4; g++) acc[g][0] = acc[g][1] = f4_t{0.f, 0.f, 0.f, 0.f};
  float* mx = reinterpret_cast<float*>(lds + L::kMx);
  float* corr_s = reinterpret_cast<float*>(lds + L::kCorr);
  // this lane's dims of the value product: 32 wave + 2 n and + 1
  const uint32_t vsh = 6u * (uint32_t)(n & 3);                          // TQ3: field of dims 2 (n & 3), + 1 of the group
  const uint32_t vsel0 = 0x0c000c00u + 0x00040000u + 0x00010001u * (uint32_t)(2 * (n & 1));   // Q8: byte 2 (n & 1)
  const uint32_t vsel1 = vsel0 + 0x00010001u;

  int b3 = 0;   // t mod 3: the tile's staging buffer and flag
  for (int t = 0; t < n_tiles; t++) {
    const int ts = lo + t * kTile;
    const uint8_t* kbuf = lds + L::kK + b3 * L::kKBuf;
    const uint8_t* vbuf = lds + L::kV + b3 * L::kVBuf;
    const float* vnorm = reinterpret_cast<const float*>(lds + L::kVn) + b3 * 2 * kTile;
    uint8_t* pbuf = lds + L::kP + (t & 1) * L::kPBuf;
    const bool dense = ts + kTile <= hi_first;   // every key visible to every column
    bool v_nonfinite = false;
    if constexpr (!VT) {
      // the scales of this wave's value block, one key per lane, to the wave's own area
      const uint32_t d = *reinterpret_cast<const uint16_t*>(vbuf + lane * kQ8Pitch + 36 * wave + 34);
      *reinterpret_cast<uint16_t*>(lds + L::kSc + (wave * kTile + lane) * 2) = (uint16_t)d;
      v_nonfinite = __builtin_amdgcn_ballot_w64((d & 0x7c00u) == 0x7c00u) != 0;
    }
    float s[2][4], ps[2] = {0.0f, 0.0f};
    // probabilities of the wave's 16 keys to LDS: column c's 16-byte unit
    // (half kg >> 1, kb), stored at unit ^ ((c >> 1) & 7), holds keys
    // 32 (kg >> 1) + 4 kb + 0..3 and + 16..19 (the k order of the value
    // product).  Returns whether a weight is out of the fp16 range kept free.
    auto put_p = [&]() {
      bool big = false;
#pragma unroll
      for (int cg = 0; cg < 2; cg++) {
        const int c = 32 * ch + 16 * cg + n;
        const float msafe = (m2[cg] == -INFINITY) ? 0.0f : m2[cg];   // no key visible yet: p = 0
        float pr[4];
#pragma unroll
        for (int r = 0; r < 4; r++) pr[r] = __builtin_amdgcn_exp2f(s[cg][r] - msafe);
        ps[cg] = (pr[0] + pr[1]) + (pr[2] + pr[3]);
        uint8_t* pd = pbuf + c * 128 + 16 * (((kg >> 1) * 4 + kb) ^ ((c >> 1) & 7)) + 8 * (kg & 1);
        if constexpr (VT) {
#pragma unroll
          for (int j = 0; j < 2; j++) {
            const f4_t vn = *reinterpret_cast<const f4_t*>(vnorm + j * kTile + 16 * kg + 4 * kb);
            h4_t w;
#pragma unroll
            for (int r = 0; r < 4; r++) {
              float x = pr[r] * vn[r];
              // (a masked key's norm may be inf or NaN: its weight is 0)
              if (!dense) x = s[cg][r] == -INFINITY ? 0.0f : x;
              big = big || x > 32768.0f;
              w[r] = (_Float16)x;
            }
            *reinterpret_cast<h4_t*>(pd + j * 64 * 128) = w;
          }
        } else {
          h4_t w;
#pragma unroll
          for (int r = 0; r < 4; r++) w[r] = (_Float16)pr[r];
          *reinterpret_cast<h4_t*>(pd) = w;
        }
      }
      return big;
    };
    if (score_live) {
      // ---- scores: D rows = keys 16 kg + 4 kb + r, D column = 32 ch + 16 cg + n
      uint32_t k[18];
      const u2_t* kr = reinterpret_cast<const u2_t*>(kbuf + (16 * kg + n) * kQ8Pitch + 72 * kb);
#pragma unroll
      for (int i = 0; i < 9; i++) {
        const u2_t c = kr[i];
        k[2 * i] = c[0];
        k[2 * i + 1] = c[1];
      }
      f4_t sa[2] = {f4_t{0.f, 0.f, 0.f, 0.f}, f4_t{0.f, 0.f, 0.f, 0.f}};
      auto slice = [&](auto S) {
        constexpr int si = decltype(S)::value;
        const h8_t a = q8_key_operand<si>(k);
#pragma unroll
        for (int cg = 0; cg < 2; cg++)
          sa[cg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, __builtin_bit_cast(h8_t, qa[cg][si]), sa[cg], 0, 0, 0);
      };
      slice(std::integral_constant<int, 0>{});
      slice(std::integral_constant<int, 1>{});
      slice(std::integral_constant<int, 2>{});
      slice(std::integral_constant<int, 3>{});
      slice(std::integral_constant<int, 4>{});
      slice(std::integral_constant<int, 5>{});
      slice(std::integral_constant<int, 6>{});
      slice(std::integral_constant<int, 7>{});
      bool over = false;
#pragma unroll
      for (int cg = 0; cg < 2; cg++) {
#pragma unroll
        for (int r = 0; r < 4; r++) s[cg][r] = sa[cg][r] * scale2;
        if (!dense) {
#pragma unroll
          for (int r = 0; r < 4; r++) s[cg][r] = ts + 16 * kg + 4 * kb + r < hi_col[cg] ? s[cg][r] : -INFINITY;
        }
        const float mt = fmaxf(fmaxf(s[cg][0], s[cg][1]), fmaxf(s[cg][2], s[cg][3]));
        over = over || mt > m2[cg] + kSlack;
      }
      over = put_p() || over;
      if (__builtin_amdgcn_ballot_w64(over) != 0 && lane == 0) flag_s[b3] = 1;
    }
    __syncthreads();   // probabilities and flag are in; buffer (t + 2) mod 3 is free
    const int raise = __builtin_amdgcn_readfirstlane(flag_s[b3]);
    const int b3n = b3 == 2 ? 0 : b3 + 1, b3nn = b3 == 0 ? 2 : b3 - 1;   // (t + 1) mod 3, (t + 2) mod 3
    if (t + 2 < n_tiles) {
      mq_stage<VT>(lds, b3nn, tid, wave, lane, rows, ra);
      if (t + 3 < n_tiles) mq_load<VT>(p, ts + 3 * kTile, h, tid, wave, lane, rows, ra);
    }
    if (tid == 0) flag_s[b3nn] = 0;   // (set by tile t + 2, after the next barrier)
    if (raise) {
      // some column's maximum rose past the slack: every column's reference
      // becomes its running maximum, accumulators and sums are rescaled and
      // the tile's probabilities are formed again
      if (score_live) {
#pragma unroll
        for (int cg = 0; cg < 2; cg++) {
          const float mt = xrow_max(fmaxf(fmaxf(s[cg][0], s[cg][1]), fmaxf(s[cg][2], s[cg][3])));
          if (kb == 0) mx[(32 * ch + 16 * cg + n) * 4 + kg] = mt;
        }
      }
      __syncthreads();
      if (score_live) {
#pragma unroll
        for (int cg = 0; cg < 2; cg++) {
          const int c = 32 * ch + 16 * cg + n;
          const f4_t mk = *reinterpret_cast<const f4_t*>(mx + 4 * c);
          const float mn = fmaxf(m2[cg], fmaxf(fmaxf(mk[0], mk[1]), fmaxf(mk[2], mk[3])));
          const float corr = __builtin_amdgcn_exp2f(m2[cg] - ((mn == -INFINITY) ? 0.0f : mn));
          lsum[cg] *= corr;
          m2[cg] = mn;
          if (kg == 0 && kb == 0) corr_s[c] = corr;
        }
        put_p();
      }
      __syncthreads();
#pragma unroll
      for (int g = 0; g < 4; g++)
        if (g < groups_live) {
          const f4_t cr = *reinterpret_cast<const f4_t*>(corr_s + 16 * g + 4 * kb);
#pragma unroll
          for (int e = 0; e < 2; e++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[g][e][r] *= cr[r];
        }
    }
#pragma unroll
    for (int cg = 0; cg < 2; cg++) lsum[cg] += ps[cg];
    // ---- values: acc[g][e] += P(16 columns x 32 keys) V(32 keys x 16 dims)
    const uint8_t* pbase = pbuf + (VT ? (wave >> 2) * 64 * 128 : 0) + n * 128;
    auto p_operand = [&](int g, int c2) {   // columns 16 g + n, keys of half c2
      return *reinterpret_cast<const h8_t*>(pbase + 16 * g * 128 + 16 * ((c2 * 4 + kb) ^ ((n >> 1) & 7)));
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
          bv[0][i] = *reinterpret_cast<const uint32_t*>(lds + (((x[i] >> vsh) & 63u) << 8 | lane4));
          bv[1][i] = *reinterpret_cast<const uint32_t*>(lds + (((x[4 + i] >> (vsh + 3u)) & 63u) << 8 | lane4));
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
    if (!VT && v_nonfinite && !dense) {
      // a key that some query of the block does not see may have an inf or NaN
      // scale: 0 * inf must not reach that query's rows, so every query takes
      // products of its own, with the keys that it does not see zeroed
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
        for (int g = 0; g < 4; g++)
          if (g < groups_live) {
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
        for (int g = 0; g < 4; g++)
          if (g < groups_live) {
            const h8_t pa = p_operand(g, c2);
#pragma unroll
            for (int e = 0; e < 2; e++)
              acc[g][e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa, __builtin_bit_cast(h8_t, bv[e]), acc[g][e], 0, 0, 0);
          }
      }
    }
    b3 = b3n;
  }

  // ---- records: the waves of a column half hold its sums per key group, every
  // wave its dims of every column
  __syncthreads();
  float* sums = reinterpret_cast<float*>(lds + L::kSum);
  int* recs = reinterpret_cast<int*>(lds + L::kSum + 5 * 64 * 4);
  const __amdgpu_buffer_rsrc_t rml = __builtin_amdgcn_make_buffer_rsrc(p.ws_ml, 0, p.ws_ml_bytes, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(p.ws_o, 0, p.ws_o_bytes, kBufferRsrcWord3);
  int gqa_m = gqa;
  asm volatile("" : "+s"(gqa_m));   // (its reciprocal is formed here, not held through the loop)
#pragma unroll
  for (int cg = 0; cg < 2; cg++) {
    const float l = xrow_sum(lsum[cg]);
    const int c = 32 * ch + 16 * cg + n;
    if (kb == 0) {
      sums[kg * 64 + c] = l;
      if (kg == 0) sums[4 * 64 + c] = m2[cg];
    }
  }
  if (tid < 64) recs[tid] = (int)rec_index(p, h * gqa_m + tid % gqa_m, t0 + min(tid, cols - 1) / gqa_m, chunk);
  __syncthreads();
  if (has_work) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int R = 16 * g + 4 * kb + r;
        if (R < cols)
          __builtin_amdgcn_raw_buffer_store_b64(f2_t{acc[g][0][r], acc[g][1][r]}, ro,
                                                (uint32_t)((recs[R] * kHD + 32 * wave + 2 * n) * 4), 0, kCoherent);
      }
    }
    if (tid < cols)
      __builtin_amdgcn_raw_buffer_store_b64(
          f2_t{sums[4 * 64 + tid], (sums[tid] + sums[64 + tid]) + (sums[128 + tid] + sums[192 + tid])}, rml,
          (uint32_t)(recs[tid] * kRecMlBytes), 0, kCoherent);
    publish_records(p, rml, h, gqa_m, t0, cols, chunk);
  } else {
    __syncthreads();   // (the barrier publish_records passes)
  }
  merge_phase_paired<kThreads, VT>(reinterpret_cast<float*>(lds + L::kRed), reinterpret_cast<f2_t*>(lds + L::kMls), p,
                                   rml, ro, out);
}

}  // namespace

hipError_t launch_mq_attn(const AttnArgs& a, bool v_tq3, uint16_t* out, hipStream_t stream) {
  const int groups = (a.sub_n + a.qpw - 1) / a.qpw * a.n_chunks;
  // One round of the GPU holds a merger for every pair of merge units: a short
  // context, whose chunks are few, gets workgroups that only merge.
  const int mergers = std::min(a.num_q * a.sub_n, kMaxWgs);
  const int per = 8 * a.num_kv;
  const int n_wg = std::max((groups + 7) / 8, (mergers + per - 1) / per) * per;
  if (v_tq3)
    hipLaunchKernelGGL(mq_attn_kernel<true>, dim3(n_wg), dim3(kThreads), 0, stream, QKV_ATTN_LEAD_ARGS(a), a, out);
  else
    hipLaunchKernelGGL(mq_attn_kernel<false>, dim3(n_wg), dim3(kThreads), 0, stream, QKV_ATTN_LEAD_ARGS(a), a, out);
  return hipGetLastError();
}

}  // namespace qkv
