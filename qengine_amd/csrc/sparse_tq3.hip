// sparse_tq3.hip -- block selection for the block-sparse TQ3 verify (gfx950).
//
// Reference: the verify path of model.cuh:4589-4662 keeps per kv head a pool
// of 64-token block signatures over the TQ3 key cache (mean and sign-
// preserving max-abs of the dequantized keys, tq3_kpool_ms_update_kern,
// attention.cuh:2445-2533), scores every block for each verify query
// against the GQA-mean query, max(q.mean, beta * q.maxabs), and keeps the
// top_k blocks (build_block_index_ms_kern, sparse_attn/sparse_index.cuh:
// 214-330).  The attention over the selected blocks is tq3_attn_kernel<2>.
//
// The kernels here reproduce the reference's values exactly: the keys are
// dequantized bit for bit (tq3_group_dequant), the signature sums run in the
// reference's order, the block scores sum exact fp16 x fp16 products pairwise
// in the reference's order, and the selection is the reference's repeated
// argmax (highest score, lower block index on ties), sorted ascending.
#include <algorithm>

#include "attn_common.h"
#include "qkv_device.h"
#include "qkv_launch.h"

// the signature and score sums keep the reference's separate roundings
#pragma clang fp contract(off)

namespace qkv {

constexpr int kSpThreads = 256;
constexpr int kSpHD = 256;
constexpr int kPoolPitch = kSpHD * 2 + 16;   // bytes per staged key row (fp16)

// One workgroup per (kv head, position block n = blk_lo + i): the block's up
// to 64 key rows are dequantized into LDS (16 lanes per 128-element TQ3
// block), then thread c reduces dimension c over the rows in position order.
__global__ __launch_bounds__(kSpThreads) void tq3_kpool_kernel(KpoolArgs a) {
  __shared__ __attribute__((aligned(16))) uint8_t rows[64 * kPoolPitch];
  __shared__ float cent[8];
  const int n_upd = a.cur_blocks - a.blk_lo;
  const int h = blockIdx.x / n_upd;
  const int n = a.blk_lo + (int)(blockIdx.x - h * n_upd);
  const int t_lo = n * a.bsn;
  const int t_hi = min(t_lo + a.bsn, a.total_kv);
  const int n_pos = t_hi - t_lo;   // >= 1: n < cur_blocks
  const int tid = threadIdx.x;
  const int part = tid & 15;
  tq3_centroid_table(cent, tid);
  const Tq3LaneConst lc = tq3_lane_const(part);
  // units (position, 128-block): 16 per pass of the workgroup, at most 8
  // passes (64 rows); every pass's loads are issued before the first is used
  constexpr int kPasses = 2 * 64 / (kSpThreads / 16);
  Tq3Group gr[kPasses];
#pragma unroll
  for (int p = 0; p < kPasses; p++) {
    const int u0 = (tid >> 4) + p * (kSpThreads / 16);
    const int u = u0 < 2 * n_pos ? u0 : 0;   // a unit past the block's rows re-reads unit 0
    const uint8_t* src = reinterpret_cast<const uint8_t*>(a.k) +
                         ((uint64_t)(uint32_t)(t_lo + (u >> 1)) * (uint32_t)a.num_kv + h) * 104u +
                         (u & 1) * 52u;
    gr[p] = tq3_group_load(src, part);
  }
  __syncthreads();   // the centroid table
#pragma unroll
  for (int p = 0; p < kPasses; p++) {
    const int u = (tid >> 4) + p * (kSpThreads / 16);
    if (u < 2 * n_pos) {   // uniform over the unit's 16 lanes (lane exchange inside)
      const int pos = u >> 1, blk = u & 1;
      uint32_t pk[4];
      tq3_group_dequant(gr[p], part, cent, lc, pk);
      *reinterpret_cast<uint4*>(rows + pos * kPoolPitch + (blk * 128 + part * 8) * 2) =
          make_uint4(pk[0], pk[1], pk[2], pk[3]);
    }
  }
  __syncthreads();
  const int c = tid;   // 256 threads: one dimension each
  float sum = 0.0f, best_mag = 0.0f, best_val = 0.0f;
  for (int pos = 0; pos < n_pos; pos++) {
    const float x = h2f(*reinterpret_cast<const uint16_t*>(rows + pos * kPoolPitch + c * 2));
    sum += x;
    const float m = fabsf(x);
    if (m > best_mag) {
      best_mag = m;
      best_val = x;
    }
  }
  const long ob = ((long)h * a.stride + n) * kSpHD + c;
  a.k_pool[ob] = (uint16_t)f2h(sum / (float)n_pos);
  a.k_pool_max[ob] = (uint16_t)f2h(best_val);
}

constexpr int kScBlocks = 32;          // blocks scored per workgroup
constexpr int kScPitchDw = 132;        // staged pool row: 128 dwords + 4 (16-byte reads of 16 rows: 64 banks)
typedef uint32_t u4a4_t __attribute__((ext_vector_type(4), aligned(4)));

// One pair of dimensions: s + (q0 m0 + q1 m1), both products exact in fp32, their
// sum rounded once (an FMA onto the other product), then added to s.  The operands
// are fp16 halves (v_fma_mix_f32; q1 m1 + 0 is exact).  (v_dot2_f32_f16 does not
// give that rounding.)
__device__ __forceinline__ float pair_add(float s, uint32_t q, uint32_t m) {
  const float hi = __builtin_fmaf(h2f(q >> 16), h2f(m >> 16), 0.0f);
  return s + __builtin_fmaf(h2f(q & 0xffffu), h2f(m & 0xffffu), hi);
}

// Block scores, one workgroup per (kv head, 32 blocks, 8 NQ queries).  The
// blocks' mean and max-abs rows are staged in LDS; the GQA-mean queries
// (fp16-rounded, as the reference forms them, sparse_index.cuh:243-252) sit in
// LDS as fp16 pairs; thread (t, b) runs block b's two dot products for queries
// t, t + 8 .. over the 128 pairs in the reference's order (pair_add).  Scores (-inf
// past the query's causal block) go to the workspace [num_kv][sub_n][n_blocks].
// Half the VALU's 3 operations per pair and product, half the latency of the inputs:
// 16 queries over 2,049 blocks, 14.3 -> 11.3 us (with converted operands and a
// 4-byte LDS read each before).  NQ = 2 (more than 8 queries) reads every staged row
// once for two queries.
template <int NQ>
__global__ __launch_bounds__(kSpThreads) void block_score_kernel(BlockIndexArgs a, float* scores) {
  constexpr int kQueries = 8 * NQ;
  __shared__ __attribute__((aligned(16))) uint32_t rows_mean[kScBlocks * kScPitchDw];
  __shared__ __attribute__((aligned(16))) uint32_t rows_max[kScBlocks * kScPitchDw];
  __shared__ __attribute__((aligned(16))) uint32_t qa2[kQueries * kSpHD / 2];   // fp16 pairs
  const int nb_wg = (a.n_blocks + kScBlocks - 1) / kScBlocks;
  const int nq_wg = (a.sub_n + kQueries - 1) / kQueries;
  const int qg = blockIdx.x % nq_wg, r = blockIdx.x / nq_wg;
  const int h = r / nb_wg, b0 = (r - h * nb_wg) * kScBlocks, t0 = qg * kQueries;
  const int nt = min(kQueries, a.sub_n - t0);
  const int tid = threadIdx.x;
  const int gqa = a.num_q / a.num_kv;
  // Every load of the query and of the staging is issued before the first one is
  // used (one memory round trip for the workgroup's inputs).  GQA-mean queries:
  // thread i forms 8 dims of query i / 32 from its 8 (or gqa) heads' 16-byte
  // pieces (heads past gqa re-read the last head and are not added; queries past
  // the last re-read the last)
  u4a4_t qv[NQ][8];
#pragma unroll
  for (int k = 0; k < NQ; k++) {
    const int tq = min((tid >> 5) + 8 * k, nt - 1);
#pragma unroll
    for (int g = 0; g < 8; g++)
      qv[k][g] = *reinterpret_cast<const u4a4_t*>(
          a.q + ((long)(t0 + tq) * a.num_q + h * gqa + min(g, gqa - 1)) * kSpHD + (tid & 31) * 8);
  }
  // 32 blocks x {mean, max} x 512 B: 2048 16-byte pieces, 8 per thread
  // (blocks past the pool's end are read at its last block and not stored)
  static_assert(kScBlocks * 64 == 8 * kSpThreads, "8 staging pieces per thread");
  u4_t pv[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int piece = tid + k * kSpThreads;
    const int b = piece >> 6, w = piece & 63;   // w < 32: mean, else max; 8 dims each
    const int nbk = min(b0 + b, a.n_blocks - 1);
    pv[k] = *reinterpret_cast<const u4_t*>((w < 32 ? a.k_pool : a.k_pool_max) +
                                           ((long)h * a.stride + nbk) * kSpHD + (w & 31) * 8);
  }
  const float inv_g = a.inv_gqa;
#pragma unroll
  for (int k = 0; k < NQ; k++) {
    float s[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};   // heads in order (the reference's sum)
#pragma unroll
    for (int g = 0; g < 8; g++) {
      const uint32_t keep = g < gqa ? 0xffffffffu : 0u;   // (+ 0 leaves the sum as it is)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        s[2 * e] += h2f(qv[k][g][e] & keep & 0xffffu);
        s[2 * e + 1] += h2f((qv[k][g][e] & keep) >> 16);
      }
    }
    uint32_t pk[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      // the reference rounds s * (1/GQA) to fp32, then to fp16: the empty asm
      // keeps the fp32 product (no fused fp16-rounding mixed FMA)
      float p0 = s[2 * e] * inv_g, p1 = s[2 * e + 1] * inv_g;
      asm volatile("" : "+v"(p0), "+v"(p1));
      pk[e] = f2h(p0) | (f2h(p1) << 16);
    }
    *reinterpret_cast<uint4*>(qa2 + (8 * k + (tid >> 5)) * (kSpHD / 2) + (tid & 31) * 4) =
        make_uint4(pk[0], pk[1], pk[2], pk[3]);
  }
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int piece = tid + k * kSpThreads;
    const int b = piece >> 6, w = piece & 63;
    *reinterpret_cast<u4_t*>((w < 32 ? rows_mean : rows_max) + b * kScPitchDw + (w & 31) * 4) = pv[k];
  }
  __syncthreads();
  // thread -> (query tq, block b): 32 lanes of a wave are the 32 blocks of one query
  const int tq = tid / kScBlocks, b = tid - tq * kScBlocks;
  const uint32_t* mn = rows_mean + b * kScPitchDw;
  const uint32_t* mx = rows_max + b * kScPitchDw;
  const uint32_t* q = qa2 + tq * (kSpHD / 2);
  float s_mean[NQ], s_max[NQ];
#pragma unroll
  for (int k = 0; k < NQ; k++) s_mean[k] = s_max[k] = 0.0f;
#pragma unroll 4
  for (int c = 0; c < kSpHD / 2; c += 4) {
    const uint4 m4 = *reinterpret_cast<const uint4*>(mn + c), x4 = *reinterpret_cast<const uint4*>(mx + c);
    const uint32_t m[4] = {m4.x, m4.y, m4.z, m4.w}, x[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
    for (int k = 0; k < NQ; k++) {
      const uint4 q4 = *reinterpret_cast<const uint4*>(q + 8 * k * (kSpHD / 2) + c);
      const uint32_t qw[4] = {q4.x, q4.y, q4.z, q4.w};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        s_mean[k] = pair_add(s_mean[k], qw[e], m[e]);
        s_max[k] = pair_add(s_max[k], qw[e], x[e]);
      }
    }
  }
#pragma unroll
  for (int k = 0; k < NQ; k++) {
    const int n = b0 + b, t = t0 + tq + 8 * k;
    if (n < a.n_blocks && tq + 8 * k < nt) {
      const float sc = fmaxf(s_mean[k], a.beta * s_max[k]);
      scores[((long)h * a.sub_n + t) * a.n_blocks + n] = n > (a.start_pos + t) / a.bsn ? -INFINITY : sc;
    }
  }
}

// Selection, one workgroup per (kv head, query t).  The reference's repeated
// argmax (ties to the lower block, -inf and NaN never chosen, -1 padding)
// picks the first top_k blocks in the order (score descending, block
// ascending), and its list is then sorted ascending: it is that set.  It is
// found without sorting by a radix select on an order-preserving 32-bit key
// of the score (-0 and +0 equal):
//   1. four 8-bit passes narrow the key T of the top_k-th pick (a 256-bin
//      histogram of the keys that share the digits found so far, and a
//      suffix scan over the bins, by every wave for itself);
//   2. the picks are the blocks with key > T and the lowest-numbered `need`
//      blocks with key == T;
//   3. their places in the ascending list follow from the counts of the waves
//      before and ballots within the wave.
// A chain of latencies, not of work: the keys stay in registers (wave w holds
// blocks 64 KPT w ..; slot j of lane l is block 64 (KPT w + j) + l) and there are
// six barriers.  2,049 blocks, 64 rows: 5 us (256 threads with the keys in LDS
// and a scan through LDS in every pass: 14).
constexpr int kTkWaves = 16, kTkThreads = 64 * kTkWaves;

__device__ __forceinline__ uint32_t order_key(float v) {
  const uint32_t b = __float_as_uint(v == 0.0f ? 0.0f : v);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ bool pickable(float v) { return v > -INFINITY; }   // false for NaN
// key of a pickable score, 0 otherwise (every pickable score, > -inf and not
// NaN, has a key above 0x007FFFFF)
__device__ __forceinline__ uint32_t select_key(float v) { return pickable(v) ? order_key(v) : 0u; }

template <int CTRL, int MASK>
__device__ __forceinline__ int dpp_add(int v) {   // v + the lane CTRL names (0 if none)
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, MASK, 0xf, false);
}
__device__ __forceinline__ int wave_scan(int v) {   // inclusive
  v = dpp_add<0x111, 0xf>(v);   // row_shr:1, 2, 4, 8
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);   // row_bcast:15, :31
  return dpp_add<0x143, 0xc>(v);
}
__device__ __forceinline__ int lanes_below(uint64_t mask) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// KPT: keys per thread.  KPT 0: any number of blocks, the keys read from the
// workspace in every pass.
template <int KPT>
__global__ __launch_bounds__(kTkThreads) void block_select_kernel(BlockIndexArgs a, const float* scores) {
  __shared__ __attribute__((aligned(16))) int hist[4][256];
  __shared__ int wcnt[2][kTkWaves];
  const int h = blockIdx.x % a.num_kv, t = blockIdx.x / a.num_kv;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float* src = scores + ((long)h * a.sub_n + t) * a.n_blocks;
  int32_t* row = a.block_index + ((long)h * a.sub_n_max + t) * a.top_k;
  const int kpt = KPT ? KPT : (a.n_blocks + kTkThreads - 1) / kTkThreads;   // slots per thread
  const int base = 64 * kpt * wave + lane;
  uint32_t key[KPT ? KPT : 1];
  if constexpr (KPT) {
    float v[KPT];
#pragma unroll
    for (int j = 0; j < KPT; j++) v[j] = src[min(base + 64 * j, a.n_blocks - 1)];
#pragma unroll
    for (int j = 0; j < KPT; j++) key[j] = base + 64 * j < a.n_blocks ? select_key(v[j]) : 0u;
  }
  auto each = [&](auto f) {   // f(slot, key): every lane of the wave, slots in order
    if constexpr (KPT) {
#pragma unroll
      for (int j = 0; j < KPT; j++) f(j, key[j]);
    } else {
      for (int j = 0; j < kpt; j++) f(j, base + 64 * j < a.n_blocks ? select_key(src[base + 64 * j]) : 0u);
    }
  };
  static_assert(kTkThreads == 4 * 256, "one thread per bin of the four histograms");
  reinterpret_cast<int*>(hist)[tid] = 0;
  __syncthreads();
  uint32_t T = 0u, mask = 0u;   // the digits of the top_k-th pick's key found so far
  int need = a.top_k;           // its rank among the keys that share them
  bool all = false;             // no more pickable blocks than picks: every one is picked
#pragma unroll
  for (int pass = 0; pass < 4; pass++) {
    const int shift = 24 - 8 * pass;
    if (!all) {
      each([&](int, uint32_t k) {
        if (k != 0u && (k & mask) == T) atomicAdd(&hist[pass][(k >> shift) & 255u], 1);
      });
    }
    __syncthreads();
    if (!all) {
      // lane l: bins 255 - 4 l .. 252 - 4 l
      const int4 c = *reinterpret_cast<const int4*>(&hist[pass][252 - 4 * lane]);
      const int sum = (c.x + c.y) + (c.z + c.w), upto = wave_scan(sum);
      if (pass == 0 && __builtin_amdgcn_readlane(upto, 63) <= a.top_k) {
        all = true;
      } else {
        // the lane whose bins reach the rank: the first whose running count does
        const int l = (int)__builtin_ctzll(__builtin_amdgcn_ballot_w64(upto >= need));
        int left = need - __builtin_amdgcn_readlane(upto - sum, l), digit = 255 - 4 * l;
        const int cnt[4] = {__builtin_amdgcn_readlane(c.w, l), __builtin_amdgcn_readlane(c.z, l),
                            __builtin_amdgcn_readlane(c.y, l), __builtin_amdgcn_readlane(c.x, l)};
        bool there = false;
#pragma unroll
        for (int e = 0; e < 3; e++) {
          there = there || left <= cnt[e];
          left -= there ? 0 : cnt[e];
          digit -= there ? 0 : 1;
        }
        T |= (uint32_t)digit << shift;
        mask |= 255u << shift;
        need = left;
      }
    }
  }
  // picks: keys above T, and the first `need` of those equal to it, in block order
  auto above = [&](uint32_t k) { return all ? k != 0u : k > T; };
  auto equal = [&](uint32_t k) { return !all && k == T; };
  int n_gt = 0, n_eq = 0;
  each([&](int, uint32_t k) {
    n_gt += __builtin_popcountll(__builtin_amdgcn_ballot_w64(above(k)));
    n_eq += __builtin_popcountll(__builtin_amdgcn_ballot_w64(equal(k)));
  });
  if (lane == 0) {
    wcnt[0][wave] = n_gt;
    wcnt[1][wave] = n_eq;
  }
  __syncthreads();
  const int sg = wave_scan(lane < kTkWaves ? wcnt[0][lane & (kTkWaves - 1)] : 0);
  const int se = wave_scan(lane < kTkWaves ? wcnt[1][lane & (kTkWaves - 1)] : 0);
  int gt = __builtin_amdgcn_readlane(sg, wave) - n_gt, eq = __builtin_amdgcn_readlane(se, wave) - n_eq;
  each([&](int j, uint32_t k) {
    const uint64_t mg = __builtin_amdgcn_ballot_w64(above(k)), me = __builtin_amdgcn_ballot_w64(equal(k));
    const int eq_here = eq + lanes_below(me);   // equal keys of lower blocks
    if (above(k) || (equal(k) && eq_here < need)) row[gt + lanes_below(mg) + min(eq_here, need)] = base + 64 * j;
    gt += __builtin_popcountll(mg);
    eq += __builtin_popcountll(me);
  });
  const int n_total = __builtin_amdgcn_readlane(sg, 63) + min(__builtin_amdgcn_readlane(se, 63), need);
  for (int j = n_total + tid; j < a.top_k; j += kTkThreads) row[j] = -1;
}

hipError_t launch_tq3_kpool(const KpoolArgs& a, hipStream_t stream) {
  const int n_upd = a.cur_blocks - a.blk_lo;
  if (n_upd <= 0) return hipSuccess;
  hipLaunchKernelGGL(tq3_kpool_kernel, dim3((unsigned)(a.num_kv * n_upd)), dim3(kSpThreads), 0,
                     stream, a);
  return hipGetLastError();
}

hipError_t launch_block_index(const BlockIndexArgs& a, float* scores, hipStream_t stream) {
  const bool two = a.sub_n > 8;   // queries per thread
  const long n_wg = (long)a.num_kv * ((a.n_blocks + kScBlocks - 1) / kScBlocks) * ((a.sub_n + (two ? 15 : 7)) / (two ? 16 : 8));
  if (n_wg <= 0) return hipErrorInvalidValue;
  if (two)
    hipLaunchKernelGGL((block_score_kernel<2>), dim3((unsigned)n_wg), dim3(kSpThreads), 0, stream, a, scores);
  else
    hipLaunchKernelGGL((block_score_kernel<1>), dim3((unsigned)n_wg), dim3(kSpThreads), 0, stream, a, scores);
  const dim3 grid((unsigned)(a.num_kv * a.sub_n)), block(kTkThreads);
  const float* sc = scores;
  if (a.n_blocks <= 4 * kTkThreads)
    hipLaunchKernelGGL((block_select_kernel<4>), grid, block, 0, stream, a, sc);
  else if (a.n_blocks <= 16 * kTkThreads)
    hipLaunchKernelGGL((block_select_kernel<16>), grid, block, 0, stream, a, sc);
  else
    hipLaunchKernelGGL((block_select_kernel<0>), grid, block, 0, stream, a, sc);
  return hipGetLastError();
}

}  // namespace qkv
