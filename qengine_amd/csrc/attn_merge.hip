// attn_merge.hip -- log-sum-exp merge of split partials (reference layout).
//
// Reference: flash_attn_split_merge (attention.cuh:1837-1891): M = max over
// splits; splits with non-finite m or l <= 0 are skipped; out = sum w*o /
// sum w*l with w = exp(m_s - M), 0 when the sum is 0; fp16 output
// [t][q_head][256].  One workgroup per (q head, t), one thread per dim.
//
// record_merge_kernel is the same merge over the records of a decode launch.
#include <algorithm>
#include <type_traits>

#include "attn_common.h"
#include "attn_fastmerge.h"
#include "qkv_launch.h"
#include "qkv_device.h"

namespace qkv {

__global__ __launch_bounds__(256) void split_merge_kernel(const float* __restrict__ pm,
                                                          const float* __restrict__ pl,
                                                          const float* __restrict__ po,
                                                          uint16_t* __restrict__ out, int num_q,
                                                          int sub_n_max, int k_splits) {
  const int qh = blockIdx.x, t = blockIdx.y, d = threadIdx.x;
  const long base = ((long)qh * sub_n_max + t) * k_splits;
  // Splits eight at a time, the loads of a round all issued before the first is used
  // (past the last split they repeat it and are not counted), the first round's ahead
  // of the maximum: up to 8 splits are one memory round trip, not one per split.
  float ms[8], ls[8], os[8];
  auto load = [&](int s0) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const long at = base + min(s0 + i, k_splits - 1);
      ms[i] = pm[at];
      ls[i] = pl[at];
      os[i] = po[at * 256 + d];
    }
  };
  load(0);
  float M = -INFINITY;
#pragma unroll
  for (int i = 0; i < 8; i++) M = fmaxf(M, ms[i]);
  for (int s0 = 8; s0 < k_splits; s0 += 8)
#pragma unroll
    for (int i = 0; i < 8; i++) M = fmaxf(M, pm[base + min(s0 + i, k_splits - 1)]);
  float L = 0.f, o = 0.f;
  for (int s0 = 0; s0 < k_splits; s0 += 8) {
    if (s0) load(s0);
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if (s0 + i >= k_splits || !__builtin_isfinite(ms[i]) || ls[i] <= 0.0f) continue;
      const float w = __expf(ms[i] - M);
      L += w * ls[i];
      o += w * os[i];
    }
  }
  const float inv = L > 0.0f ? 1.0f / L : 0.0f;
  out[((long)t * num_q + qh) * 256 + d] = (uint16_t)f2h(o * inv);
}

hipError_t launch_split_merge(const float* m, const float* l, const float* o, uint16_t* out,
                              int num_q, int sub_n, int sub_n_max, int k_splits,
                              hipStream_t stream) {
  dim3 grid(num_q, sub_n);
  hipLaunchKernelGGL(split_merge_kernel, grid, dim3(256), 0, stream, m, l, o, out, num_q,
                     sub_n_max, k_splits);
  return hipGetLastError();
}

// Zero-fill by a kernel, so that a caller that captures the reset into a HIP
// graph records a kernel node rather than a memset node.
__global__ __launch_bounds__(256) void fill_zero_kernel(uint32_t* __restrict__ p, size_t n_words) {
  for (size_t i = blockIdx.x * 256ul + threadIdx.x; i < n_words; i += (size_t)gridDim.x * 256)
    p[i] = 0u;
}

hipError_t launch_fill_zero(void* p, size_t bytes, hipStream_t stream) {
  const size_t n = bytes / 4;
  const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
  hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks), dim3(256), 0, stream,
                     static_cast<uint32_t*>(p), n);
  return hipGetLastError();
}

// The health word of a fast-path workspace (header word kWsErrorWord) turned
// into a status and stored to `status` (device memory, or host memory the
// device can write) by one thread: ok_value while the word is 0, else
// timeout_value.  Stream-ordered, no host synchronization.
__global__ __launch_bounds__(64) void ws_status_kernel(const int* __restrict__ header, int* status,
                                                       int ok_value, int timeout_value) {
  if (threadIdx.x == 0) {
    const int w = __hip_atomic_load(header + kWsErrorWord, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *status = w == 0 ? ok_value : timeout_value;
  }
}

hipError_t launch_ws_status(const void* workspace, int* status, int ok_value, int timeout_value,
                            hipStream_t stream) {
  hipLaunchKernelGGL(ws_status_kernel, dim3(1), dim3(64), 0, stream, static_cast<const int*>(workspace),
                     status, ok_value, timeout_value);
  return hipGetLastError();
}

// The records of a decode launch, which precedes this one on the stream, to the output:
// one workgroup per (query, q head, 128-dim block) unit.  A launch of its own for calls
// whose units are many (merges_apart) and for attn_mq.hip: workgroups that wait for
// records in the launch that writes them hold the CUs that its other workgroups, or
// those of a launch on another stream, are still to run on.  The records are complete
// here, so their scalars and rows are loaded at once, one memory round trip; the
// arguments are scalars that arrive in registers with the wave (attn_common.h) and the
// unit comes from the three grid dimensions, without a division.
// A tag that is missing all the same (the workspace is in use by another call, or the
// poll limit is 0) is the timeout of the in-launch merges: NaN rows and the sticky error.
// Against the merge within attn_mq.hip's launch, us for the call, TQ3, 16 q heads:
// 8 queries over 301 keys 15.0 -> 13.0, 5 over 18,016 21.2 -> 20.0, 16 over 32,767
// 36.4 -> 36.4; Q8_0, 16 over 4,096 19.1 -> 18.4, 2 over 18,016 20.9 -> 21.8.
constexpr int kRecThreads = 256;

// Sum over the wave, in every lane (the steps of wave_sum, attn_common.h).
__device__ __forceinline__ int wave_sum_int(int v) {
  auto add = [&](auto ctrl, auto rows) {
    v += __builtin_amdgcn_update_dpp(0, v, decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
  };
  using std::integral_constant;
  add(integral_constant<int, 0xB1>{}, integral_constant<int, 0xf>{});    // quad_perm [1,0,3,2]
  add(integral_constant<int, 0x4E>{}, integral_constant<int, 0xf>{});    // quad_perm [2,3,0,1]
  add(integral_constant<int, 0x124>{}, integral_constant<int, 0xf>{});   // row_ror:4
  add(integral_constant<int, 0x128>{}, integral_constant<int, 0xf>{});   // row_ror:8
  add(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});   // row_bcast:15
  add(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});   // row_bcast:31
  return __builtin_amdgcn_readlane(v, 63);
}

// slot_shares (attn_fastmerge.h) by a wave: a slot per lane, one round of loads and of
// divisions instead of one per slot.
__device__ __forceinline__ void wave_slot_shares(const AttnArgs& p, int s, int& first, int& count) {
  const int lane = threadIdx.x & 63;
  long total = 0;
  for (int i0 = 0; i0 < p.sub_n; i0 += 64) {
    const int keys = i0 + lane < p.sub_n ? slot_keys(p, i0 + lane) : 0;
    total += ((long)wave_sum_int(keys >> 16) << 16) + wave_sum_int(keys & 0xffff);
  }
  first = count = 0;
  for (int i0 = 0; i0 <= s; i0 += 64) {
    const int w = i0 + lane <= s ? share_count(p, i0 + lane, total) : 0;
    first += wave_sum_int(i0 + lane < s ? w : 0);
    if (s - i0 < 64) count = __builtin_amdgcn_readlane(w, s - i0);
  }
}

template <bool ROTATE, bool RAGGED>
__global__ __launch_bounds__(kRecThreads) void record_merge_kernel(float* ws_ml, float* ws_o, int* ws_header,
                                                                   uint16_t* out, uint32_t ws_ml_bytes,
                                                                   uint32_t ws_o_bytes, int num_q, int sub_n,
                                                                   int n_chunks, int spin_limit,
                                                                   const int32_t* ctx_lens, int ctx_max) {
  using ML = MergeLayout<kRecThreads>;
  __shared__ __attribute__((aligned(16))) float red[ML::kRedFloats];
  __shared__ f2_t mls[128];
  AttnArgs p{};
  p.num_q = num_q;
  p.sub_n = sub_n;
  p.n_slots = p.n_chunks = n_chunks;
  const int tid = threadIdx.x;
  const int t = blockIdx.x, qh = blockIdx.y, blk = blockIdx.z;
  long base = rec_index(p, qh, t, 0);
  int n = n_chunks;
  if constexpr (RAGGED) {   // the slot's shares of the kv head's records
    p.ctx_lens = ctx_lens;
    p.ctx_max = ctx_max;
    int first;
    wave_slot_shares(p, t, first, n);
    base = rec_index(p, qh, 0, first);
  }
  const __amdgpu_buffer_rsrc_t rml = __builtin_amdgcn_make_buffer_rsrc(ws_ml, 0, ws_ml_bytes, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(ws_o, 0, ws_o_bytes, kBufferRsrcWord3);
  const bool poisoned = __hip_atomic_load(ws_header + kWsErrorWord, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  f4_t r = {0.f, 0.f, 0.f, 0.f};
  if (tid < n)
    r = __builtin_amdgcn_raw_buffer_load_b128(rml, (uint32_t)((base + tid) * kRecMlBytes), 0, kCoherent);
  f4_t v[ML::kRecPerThread];
#pragma unroll
  for (int i = 0; i < ML::kRecPerThread; i++) {
    const int c = (tid >> 5) + ML::kSlices * i;
    v[i] = c < n ? __builtin_amdgcn_raw_buffer_load_b128(
                       ro, (uint32_t)(((base + c) * 256 + blk * 128 + 4 * (tid & 31)) * 4), 0, kCoherent)
                 : f4_t{0.f, 0.f, 0.f, 0.f};
  }
  if (poisoned) {   // (uniform) left inconsistent by an earlier timeout: NaN rows until it is reset
    write_nan_unit(p, t, qh, blk, out);
    return;
  }
  const bool seen = tid < n && spin_limit > 0 && __float_as_uint(blk ? r[3] : r[2]) == kTagValid;
  if (tid < n) mls[tid] = f2_t{r[0], r[1]};
  if (seen)   // clear: the state that the next launch on this workspace starts from
    __builtin_amdgcn_raw_buffer_store_b32(0u, rml, (uint32_t)((base + tid) * kRecMlBytes + 8 + 4 * blk), 0,
                                          kCoherent);
  if (!block_and<kRecThreads>(seen || tid >= n, reinterpret_cast<int*>(red + ML::kVote))) {
    write_nan_unit(p, t, qh, blk, out);
    if (tid == 0)
      __hip_atomic_store(ws_header + kWsErrorWord, kWsErrorTimeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  fold_unit<kRecThreads, ROTATE>(red, mls, p, v, n, qh, t, blk, out);
}

hipError_t launch_record_merge(const AttnArgs& a, bool rotate, uint16_t* out, hipStream_t stream) {
  const dim3 grid(a.sub_n, a.num_q, 2), block(kRecThreads);
  auto* kernel = a.ctx_lens ? record_merge_kernel<true, true>   // (paged caches are TQ3)
                 : rotate   ? record_merge_kernel<true, false>
                            : record_merge_kernel<false, false>;
  hipLaunchKernelGGL(kernel, grid, block, 0, stream, a.ws_ml, a.ws_o, a.ws_header, out, a.ws_ml_bytes, a.ws_o_bytes,
                     a.num_q, a.sub_n, a.n_chunks, a.spin_limit, a.ctx_lens, a.ctx_max);
  return hipGetLastError();
}

}  // namespace qkv
