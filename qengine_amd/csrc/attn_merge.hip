// attn_merge.hip -- log-sum-exp merge of split partials (reference layout).
//
// Reference: flash_attn_split_merge (attention.cuh:1837-1891): M = max over
// splits; splits with non-finite m or l <= 0 are skipped; out = sum w*o /
// sum w*l with w = exp(m_s - M), 0 when the sum is 0; fp16 output
// [t][q_head][256].  One workgroup per (q head, t), one thread per dim.
#include <algorithm>

#include "attn_common.h"
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

}  // namespace qkv
