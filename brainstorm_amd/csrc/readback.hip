// A few words from the device to a host that waits for them.
//
// The reference reads loads with `.sum().item()` (src/backend/torch/router.cc:197-201): a copy and a wait for the
// stream.  Both cost more than the words: the copy is a launch of the runtime's, and the wait ends when the runtime has
// seen the launch's completion signal.  Here one small kernel stores the words into host memory and a last one behind
// them, which the host watches.  Bound by latency alone (one read of the words, one write across the link): behind
// a kernel of 5 us the host has them 12.9 us after it started to launch, 17.9 us with copy and wait.
#include "common.hpp"

namespace brt {
namespace {

__global__ __launch_bounds__(256) void copy_to_host_kernel(const int* __restrict__ src, int* host, int words) {
  for (int i = threadIdx.x; i < words; i += blockDim.x) host[i] = src[i];
  __threadfence_system();  // every wavefront's words are on their way before ...
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(host + words, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);  // ... this one
}

}  // namespace
}  // namespace brt

using namespace brt;

extern "C" int brt_hip_copy_to_host(const int32_t* src, int32_t* host, int words, void* stream) {
  if (words <= 0) return fail(BRT_E_INVALID, "no words to copy (%d)", words);
  if (!src || !host) return fail(BRT_E_INVALID, "null argument");
  if (!aligned(src, 4) || !aligned(host, 4)) return fail(BRT_E_INVALID, "src/host must be 4-byte aligned");
  hipLaunchKernelGGL(copy_to_host_kernel, dim3(1), dim3(words <= kWave ? kWave : 256), 0, as_stream(stream), src, host, words);
  return check_launch("copy_to_host_kernel");
}
