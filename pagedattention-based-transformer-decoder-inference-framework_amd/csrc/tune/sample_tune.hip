// Tuning build only: exp_below against expf over bit patterns (tests).
#include "../exp_below.hpp"

namespace llm {

__global__ __launch_bounds__(256) void exp_below_kernel(uint32_t first, uint32_t* differ) {
  const uint32_t bits = first + blockIdx.x * 256 + threadIdx.x;
  const float x = __uint_as_float(bits), a = exp_below(x), b = expf(x);
  const bool same = __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b);
  if (!same && atomicAdd(differ, 1u) == 0) differ[1] = bits;
}

}  // namespace llm

// differ (device, 0 before): how many of the patterns [first, first + 256 blocks) differ, one of them.
extern "C" int exp_below_differs(uint32_t first, unsigned blocks, uint32_t* differ, void* stream) {
  if (blocks == 0) return 0;
  hipLaunchKernelGGL(llm::exp_below_kernel, dim3(blocks), dim3(256), 0, static_cast<hipStream_t>(stream), first, differ);
  return hipGetLastError() == hipSuccess ? 0 : 1;
}
