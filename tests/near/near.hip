// Goes through every float of fx_near.hpp's range, and the floats beside its
// ends, and counts those where near_sqrt or near_rcp differ from sqrtf and
// the division; prints one JSON line.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "fx_near.hpp"

__global__ void check(unsigned first, unsigned count, unsigned long long* out) {
  const unsigned stride = gridDim.x * blockDim.x;
  unsigned long long inside = 0, bad_sqrt = 0, bad_rcp = 0;
  for (unsigned long long k = blockIdx.x * blockDim.x + threadIdx.x; k < count; k += stride) {
    const float x = __uint_as_float(first + (unsigned)k);
    if (near_bits(x) >= FX_NEAR_SPAN) continue;
    inside++;
    if (__float_as_uint(near_sqrt(x)) != __float_as_uint(sqrtf(x))) bad_sqrt++;
    if (__float_as_uint(near_rcp(x)) != __float_as_uint(1.0f / x)) bad_rcp++;
  }
  atomicAdd(&out[0], inside);
  atomicAdd(&out[1], bad_sqrt);
  atomicAdd(&out[2], bad_rcp);
}

int main() {
  unsigned long long* d = nullptr;
  unsigned long long h[3] = {0, 0, 0};
  if (hipMalloc(reinterpret_cast<void**>(&d), sizeof(h)) != hipSuccess ||
      hipMemcpy(d, h, sizeof(h), hipMemcpyHostToDevice) != hipSuccess)
    return 1;
  hipLaunchKernelGGL(check, dim3(4096), dim3(256), 0, 0, 0u, 0xffffffffu, d);  // every bit pattern but the last NaN
  if (hipDeviceSynchronize() != hipSuccess || hipMemcpy(h, d, sizeof(h), hipMemcpyDeviceToHost) != hipSuccess) return 1;
  (void)hipFree(d);
  printf("{\"inside\": %llu, \"bad_sqrt\": %llu, \"bad_rcp\": %llu}\n", h[0], h[1], h[2]);
  return 0;
}
