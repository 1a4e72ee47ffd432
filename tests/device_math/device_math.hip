// q3_device.h's scalar functions over runs of float bit patterns, for
// tests/test_gpu_device_math.py (built by qwen3-tile-ops_amd/build.py).
#include "q3_device.h"

namespace {

// out[i] = rcp_ge1 of the float with bits first + i
__global__ void rcp_kernel(uint32_t first, uint32_t n, float *out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = q3::rcp_ge1(q3::bits_f32(first + i));
}

// floats in [-151, 200] with bits first .. first + n - 1: how many, and on how
// many exp2f_fast differs from exp2f_glibc
__global__ void exp2_kernel(uint32_t first, uint32_t n, unsigned long long *count) {
  __shared__ uint64_t tab[32];
  if (threadIdx.x == 0) q3::stage_exp2_table(tab);
  __syncthreads();
  unsigned long long seen = 0, bad = 0;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
    const float x = q3::bits_f32(first + static_cast<uint32_t>(i));
    if (!(x >= -151.0f && x <= 200.0f)) continue;
    ++seen;
    bad += q3::f32_bits(q3::exp2f_fast(x, tab)) != q3::f32_bits(q3::exp2f_glibc(x));
  }
  atomicAdd(count, seen);
  atomicAdd(count + 1, bad);
}

}  // namespace

extern "C" int device_math_rcp_ge1(uint32_t first, uint32_t n, float *out, void *stream) {
  if (n == 0 || n > (1u << 24) || !out) return 1;
  hipLaunchKernelGGL(rcp_kernel, dim3((n + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream), first, n, out);
  return hipGetLastError() != hipSuccess;
}

extern "C" int device_math_exp2_mismatches(uint32_t first, uint32_t n, unsigned long long *count, void *stream) {
  if (n == 0 || !count) return 1;
  hipLaunchKernelGGL(exp2_kernel, dim3(2048), dim3(256), 0, static_cast<hipStream_t>(stream), first, n, count);
  return hipGetLastError() != hipSuccess;
}
