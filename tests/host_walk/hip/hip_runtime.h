// The few HIP names csrc/ct_internal.h and ct_device.h use, for a host build.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>
#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define CT_RCP(x) (1.0f / (x))
struct float2 { float x, y; };
struct float4 { float x, y, z, w; };
struct uint2 { uint32_t x, y; };
struct uint4 { uint32_t x, y, z, w; };
inline float4 make_float4(float a, float b, float c, float d) { return {a, b, c, d}; }
inline uint2 make_uint2(uint32_t a, uint32_t b) { return {a, b}; }
inline uint4 make_uint4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) { return {a, b, c, d}; }
inline uint32_t __float_as_uint(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }
inline float __uint_as_float(uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }
inline uint32_t min(uint32_t a, uint32_t b) { return a < b ? a : b; }
#define __builtin_amdgcn_ballot_w64(b) ((b) ? 1ull : 0ull)  // a wave of one lane
inline float __builtin_amdgcn_fmed3f(float a, float b, float c) { return std::fmax(std::fmin(a, b), std::fmin(std::fmax(a, b), c)); }
inline float __builtin_amdgcn_fractf(float x) { return std::fmin(x - std::floor(x), 0.99999994f); }
inline int __popcll(uint64_t v) { return __builtin_popcountll(v); }
inline int __ffs(int v) { return __builtin_ffs(v); }
using std::isnan;
typedef void *hipStream_t, *hipEvent_t;
typedef int hipError_t;
constexpr int hipSuccess = 0, hipHostMallocDefault = 0;
inline hipError_t hip_last_error = hipSuccess;  // hipMalloc refuses every request
inline hipError_t hipMalloc(void **, size_t) { return hip_last_error = 2; }
inline hipError_t hipGetLastError() {
  const hipError_t e = hip_last_error;
  hip_last_error = hipSuccess;
  return e;
}
inline hipError_t hipFree(void *) { return 0; }
inline hipError_t hipHostMalloc(void **, size_t, int) { return 1; }
inline hipError_t hipHostFree(void *) { return 0; }
inline const char *hipGetErrorString(hipError_t) { return ""; }
