// gvv_calib.hip -- measurement support: the float-atomic throughput of this GPU, against which
// the rasterizer's atomic rate is quoted (include/gvv_renderer.h, gvv_calibrate_atomics), and the
// device check of the correctly rounded operations of gvv_math.hpp (gvv_check_rounding).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "../../include/gvv_renderer.h"
#include "gvv_math.hpp"

namespace gvv {
int set_last_error(const std::string& m);
}

namespace {

__device__ __forceinline__ uint32_t mix(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  x ^= x >> 16;
  return x;
}

// Each thread issues `per_thread` atomicAdd(+1) into buf[0, n): scattered (hashed) addresses,
// or streaming ones where consecutive lanes hit consecutive floats.
__global__ void __launch_bounds__(256) k_atomic_rate(float* __restrict__ buf, uint32_t n, uint32_t per_thread,
                                                     int scattered) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t i = 0; i < per_thread; ++i) {
    const uint32_t a = scattered ? mix(t * per_thread + i) % n : (t + i * stride) % n;
    atomicAdd(buf + a, 1.0f);
  }
}

__device__ __forceinline__ bool same(float a, float b) {
  return __float_as_uint(a) == __float_as_uint(b) || (a != a && b != b);
}

// Each bit pattern x of [first, first + count): the operations of gvv_math.hpp on it against the IEEE
// operations, mismatches counted per operation.
__global__ void __launch_bounds__(256) k_check_rounding(uint64_t first, uint64_t count, unsigned long long* bad) {
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < count; i += stride) {
    const uint32_t bits = (uint32_t)(first + i);
    const float x = __uint_as_float(bits), a = __uint_as_float(mix(bits ^ 0x9e3779b9u));
    if (!same(gvv::rcp_rn(x), 1.0f / x)) atomicAdd(bad + 0, 1ull);
    if (!same(gvv::sqrt_rn(x), sqrtf(x))) atomicAdd(bad + 1, 1ull);
    // any numerator, and one whose quotient is near 1 (the significands' full range of carries)
    const float n = __uint_as_float((bits & 0xff800000u) | (mix(bits) & 0x007fffffu));
    const double r = gvv::recip64(x);
    if (!same(gvv::quot(a, x, r), a / x)) atomicAdd(bad + 2, 1ull);
    if (!same(gvv::quot(n, x, r), n / x)) atomicAdd(bad + 2, 1ull);
    // the saturating conversion
    const int32_t t = !(x == x) ? 0 : x >= 2147483648.0f ? INT32_MAX : x <= -2147483648.0f ? INT32_MIN : (int32_t)x;
    if (gvv::sat_i32(x) != t) atomicAdd(bad + 3, 1ull);
    // depth keys of an inside hit: barycentrics spread over magnitudes, depths from the projection's clamp on
    const float s = __uint_as_float(mix(bits) & 0x3fffffffu), u = fminf(s, 1.0f), v = (1.0f - u) * (mix(bits + 1) * 0x1p-32f);
    const float z0 = fmaxf(fabsf(x), 1e-7f), z1 = fmaxf(fabsf(a), 1e-7f), z2 = 1000.f + 1e-3f * (float)(mix(bits + 2) >> 8);
    const gvv::V3 abc = gvv::v3(u, v, 1.f - u - v);
    if (gvv::depth_key(abc, gvv::depth_recip(z0, z1, z2)) != gvv::depth_key(abc, z0, z1, z2)) atomicAdd(bad + 4, 1ull);
  }
}

}  // namespace

extern "C" int gvv_check_rounding(uint64_t first, uint64_t count, uint64_t* mismatches, void* stream) {
  if (!mismatches || count == 0 || first > UINT32_MAX || count > (1ull << 32) - first)
    return gvv::set_last_error("check rounding: need a device buffer of 5 counters and bit patterns within 2^32");
  hipLaunchKernelGGL(k_check_rounding, dim3(8192), dim3(256), 0, (hipStream_t)stream, first, count,
                     reinterpret_cast<unsigned long long*>(mismatches));
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gvv::set_last_error(std::string("check rounding: ") + hipGetErrorString(e));
  return 0;
}

extern "C" int gvv_calibrate_atomics(float* buf, int64_t n_floats, int64_t updates, int32_t scattered, void* stream) {
  if (!buf || n_floats <= 0 || n_floats > (int64_t)UINT32_MAX || updates <= 0)
    return gvv::set_last_error("calibrate atomics: need a buffer of 1 .. 2^32-1 floats and updates > 0");
  const uint32_t threads = 1u << 20;
  const uint32_t per = (uint32_t)((updates + threads - 1) / threads);
  hipLaunchKernelGGL(k_atomic_rate, dim3(threads / 256), dim3(256), 0, (hipStream_t)stream, buf, (uint32_t)n_floats,
                     per, scattered ? 1 : 0);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gvv::set_last_error(std::string("calibrate atomics: ") + hipGetErrorString(e));
  return 0;
}
