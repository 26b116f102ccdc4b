// Requantisers: float voltages -> the packed station layouts the F-stage
// reads.  gpubench packs filterbank output to 2 bits on the GPU
// (examples/chris/bench/gpubench.cu:64-130); here the codes are fxkernel's
// (the LUT of fxkernel/src/fxkernel.cpp:15-28 decodes 0,1,2,3 to -HI,-1,+1,+HI):
//   x < -t -> 0,  -t <= x < 0 -> 1,  0 <= x < t -> 2,  x >= t -> 3  (NaN -> 1),
// packed LSB first [A_t, B_t, A_t+1, B_t+1]; and complex 8-bit
//   q = clamp(rint(x * scale), -127, 127) (NaN -> 0), bytes [Are, Aim, Bre, Bim].
// Both are bound by the reading of the floats: neighbouring lanes take
// neighbouring 16 bytes of either polarisation and store 2 or 8 bytes; 1e8
// samples to 2 bits 193 -> 140 us (6.1 TB/s) against 16 samples of one lane in
// four loads of 64-byte stride.  Two such loads in flight per lane and
// polarisation (four: 144 us, eight: 146), nontemporal (otherwise 157).
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include "gxc_requant.hpp"

namespace gxc {
namespace {

__device__ __forceinline__ unsigned code2(float x, float t) {
  unsigned c = 1u;
  if (x >= 0.f) c = 2u;
  if (x >= t) c = 3u;
  if (x < -t) c = 0u;
  return c;
}

__device__ __forceinline__ unsigned q8(float x, float scale) {
  const float y = rintf(x * scale);
  const float z = isnan(y) ? 0.f : fminf(fmaxf(y, -127.f), 127.f);
  return (unsigned)(int)z & 0xffu;
}

typedef float floatx4 __attribute__((ext_vector_type(4)));
// four floats that nothing reads again
__device__ __forceinline__ floatx4 load4(const float *p) {
  return __builtin_nontemporal_load(reinterpret_cast<const floatx4 *>(p));
}

constexpr int kGroups = 2;                // 16-byte loads per lane and polarisation
constexpr int kBlock2 = 256 * 4 * kGroups;  // time samples of a workgroup, 2-bit
constexpr int kBlock8 = 256 * 2 * kGroups;  // and complex 8-bit

// Group k of a lane: 4 time samples, bytes [s / 2, s / 2 + 2) of the output.
__global__ void __launch_bounds__(256) requant2_kernel(const float *__restrict__ a, const float *__restrict__ b,
                                                       long long n, float t, uint8_t *__restrict__ out) {
  const long long s0 = (long long)blockIdx.x * kBlock2 + 4 * threadIdx.x;
  auto pack = [&](const floatx4 &u, const floatx4 &v) {
    unsigned w = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) w |= (code2(u[i], t) | code2(v[i], t) << 2) << (4 * i);
    return (uint16_t)w;
  };
  if ((long long)(blockIdx.x + 1) * kBlock2 <= n) {
    floatx4 u[kGroups], v[kGroups];
#pragma unroll
    for (int k = 0; k < kGroups; k++) u[k] = load4(a + s0 + 1024 * k), v[k] = load4(b + s0 + 1024 * k);
#pragma unroll
    for (int k = 0; k < kGroups; k++) *reinterpret_cast<uint16_t *>(out + ((s0 + 1024 * k) >> 1)) = pack(u[k], v[k]);
  } else {  // the last workgroup: n is even, one byte per two samples
    for (int k = 0; k < kGroups; k++)
      for (long long s = s0 + 1024 * k; s < n && s < s0 + 1024 * k + 4; s += 2)
        out[s >> 1] = (uint8_t)(code2(a[s], t) | code2(b[s], t) << 2 | code2(a[s + 1], t) << 4 | code2(b[s + 1], t) << 6);
  }
}

// Group k of a lane: 2 complex time samples, bytes [4 s, 4 s + 8) of the output.
__global__ void __launch_bounds__(256) requant8_kernel(const float *__restrict__ a, const float *__restrict__ b,
                                                       long long n, float scale, uint8_t *__restrict__ out) {
  const long long s0 = (long long)blockIdx.x * kBlock8 + 2 * threadIdx.x;
  if ((long long)(blockIdx.x + 1) * kBlock8 <= n) {
    floatx4 u[kGroups], v[kGroups];
#pragma unroll
    for (int k = 0; k < kGroups; k++) u[k] = load4(a + 2 * (s0 + 512 * k)), v[k] = load4(b + 2 * (s0 + 512 * k));
#pragma unroll
    for (int k = 0; k < kGroups; k++)
      *reinterpret_cast<uint2 *>(out + 4 * (s0 + 512 * k)) = make_uint2(
          q8(u[k].x, scale) | q8(u[k].y, scale) << 8 | q8(v[k].x, scale) << 16 | q8(v[k].y, scale) << 24,
          q8(u[k].z, scale) | q8(u[k].w, scale) << 8 | q8(v[k].z, scale) << 16 | q8(v[k].w, scale) << 24);
  } else {
    for (int k = 0; k < kGroups; k++)
      for (long long s = s0 + 512 * k; s < n && s < s0 + 512 * k + 2; s++)
        *reinterpret_cast<unsigned *>(out + 4 * s) = q8(a[2 * s], scale) | q8(a[2 * s + 1], scale) << 8 |
                                                     q8(b[2 * s], scale) << 16 | q8(b[2 * s + 1], scale) << 24;
  }
}

}  // namespace

// (in pieces: a grid has fewer than 2^32 work items, 8 samples each)
hipError_t launch_requant2(const float *a, const float *b, long long n, float t, uint8_t *out, hipStream_t s) {
  constexpr long long kMost = 1LL << 34;
  for (long long at = 0; at < n; at += kMost) {
    const long long m = n - at < kMost ? n - at : kMost;
    hipLaunchKernelGGL(requant2_kernel, dim3((unsigned)((m + kBlock2 - 1) / kBlock2)), dim3(256), 0, s, a + at, b + at,
                       m, t, out + at / 2);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_requant8(const float *a, const float *b, long long n, float scale, uint8_t *out, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(requant8_kernel, dim3((unsigned)((n + kBlock8 - 1) / kBlock8)), dim3(256), 0, s, a, b, n, scale, out);
  return hipGetLastError();
}

}  // namespace gxc
