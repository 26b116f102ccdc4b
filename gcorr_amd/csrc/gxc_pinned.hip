#include "gxc_pinned.hpp"

#include <algorithm>
#include <cstring>

namespace gxc {
namespace {

// n units of 16 bytes; either side may be pinned host memory.
__global__ void __launch_bounds__(256) copy_kernel(uint4 *__restrict__ dst, const uint4 *__restrict__ src, size_t n) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) dst[i] = src[i];
}

hipError_t launch_copy(void *dst, const void *src, size_t bytes, hipStream_t s) {
  const size_t n = bytes / 16;
  hipLaunchKernelGGL(copy_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 256)), dim3(256), 0, s,
                     static_cast<uint4 *>(dst), static_cast<const uint4 *>(src), n);
  return hipGetLastError();
}

constexpr size_t kChunk = 512 << 10;
size_t round16(size_t n) { return (n + 15) / 16 * 16; }

}  // namespace

namespace host {

hipError_t Mailbox::create(size_t in_bytes, size_t out_bytes, size_t spare_bytes) {
  in = round16(in_bytes);
  const size_t n = (in + out_bytes + 4095) / 4096 * 4096;  // spare: whole pages
  hipError_t e = hipHostMalloc((void **)&h, n + spare_bytes, hipHostMallocDefault);
  if (e != hipSuccess) return e;
  std::memset(h, 0, n);
  spare = h + n;
  if ((e = hipMalloc((void **)&d, in)) != hipSuccess) return e;
  dirty = true;
  return hipSuccess;
}

hipError_t Mailbox::flush(hipStream_t s) {
  if (!dirty) return hipSuccess;
  const hipError_t e = launch_copy(d, h, in, s);
  dirty = e != hipSuccess;
  return e;
}

void Mailbox::release() {
  if (h) hipHostFree(h);
  hipFree(d);
  h = d = spare = nullptr;
}

size_t HostOut::bytes(size_t largest) { return largest > kChunk ? 2 * kChunk : round16(largest); }

hipError_t HostOut::create(unsigned char *pinned, size_t largest) {
  buf_ = pinned;
  chunk_ = std::min(round16(std::max<size_t>(largest, 1)), kChunk);
  hipError_t e = hipSuccess;
  for (hipEvent_t &ev : ev_)
    if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
  return e;
}

hipError_t HostOut::copy(void *dst, const void *src, size_t n, hipStream_t s) {
  // pinned or device memory takes the copy directly
  hipPointerAttribute_t at{};
  const bool pageable = hipPointerGetAttributes(&at, dst) != hipSuccess || at.type == hipMemoryTypeUnregistered;
  if (!pageable || n % 16 || !buf_) {
    const hipError_t e = hipStreamSynchronize(s);
    return e != hipSuccess ? e : hipMemcpy(dst, src, n, hipMemcpyDeviceToHost);
  }
  (void)hipGetLastError();  // of the query
  std::lock_guard<std::mutex> lock(mu_);
  auto fill = [&](size_t at0, int b) {
    const hipError_t e = launch_copy(buf_ + b * chunk_, static_cast<const unsigned char *>(src) + at0,
                                     std::min(chunk_, n - at0), s);
    return e != hipSuccess ? e : hipEventRecord(ev_[b], s);
  };
  hipError_t e = hipSuccess;
  int b = 0;
  if (n > 0) e = fill(0, 0);
  for (size_t at0 = 0; at0 < n && e == hipSuccess; at0 += chunk_, b ^= 1) {
    if (at0 + chunk_ < n) e = fill(at0 + chunk_, b ^ 1);
    if (e == hipSuccess) e = hipEventSynchronize(ev_[b]);
    if (e == hipSuccess)
      std::memcpy(static_cast<unsigned char *>(dst) + at0, buf_ + b * chunk_, std::min(chunk_, n - at0));
  }
  if (e != hipSuccess) (void)hipStreamSynchronize(s);  // no fill outlives the lock
  return e;
}

void HostOut::release() {
  for (hipEvent_t &ev : ev_)
    if (ev) hipEventDestroy(ev);
  buf_ = nullptr;
  ev_[0] = ev_[1] = nullptr;
}

}  // namespace host
}  // namespace gxc
