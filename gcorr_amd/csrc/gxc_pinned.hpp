// Host memory that the device reads and writes by itself, for the small
// transfers around a subintegration: a blocking hipMemcpy of a few hundred
// bytes takes 12-15 us, as long as a small array's F-stage, and a pass has four
// (pointers, delays, counts, visibilities).  With both classes and delay rows
// passed by address: 3 stations x 256 channels x 64 FFTs 112 -> 69 us, 4 x 128 x
// 12500 164 -> 117 us, a batch of 8 subbands 10.31 -> 10.02 ms.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>

namespace gxc {
namespace host {

// A pinned block: its first `in` bytes are parameters that the host writes and
// flush() copies to the device mirror, the `out` bytes after them results that
// kernels write, the rest spare.  The host writes parameters only while no flush
// is queued (after a synchronisation of the stream), then sets dirty.  One block
// per handle, since a pinned allocation takes 11 us, whatever its size, and
// its release 12: creating and destroying a handle of 3 stations x 256 channels
// takes 232 us with two blocks, 210 with one, 180 with none.
struct Mailbox {
  unsigned char *h = nullptr, *d = nullptr;
  size_t in = 0;
  bool dirty = false;
  unsigned char *spare = nullptr;
  hipError_t create(size_t in_bytes, size_t out_bytes, size_t spare_bytes);
  hipError_t flush(hipStream_t s);
  void release();
};

// Device-to-host copies into pageable memory through two pinned chunks: the
// device fills one while the host empties the other (the runtime's own staging
// fills and empties in turn).  Visibilities of any size take them: the runtime's
// copy -> this, into memory written before: 0.05 MB 28 -> 15 us, 0.33 MB (one
// chunk, in turn here too) 23 -> 25, 3.6 MB 204 -> 131, 18 MB 1.04 -> 0.59 ms, 71 MB
// 4.06 -> 3.64, 277 MB 15.7 -> 15.0; into fresh pages 277 MB 27 -> 20.
class HostOut {
 public:
  static size_t bytes(size_t largest);  // of pinned memory for copies up to `largest` bytes
  hipError_t create(unsigned char *pinned, size_t largest);
  // Waits for the stream; dst may be any host memory.
  hipError_t copy(void *dst, const void *src, size_t n, hipStream_t s);
  void release();

 private:
  std::mutex mu_;  // callers may read results from several threads
  unsigned char *buf_ = nullptr;
  size_t chunk_ = 0;
  hipEvent_t ev_[2] = {nullptr, nullptr};
};

}  // namespace host
}  // namespace gxc
