// Copies between device memory and the caller's host memory.
#pragma once

#include "tensor.hpp"

namespace cc4s_amd {

// A transfer of at least kStagedBytes from or to pageable memory goes through a ring
// of pinned chunks (pinned memory is copied by the link itself): the DMA of one
// chunk runs while threads of this call copy another between the ring and the
// caller's memory.  The runtime's own pageable path copies with one thread, which
// also takes the page faults of a freshly allocated result: 8.5 GB/s measured,
// against 55 GB/s of the link.  Measured with the ring (4 chunks of 4 MiB, 8
// threads), one pass and its amplitudes: complex No=32, Nv=256 (1.1 GB) 541 -> 466
// ms, No=17, Nv=131 (79 MB) 21.8 -> 15.5 ms, real Drccd No=24, Nv=160 (118 MB) 16.5
// -> 8.0 ms; smaller transfers take under 2 ms either way and keep the runtime's
// path, and so does a call that gets no pinned memory or no thread.  The ring
// belongs to one context, is made on its first large transfer and freed with it.
// The data has arrived, and the caller's memory been read, when the stream has been
// waited for.
class HostTransfer {
 public:
  HostTransfer() = default;
  ~HostTransfer();
  HostTransfer(const HostTransfer &) = delete;
  HostTransfer &operator=(const HostTransfer &) = delete;
  void download(void *host, const void *device, size_t bytes, hipStream_t s);
  void upload(void *device, const void *host, size_t bytes, hipStream_t s);

 private:
  static constexpr size_t kStagedBytes = size_t(16) << 20;
  static constexpr size_t kChunk = size_t(4) << 20;
  static constexpr int kRing = 4;
  bool ring();  // false: no pinned memory, use the runtime's path
  HostBuffer buf_[kRing];
  hipEvent_t event_[kRing] = {};
  bool tried_ = false, ready_ = false;
};

}  // namespace cc4s_amd
