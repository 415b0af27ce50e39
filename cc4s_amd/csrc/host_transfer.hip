// Pinned-ring copies.  Bound by the host side: every byte is written once by a
// copying thread, on a fresh result behind a page fault.
#include "host_transfer.hpp"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace cc4s_amd {

namespace {

// Worker threads that copy their slice of chunk 0, 1, ... n-1 as the chunks are
// opened, and count it done.  As many as the system grants: the slices are those of
// the threads there are, which is settled before the first chunk is opened.  The
// destructor ends and joins them.
class Copiers {
 public:
  Copiers(size_t n, std::function<void(size_t chunk, int slice, int slices)> copy)
      : n_(n), copy_(std::move(copy)), done_(n, 0) {
    const unsigned hw = std::thread::hardware_concurrency();
    const int want = static_cast<int>(std::min(8u, std::max(1u, hw / 2)));
    threads_.reserve(want);
    try {
      while (count_ < want) {
        threads_.emplace_back([this, t = count_] { work(t); });
        ++count_;
      }
    } catch (const std::system_error &) {  // no more of them
    } catch (...) {
      end();
      throw;
    }
  }
  int count() const { return count_; }
  ~Copiers() { end(); }
  // chunks [0, upto) may be copied
  void open(size_t upto) {
    {
      std::lock_guard<std::mutex> l(m_);
      open_ = std::max(open_, upto);
    }
    opened_.notify_all();
  }
  void wait(size_t chunk) {
    std::unique_lock<std::mutex> l(m_);
    finished_.wait(l, [&] { return done_[chunk] == count_; });
  }

 private:
  void work(int t) {
    for (size_t c = 0; c < n_; ++c) {
      {
        std::unique_lock<std::mutex> l(m_);
        opened_.wait(l, [&] { return open_ > c || end_; });
        if (open_ <= c) return;
      }
      copy_(c, t, count_);
      bool last;
      {
        std::lock_guard<std::mutex> l(m_);
        last = ++done_[c] == count_;
      }
      if (last) finished_.notify_one();
    }
  }
  void end() {
    {
      std::lock_guard<std::mutex> l(m_);
      end_ = true;
    }
    opened_.notify_all();
    for (auto &t : threads_)
      if (t.joinable()) t.join();
    threads_.clear();
  }
  size_t n_;
  std::function<void(size_t, int, int)> copy_;
  std::vector<int> done_;
  int count_ = 0;  // workers read it after the first chunk was opened
  size_t open_ = 0;
  bool end_ = false;
  std::mutex m_;
  std::condition_variable opened_, finished_;
  std::vector<std::thread> threads_;
};

// [begin, end) of a slice of `bytes`, on 4 KiB boundaries so that no two
// threads fault the same page of an aligned destination
void slice_of(size_t bytes, int slice, int slices, size_t &begin, size_t &end) {
  const size_t pages = (bytes + 4095) / 4096;
  begin = std::min(bytes, pages * slice / slices * 4096);
  end = std::min(bytes, pages * (slice + 1) / slices * 4096);
}

// memory the runtime knows (pinned, managed, a device's) is no matter of the ring
bool pageable(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();  // memory it has never seen
  return true;
}

}  // namespace

HostTransfer::~HostTransfer() {
  for (auto &e : event_)
    if (e) (void)hipEventDestroy(e);
}

bool HostTransfer::ring() {
  if (tried_) return ready_;
  tried_ = true;
  for (int k = 0; k < kRing; ++k) {
    buf_[k] = HostBuffer(kChunk);
    if (!buf_[k].pinned()) return false;
    CC4S_HIP(hipEventCreateWithFlags(&event_[k], hipEventDisableTiming));
  }
  return ready_ = true;
}

void HostTransfer::download(void *host, const void *device, size_t bytes, hipStream_t s) {
  auto direct = [&] {
    CC4S_HIP(hipMemcpyAsync(host, device, bytes, hipMemcpyDeviceToHost, s));
  };
  if (bytes < kStagedBytes || !pageable(host) || !ring()) return direct();
  const size_t n = (bytes + kChunk - 1) / kChunk;
  auto len = [&](size_t c) { return std::min(kChunk, bytes - c * kChunk); };
  Copiers copiers(n, [&](size_t c, int slice, int slices) {
    size_t b, e;
    slice_of(len(c), slice, slices, b, e);
    if (e > b)
      std::memcpy(static_cast<char *>(host) + c * kChunk + b,
                  static_cast<const char *>(buf_[c % kRing].get()) + b, e - b);
  });
  if (!copiers.count()) return direct();
  size_t issued = 0;
  for (size_t c = 0; c < n; ++c) {
    // one buffer less than the ring in flight: the wait for a free one is for a
    // chunk that was opened two chunks ago
    for (; issued < std::min(n, c + kRing - 1); ++issued) {
      if (issued >= kRing) copiers.wait(issued - kRing);
      CC4S_HIP(hipMemcpyAsync(buf_[issued % kRing].get(),
                              static_cast<const char *>(device) + issued * kChunk, len(issued),
                              hipMemcpyDeviceToHost, s));
      CC4S_HIP(hipEventRecord(event_[issued % kRing], s));
    }
    CC4S_HIP(hipEventSynchronize(event_[c % kRing]));
    copiers.open(c + 1);
  }
  copiers.wait(n - 1);
}

void HostTransfer::upload(void *device, const void *host, size_t bytes, hipStream_t s) {
  auto direct = [&] {
    CC4S_HIP(hipMemcpyAsync(device, host, bytes, hipMemcpyHostToDevice, s));
  };
  if (bytes < kStagedBytes || !pageable(host) || !ring()) return direct();
  const size_t n = (bytes + kChunk - 1) / kChunk;
  auto len = [&](size_t c) { return std::min(kChunk, bytes - c * kChunk); };
  {
    Copiers copiers(n, [&](size_t c, int slice, int slices) {
      size_t b, e;
      slice_of(len(c), slice, slices, b, e);
      if (e > b)
        std::memcpy(static_cast<char *>(buf_[c % kRing].get()) + b,
                    static_cast<const char *>(host) + c * kChunk + b, e - b);
    });
    if (!copiers.count()) return direct();
    copiers.open(kRing);
    for (size_t c = 0; c < n; ++c) {
      copiers.wait(c);
      CC4S_HIP(hipMemcpyAsync(static_cast<char *>(device) + c * kChunk, buf_[c % kRing].get(),
                              len(c), hipMemcpyHostToDevice, s));
      CC4S_HIP(hipEventRecord(event_[c % kRing], s));
      if (c >= 1) {  // the chunk before has left its buffer
        CC4S_HIP(hipEventSynchronize(event_[(c - 1) % kRing]));
        copiers.open(c + kRing);
      }
    }
  }
  CC4S_HIP(hipStreamSynchronize(s));
}

}  // namespace cc4s_amd
