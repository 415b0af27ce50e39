// Allocation of device memory and the registry of what can be given back.
#include "device_memory.hpp"

#include <algorithm>
#include <condition_variable>
#include <mutex>
#include <vector>

namespace cc4s_amd {

namespace {
// never destroyed: contexts may outlive the objects of this file at process exit
struct Registry {
  std::mutex lock;  // of all that follows and of every SpareMemory's flags
  std::vector<SpareMemory *> all;
  std::condition_variable use_ended;
  int waiting = 0;       // threads that wait for memory in use
  uint64_t releases = 0; // times that memory was given back
};
Registry &registry() {
  static auto *r = new Registry;
  return *r;
}
thread_local int t_uses = 0;  // of this thread: it must not wait for another's
}  // namespace

SpareMemory::SpareMemory(std::function<void()> give_back) : give_back_(std::move(give_back)) {
  CC4S_HIP(hipGetDevice(&device_));
  std::lock_guard<std::mutex> l(registry().lock);
  registry().all.push_back(this);
}

SpareMemory::~SpareMemory() {
  std::lock_guard<std::mutex> l(registry().lock);
  auto &all = registry().all;
  all.erase(std::remove(all.begin(), all.end(), this), all.end());
}

void SpareMemory::begin_use() {
  std::lock_guard<std::mutex> l(registry().lock);
  used_ = true;
  ++t_uses;
}

void SpareMemory::end_use() {
  Registry &r = registry();
  std::lock_guard<std::mutex> l(r.lock);
  used_ = false;
  --t_uses;
  if (!r.waiting) return;
  release_locked();  // the next use could begin before a waiting thread runs
  r.use_ended.notify_all();
}

void SpareMemory::set_held(bool held) {
  std::lock_guard<std::mutex> l(registry().lock);
  held_ = held;
}

bool SpareMemory::release_locked() {
  if (used_ || !held_) return false;
  give_back_();
  held_ = false;
  ++registry().releases;
  return true;
}

bool SpareMemory::release() {
  std::lock_guard<std::mutex> l(registry().lock);
  return release_locked();
}

// every context's on this device that is not in use, or what is when its use ends;
// whether any was given back
bool release_spare_memory(int device) {
  Registry &r = registry();
  std::unique_lock<std::mutex> l(r.lock);
  bool any = false;
  for (SpareMemory *s : r.all)
    if (s->device_ == device) any = s->release_locked() || any;
  if (any || t_uses) return any;
  const uint64_t before = r.releases;
  auto in_use = [&] {
    for (SpareMemory *s : r.all)
      if (s->device_ == device && s->used_ && s->held_) return true;
    return false;
  };
  ++r.waiting;
  r.use_ended.wait(l, [&] { return r.releases != before || !in_use(); });
  --r.waiting;
  return r.releases != before;
}

void *device_malloc(size_t bytes) {
  void *p = nullptr;
  int device = 0;
  hipError_t e = hipMalloc(&p, bytes);
  while (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();  // not an error of the next call
    CC4S_HIP(hipGetDevice(&device));
    if (!release_spare_memory(device))
      throw OutOfMemory("HIP error '" + std::string(hipGetErrorString(e)) + "' allocating " +
                        std::to_string(bytes) + " bytes");
    e = hipMalloc(&p, bytes);
  }
  CC4S_HIP(e);
  return p;
}

size_t device_free_bytes(size_t wanted) {
  size_t free_b = 0, total_b = 0;
  int device = 0;
  CC4S_HIP(hipGetDevice(&device));
  CC4S_HIP(hipMemGetInfo(&free_b, &total_b));
  while (free_b < wanted && release_spare_memory(device))
    CC4S_HIP(hipMemGetInfo(&free_b, &total_b));
  return free_b;
}

}  // namespace cc4s_amd
