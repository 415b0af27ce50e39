// Allocation of device memory and the registry of what can be given back.
#include "device_memory.hpp"

#include <algorithm>
#include <vector>

namespace cc4s_amd {

namespace {
// never destroyed: contexts may outlive the objects of this file at process exit
std::mutex &registry_lock() {
  static auto *m = new std::mutex;
  return *m;
}
std::vector<SpareMemory *> &registry() {
  static auto *r = new std::vector<SpareMemory *>;
  return *r;
}
}  // namespace

SpareMemory::SpareMemory(std::function<void()> give_back) : give_back_(std::move(give_back)) {
  CC4S_HIP(hipGetDevice(&device_));
  std::lock_guard<std::mutex> l(registry_lock());
  registry().push_back(this);
}

SpareMemory::~SpareMemory() {
  std::lock_guard<std::mutex> l(registry_lock());
  auto &r = registry();
  r.erase(std::remove(r.begin(), r.end(), this), r.end());
}

void SpareMemory::set_used(bool used) {
  std::lock_guard<std::mutex> l(m_);
  used_ = used;
}

void SpareMemory::set_held(bool held) {
  std::lock_guard<std::mutex> l(m_);
  held_ = held;
}

bool SpareMemory::release() {
  std::lock_guard<std::mutex> l(m_);
  if (used_ || !held_) return false;
  give_back_();
  held_ = false;
  return true;
}

// every context's on this device that is not in use; whether there was any
bool release_spare_memory(int device) {
  std::lock_guard<std::mutex> l(registry_lock());
  bool any = false;
  for (SpareMemory *s : registry())
    if (s->device_ == device) any = s->release() || any;
  return any;
}

void *device_malloc(size_t bytes) {
  void *p = nullptr;
  hipError_t e = hipMalloc(&p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();  // not an error of the next call
    int device = 0;
    CC4S_HIP(hipGetDevice(&device));
    if (release_spare_memory(device)) e = hipMalloc(&p, bytes);
    if (e == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      throw OutOfMemory("HIP error '" + std::string(hipGetErrorString(e)) + "' allocating " +
                        std::to_string(bytes) + " bytes");
    }
  }
  CC4S_HIP(e);
  return p;
}

size_t device_free_bytes(size_t wanted) {
  size_t free_b = 0, total_b = 0;
  CC4S_HIP(hipMemGetInfo(&free_b, &total_b));
  if (free_b < wanted) {
    int device = 0;
    CC4S_HIP(hipGetDevice(&device));
    if (release_spare_memory(device)) CC4S_HIP(hipMemGetInfo(&free_b, &total_b));
  }
  return free_b;
}

}  // namespace cc4s_amd
