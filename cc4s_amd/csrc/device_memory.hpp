// Device memory: allocation, and memory that can be given back.
#pragma once

#include "common.hpp"

#include <functional>
#include <mutex>

namespace cc4s_amd {

// the device is full
struct OutOfMemory : Error {
  using Error::Error;
};

// Allocates on the current device.  If that is full, spare memory is given back
// and the allocation tried again.
void *device_malloc(size_t bytes);

// Free bytes of the current device; where that is less than `wanted`, after spare
// memory was given back.
size_t device_free_bytes(size_t wanted);

// Memory that a context keeps only to be faster.  While no Use of it exists, an
// allocation that finds the device full, of any context and on any thread, has it
// given back by `give_back`.  The registry of these objects and every object are
// locked while that runs, so it only frees.
class SpareMemory {
 public:
  explicit SpareMemory(std::function<void()> give_back);
  ~SpareMemory();
  SpareMemory(const SpareMemory &) = delete;
  SpareMemory &operator=(const SpareMemory &) = delete;

  // keeps the memory where it is
  class Use {
   public:
    explicit Use(SpareMemory &m) : m_(m) { m_.set_used(true); }
    ~Use() { m_.set_used(false); }
    Use(const Use &) = delete;
    Use &operator=(const Use &) = delete;

   private:
    SpareMemory &m_;
  };
  void set_held(bool held);  // in a Use: there is memory to give back
  // gives it back unless it is in use; whether there was any
  bool release();

 private:
  friend bool release_spare_memory(int device);
  void set_used(bool used);
  std::function<void()> give_back_;
  int device_ = 0;
  std::mutex m_;
  bool used_ = false, held_ = false;
};

}  // namespace cc4s_amd
