// Device memory: allocation, and memory that can be given back.
#pragma once

#include "common.hpp"

#include <functional>

namespace cc4s_amd {

// the device is full
struct OutOfMemory : Error {
  using Error::Error;
};

// Allocates on the current device.  While that is full, spare memory is given back
// and the allocation tried again.
void *device_malloc(size_t bytes);

// Free bytes of the current device; while that is less than `wanted`, spare memory is
// given back.
size_t device_free_bytes(size_t wanted);

// Memory that a context keeps only to be faster.  An allocation that finds the device
// full, of any context and on any thread, has it given back by `give_back`: at once
// where no Use of it exists, else, unless the asking thread has a Use itself, when the
// Use ends.  One lock is held while that runs, so it only frees.
class SpareMemory {
 public:
  explicit SpareMemory(std::function<void()> give_back);
  ~SpareMemory();
  SpareMemory(const SpareMemory &) = delete;
  SpareMemory &operator=(const SpareMemory &) = delete;

  // keeps the memory where it is; for one thread at a time
  class Use {
   public:
    explicit Use(SpareMemory &m) : m_(m) { m_.begin_use(); }
    ~Use() { m_.end_use(); }
    Use(const Use &) = delete;
    Use &operator=(const Use &) = delete;

   private:
    SpareMemory &m_;
  };
  void set_held(bool held);  // in a Use: there is, or is about to be, memory to give back
  // gives it back unless it is in use; whether there was any
  bool release();

 private:
  friend bool release_spare_memory(int device);
  void begin_use();
  void end_use();
  bool release_locked();
  std::function<void()> give_back_;
  int device_ = 0;
  bool used_ = false, held_ = false;
};

}  // namespace cc4s_amd
