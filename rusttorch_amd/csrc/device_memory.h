// Device memory that can be done without, given back when an allocation fails.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace rtg {

// Something that holds device memory it can do without (a model's second,
// tile-ordered copy of its weights). give_back is called from any thread; it
// returns true if it freed memory.
class SpareMemory {
 public:
  virtual bool give_back(int device) = 0;

 protected:
  ~SpareMemory() = default;
};
void register_spare(SpareMemory* s);
// Once it returns, give_back is not running and will not be called.
void unregister_spare(SpareMemory* s);

// hipMalloc on the current device; where that fails, every registered holder
// gives its memory back and it is tried once more.
hipError_t device_malloc_bytes(void** p, size_t n);
template <class T>
hipError_t device_malloc(T** p, size_t n) {
  return device_malloc_bytes(reinterpret_cast<void**>(p), n);
}

}  // namespace rtg
