#include "device_memory.h"

#include <stdlib.h>

#include <algorithm>
#include <mutex>
#include <vector>

namespace rtg {

namespace {
struct Spares {
  std::mutex mu;
  std::vector<SpareMemory*> all;
};
Spares& spares() {
  static Spares* s = new Spares();  // (kept to the process's end)
  return *s;
}
bool give_all_back(int device) {
  std::lock_guard<std::mutex> g(spares().mu);
  bool any = false;
  for (SpareMemory* s : spares().all) any |= s->give_back(device);
  return any;
}
}  // namespace

void register_spare(SpareMemory* s) {
  std::lock_guard<std::mutex> g(spares().mu);
  spares().all.push_back(s);
}
void unregister_spare(SpareMemory* s) {
  std::lock_guard<std::mutex> g(spares().mu);
  auto& all = spares().all;
  all.erase(std::remove(all.begin(), all.end(), s), all.end());
}

hipError_t device_malloc_bytes(void** p, size_t n) {
  // test hook RTG_TEST_MALLOC_FAIL=1: as if the memory held in spare were
  // missing here
  const char* t = getenv("RTG_TEST_MALLOC_FAIL");
  hipError_t e = t && t[0] == '1' ? hipErrorOutOfMemory : hipMalloc(p, n);
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  int device = 0;
  const bool freed = hipGetDevice(&device) == hipSuccess && give_all_back(device);
  return freed || (t && t[0] == '1') ? hipMalloc(p, n) : e;
}

}  // namespace rtg
