// The context's growing buffers (iroiro_amd/csrc/ii_api.hip) where an allocation
// fails, compiled for the host against a stand-in for the HIP calls: what was
// freed to make room must not be handed out, or freed, again.
#include "../../iroiro_amd/csrc/ii_api.hip"

#include <cstdio>
#include <cstdlib>
#include <set>

#define CHECK(c, ...)                                     \
  do {                                                    \
    if (!(c)) {                                           \
      std::fprintf(stderr, "alloc_check: " __VA_ARGS__); \
      std::fprintf(stderr, "\n");                         \
      std::_Exit(1);                                      \
    }                                                     \
  } while (0)

namespace sim {
std::set<void*> live;
bool fail = false;
hipError_t get(void** p, size_t n) {
  if (fail) return hipErrorOutOfMemory;  // *p as it was
  *p = std::malloc(16);
  live.insert(*p);
  return hipSuccess;
}
hipError_t put(void* p) {
  CHECK(!p || live.erase(p), "freed twice");
  std::free(p);
  return hipSuccess;
}
}  // namespace sim

// the allocation calls, and no others, under their own names
extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return sim::get(p, n); }
hipError_t hipFree(void* p) { return sim::put(p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return sim::get(p, n); }
hipError_t hipHostFree(void* p) { return sim::put(p); }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
}

int main() {
  using namespace ii;
  for (int which = 0; which < 4; ++which) {
    ii_context c;
    auto grow = [&](int n, void** p) -> ii_status {
      ii_status st = II_OK;
      if (which == 0) {
        st = ensure_partials(&c, (size_t)n * 100000);
        *p = c.partials;
      } else if (which == 1) {
        st = ensure_scalars(&c, n * 100);
        *p = c.scal;
      } else if (which == 2) {
        st = ensure_host_pin(&c, n, p);
      } else {
        st = workspace(&c, 3, n, p);
      }
      return st;
    };
    void* p = nullptr;
    CHECK(grow(2, &p) == II_OK && sim::live.count(p), "buffer %d", which);
    sim::fail = true;
    CHECK(grow(3, &p) != II_OK, "buffer %d grew without memory", which);
    sim::fail = false;
    p = nullptr;
    CHECK(grow(1, &p) == II_OK, "buffer %d after a failure", which);
    CHECK(sim::live.count(p), "buffer %d handed out after it was freed", which);
    CHECK(grow(4, &p) == II_OK && sim::live.count(p), "buffer %d grows again", which);
  }
  std::printf("alloc_check: ok\n");
  return 0;
}
