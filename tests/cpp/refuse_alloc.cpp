// A hipMalloc that refuses requests above a limit, for tests/test_gpu_refusals.py: loaded
// with RTLD_GLOBAL before the library, it stands before the runtime's own.
#include <dlfcn.h>

#include <cstddef>
#include <cstdint>

static size_t limit_bytes = SIZE_MAX;
static int refused_calls = 0;

extern "C" void refuse_above(size_t bytes) {
  limit_bytes = bytes;
  refused_calls = 0;
}
extern "C" int refused() { return refused_calls; }

extern "C" int hipMalloc(void **p, size_t bytes) {
  if (bytes > limit_bytes) {
    ++refused_calls;
    return 2;  // hipErrorOutOfMemory
  }
  static auto real = reinterpret_cast<int (*)(void **, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
  return real(p, bytes);
}
