// hipMalloc that finds no memory for blocks of the size fail_bytes; loaded
// before the library, whose calls then resolve to it.
#include <dlfcn.h>

#include <cstddef>

extern "C" {
size_t fail_bytes = 0;
int failed = 0;

int hipMalloc(void** p, size_t bytes) {
  constexpr int kOutOfMemory = 2;
  using F = int (*)(void**, size_t);
  static F real = nullptr;
  if (!real) {
    void* h = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    real = h ? reinterpret_cast<F>(dlsym(h, "hipMalloc")) : nullptr;
    if (!real) return kOutOfMemory;
  }
  if (fail_bytes && bytes == fail_bytes) {
    ++failed;
    return kOutOfMemory;
  }
  return real(p, bytes);
}
}
