// Counts hipHostMalloc calls of a process that loads it, globally, before anything that makes them.
#include <dlfcn.h>
#include <stddef.h>

static int calls = 0;

extern "C" int host_allocations() { return calls; }

extern "C" int hipHostMalloc(void** p, size_t bytes, unsigned flags) {
  ++calls;
  static void* const hip = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);   // as the libraries that call this have loaded it
  static auto* const real = hip ? (int (*)(void**, size_t, unsigned))dlsym(hip, "hipHostMalloc") : nullptr;
  return real ? real(p, bytes, flags) : 1;   // hipErrorInvalidValue: the test then misses the allocation it expects
}
