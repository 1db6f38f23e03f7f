// hipMalloc with a countdown, for programs that load this library first and
// globally: the call that the countdown meets reports that the device is out of
// memory.
#include <dlfcn.h>

#include <cstddef>

static int left = -1;

extern "C" void malloc_limit(int calls) { left = calls; }

extern "C" int hipMalloc(void **p, size_t bytes) {
    if (left >= 0 && left-- == 0) return 2;  // hipErrorOutOfMemory
    static const auto real = reinterpret_cast<int (*)(void **, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
    static const auto late = [] {
        void *h = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD);
        return h ? reinterpret_cast<int (*)(void **, size_t)>(dlsym(h, "hipMalloc")) : nullptr;
    }();
    return real ? real(p, bytes) : late(p, bytes);
}
