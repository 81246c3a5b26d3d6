// Device and pinned allocations of at least 1 MB, counted; device memory refused
// on demand (1: those, -1: the next of any size).  Loaded with RTLD_GLOBAL before libepic_gpu.so, whose calls then come here.
#include <dlfcn.h>

#include <cstddef>

extern "C" {
int watch_refuse_device = 0;
long watch_device = 0, watch_pinned = 0;
}

namespace {
template <class F> F real(const char *name)
{
    return (F)dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD), name);
}
constexpr size_t LARGE = size_t(1) << 20;
}  // namespace

extern "C" int hipMalloc(void **p, size_t n)
{
    if (watch_refuse_device < 0 || (watch_refuse_device > 0 && n >= LARGE)) {
        if (watch_refuse_device < 0) watch_refuse_device = 0;
        *p = nullptr;
        return 2;   // hipErrorOutOfMemory
    }
    if (n >= LARGE) ++watch_device;
    return real<int (*)(void **, size_t)>("hipMalloc")(p, n);
}

extern "C" int hipHostMalloc(void **p, size_t n, unsigned flags)
{
    if (n >= LARGE) ++watch_pinned;
    return real<int (*)(void **, size_t, unsigned)>("hipHostMalloc")(p, n, flags);
}
