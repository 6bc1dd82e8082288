// pinned_shim.cpp -- a hipHostMalloc that can be told to refuse requests of
// `refuse_from` bytes and more (0: none), loaded ahead of the library by
// test_gpu_pinned.py: pinned memory that is not to be had.
#include <dlfcn.h>
#include <stddef.h>

extern "C" {
long refuse_from = 0, refused = 0;
int hipHostMalloc(void** p, size_t bytes, unsigned flags)
{
    typedef int (*Fn)(void**, size_t, unsigned);
    static const Fn real = (Fn)dlsym(RTLD_NEXT, "hipHostMalloc");
    if (refuse_from > 0 && bytes >= (size_t)refuse_from) {
        ++refused;
        *p = nullptr;
        return 2; // hipErrorOutOfMemory
    }
    return real(p, bytes, flags);
}
}
