// HIP calls of libtdvmc.so seen and refused from a test: loaded before it with
// RTLD_GLOBAL, this library's definitions are the ones it calls.
#include <dlfcn.h>
#include <stddef.h>

extern "C" {

int shim_refuse_pinned = 0;    // hipHostMalloc returns hipErrorOutOfMemory
int shim_refused = 0;          // how often it did

int hipHostMalloc(void** ptr, size_t size, unsigned flags)
{
    if (shim_refuse_pinned) {
        shim_refused++;
        *ptr = nullptr;
        return 2;
    }
    using F = int (*)(void**, size_t, unsigned);
    static const F next = reinterpret_cast<F>(dlsym(RTLD_NEXT, "hipHostMalloc"));
    return next(ptr, size, flags);
}

}
