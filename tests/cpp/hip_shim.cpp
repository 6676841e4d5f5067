// HIP calls of libtdvmc.so seen and refused from a test: loaded before it with
// RTLD_GLOBAL, this library's definitions are the ones it calls.
#include <dlfcn.h>
#include <stddef.h>

struct ShimDim3 {
    unsigned x, y, z;
};

extern "C" {

int shim_refuse_pinned = 0;    // hipHostMalloc returns hipErrorOutOfMemory
int shim_refused = 0;          // how often it did
size_t shim_pinned = 0;        // bytes asked of hipHostMalloc
size_t shim_most_lds = 0;      // largest dynamic LDS of the launches since it was cleared

int hipHostMalloc(void** ptr, size_t size, unsigned flags)
{
    shim_pinned += size;
    if (shim_refuse_pinned) {
        shim_refused++;
        *ptr = nullptr;
        return 2;
    }
    using F = int (*)(void**, size_t, unsigned);
    static const F next = reinterpret_cast<F>(dlsym(RTLD_NEXT, "hipHostMalloc"));
    return next(ptr, size, flags);
}

// what every kernel<<<>>> launch passes its shape through
unsigned __hipPushCallConfiguration(ShimDim3 grid, ShimDim3 block, size_t lds, void* stream)
{
    if (lds > shim_most_lds) shim_most_lds = lds;
    using F = unsigned (*)(ShimDim3, ShimDim3, size_t, void*);
    static const F next = reinterpret_cast<F>(dlsym(RTLD_NEXT, "__hipPushCallConfiguration"));
    return next(grid, block, lds, stream);
}

}
