// hipMalloc for a test of low device memory: loaded before libxpose.so with its
// symbols global, it takes the calls that libxpose.so makes. A request above
// the limit is passed on as one of 2^50 bytes, so that the runtime itself
// refuses it, with all that a refusal leaves behind.
#include <dlfcn.h>

#include <cstddef>

extern "C" {

size_t alloc_limit = ~size_t(0);   // bytes
size_t alloc_allow = 0;            // a size let through all the same
unsigned alloc_calls = 0, alloc_refused = 0;
size_t alloc_largest = 0;          // of those let through

int hipMalloc(void** p, size_t bytes) {
    static int (*next)(void**, size_t) = reinterpret_cast<int (*)(void**, size_t)>(dlsym(RTLD_NEXT, "hipMalloc"));
    ++alloc_calls;
    if (bytes > alloc_limit && bytes != alloc_allow) {
        ++alloc_refused;
        return next(p, size_t(1) << 50);
    }
    if (bytes > alloc_largest) alloc_largest = bytes;
    return next(p, bytes);
}

}
