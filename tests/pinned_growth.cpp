// Counts the pinned allocations of a buffer (HBuf) that every call asks to
// hold a little more, with the HIP runtime's two calls replaced by the host's
// heap.  Prints "allocations bytes" for steps of argv[2] bytes from argv[1] up
// to argv[3]; a request that fits must keep the allocation.  No allocation may
// pass argv[4] bytes: what is asked for must still be given when the reserve
// that the buffer would like is not to be had.
#include "mtpx_internal.hpp"

#include <cstdio>
#include <cstdlib>

static int allocations = 0;
static size_t limit = 0;

extern "C" hipError_t hipHostMalloc(void **p, size_t bytes, unsigned)
{
    if (bytes > limit) {
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    ++allocations;
    *p = std::malloc(bytes);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
extern "C" hipError_t hipHostFree(void *p)
{
    std::free(p);
    return hipSuccess;
}

int main(int, char **argv)
{
    const size_t from = std::strtoul(argv[1], nullptr, 10), step = std::strtoul(argv[2], nullptr, 10),
                 to = std::strtoul(argv[3], nullptr, 10);
    limit = std::strtoul(argv[4], nullptr, 10);
    mtpx::HBuf b;
    for (size_t n = from; n <= to; n += step) {
        const void *before = b.p;
        const bool fits = b.p && n <= b.bytes;
        if (b.ensure(n) != hipSuccess || b.bytes < n || (fits && b.p != before))
            return 1;
    }
    std::printf("%d %zu\n", allocations, b.bytes);
    b.release();
    return b.p || b.bytes;
}
