// x0ne_arena_scrub over a stream whose calls this program answers in the HIP runtime's place (its
// definitions come before the runtime library's): whether the fills are accepted or refused, the
// stream is drained before the call returns, after the last fill. A request's copies out of its
// caller's memory are queued without a wait and rely on that. Exit status 0: all hold.
#include <cstdio>
#include <cstdlib>

#include "internal.h"

static bool refuse = false;
static int fills = 0, drains = 0, fills_before_drain = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return (*p = std::malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) {
    ++fills;
    return refuse ? hipErrorInvalidValue : hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    ++drains;
    fills_before_drain = fills;
    return hipSuccess;
}
}

#define CHECK(c)                                              \
    do {                                                      \
        if (!(c)) {                                           \
            std::fprintf(stderr, "%s (line %d)\n", #c, __LINE__); \
            std::exit(1);                                     \
        }                                                     \
    } while (0)

int main() {
    x0ne_gpu gpu;
    x0ne_arena* a = nullptr;
    x0ne_slice s[4];
    CHECK(x0ne_arena_new(&a) == X0NE_OK);
    const uint32_t cls[4] = {X0NE_CLASS_CLIENT_DATA, X0NE_CLASS_CLIENT_DATA, X0NE_CLASS_WEIGHTS, X0NE_CLASS_CLIENT_DATA};
    for (int i = 0; i < 4; ++i) CHECK(x0ne_arena_alloc(a, "r", 100, cls[i], &s[i]) == X0NE_OK);
    CHECK(x0ne_arena_freeze(a, &gpu) == X0NE_OK);
    uint64_t zeroed = 0;
    CHECK(x0ne_arena_scrub(a, &zeroed) == X0NE_OK);
    CHECK(zeroed == 300 && fills == 2 && drains == 1 && fills_before_drain == 2);
    refuse = true;
    CHECK(x0ne_arena_scrub(a, &zeroed) == X0NE_ERR_GPU);
    CHECK(drains == 2 && fills_before_drain == fills);
    x0ne_arena_free(a);
}
