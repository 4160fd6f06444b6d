// The pool of device memory and context parts (csrc/device_pool.h) against a runtime of this file's own: host memory
// instead of device memory, and any of its calls made to fail.  No GPU, no HIP library.
#include "device_pool.h"

#include <cstdio>
#include <cstdlib>
#include <set>

static int failures = 0;
#define CHECK(cond, ...)                                                        \
    do {                                                                        \
        if (!(cond)) {                                                          \
            ++failures;                                                         \
            std::printf("FAILED %s:%d: %s: ", __FILE__, __LINE__, #cond);       \
            std::printf(__VA_ARGS__);                                           \
            std::printf("\n");                                                  \
        }                                                                       \
    } while (0)

// ---- the runtime --------------------------------------------------------------------------------------------------
namespace rt {
std::set<void *> live;                 // what was created and not yet destroyed
int calls = 0;                         // of those that create something
int fail_from = -1, fail_count = 0;    // calls [fail_from, fail_from + fail_count) fail
hipError_t fail_with = hipErrorOutOfMemory;
int bad_destroys = 0;                  // of something that is not there

hipError_t create(void **out, size_t bytes) {
    const int n = calls++;
    if (fail_from >= 0 && n >= fail_from && n < fail_from + fail_count) return fail_with;
    *out = std::malloc(bytes);
    live.insert(*out);
    return hipSuccess;
}
hipError_t destroy(void *p) {
    if (!live.erase(p)) {
        ++bad_destroys;
        return hipErrorInvalidValue;
    }
    std::free(p);
    return hipSuccess;
}
void fail(int from, int count, hipError_t with = hipErrorOutOfMemory) {
    calls = 0;
    fail_from = from;
    fail_count = count;
    fail_with = with;
}
}  // namespace rt

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t bytes) { return rt::create(p, bytes); }
hipError_t hipFree(void *p) { return rt::destroy(p); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned int) { return rt::create(p, bytes); }
hipError_t hipHostFree(void *p) { return rt::destroy(p); }
hipError_t hipStreamCreate(hipStream_t *s) { return rt::create((void **)s, 1); }
hipError_t hipStreamDestroy(hipStream_t s) { return rt::destroy((void *)s); }
hipError_t hipEventCreate(hipEvent_t *e) { return rt::create((void **)e, 1); }
hipError_t hipEventDestroy(hipEvent_t e) { return rt::destroy((void *)e); }
}

using namespace sddmm;

static bool whole(const ContextParts &c) { return c.stream && c.ev0 && c.ev1 && c.counters && c.host_counters; }

// Every step of making a context's parts fails, for good or only until the pool has given memory back: an error that
// leaves nothing behind, or a whole set.
static void parts_that_fail() {
    for (hipError_t with : {hipErrorOutOfMemory, hipErrorUnknown})
        for (int at = 0; at < 5; ++at)
            for (int count : {1, 1000}) {
                void *block = nullptr;
                rt::fail(-1, 0);
                CHECK(pool_alloc(&block, 4096) == hipSuccess, "block");
                pool_free(block, true);                      // something that the pool can give back
                rt::fail(at, count, with);
                ContextParts c;
                const hipError_t e = take_parts(&c, 0, 64);
                const bool again = with == hipErrorOutOfMemory && count == 1;
                CHECK((e == hipSuccess) == again, "step %d, %d failures of %d: %d", at, count, (int)with, (int)e);
                CHECK(e == hipSuccess ? whole(c) : e == with, "step %d, %d failures of %d: a set with holes", at, count, (int)with);
                rt::fail(-1, 0);
                if (e == hipSuccess) give_parts(c, true);
                ContextParts next;                           // and the next context gets a whole set
                CHECK(take_parts(&next, 0, 64) == hipSuccess && whole(next), "after step %d", at);
                give_parts(next, true);
                pool_trim();
                CHECK(rt::live.empty(), "step %d, %d failures: %zu left behind", at, count, rt::live.size());
                CHECK(rt::bad_destroys == 0, "step %d: destroyed twice", at);
            }
}

int main() {
    parts_that_fail();
    std::printf("%d failed\n", failures);
    return failures != 0;
}
