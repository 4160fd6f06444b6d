// The pool of device memory and context parts (csrc/device_pool.h) against a runtime of this file's own: host memory
// instead of device memory, and any of its calls made to fail.  No GPU, no HIP library.
#include "device_pool.h"

#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include <vector>

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
std::map<void *, size_t> sizes;
int calls = 0;                         // of those that create something
int fail_from = -1, fail_count = 0;    // calls [fail_from, fail_from + fail_count) fail
hipError_t fail_with = hipErrorOutOfMemory;
int frees = 0;                         // calls of hipFree: each waits for the device
int bad_destroys = 0;                  // of something that is not there

hipError_t create(void **out, size_t bytes) {
    const int n = calls++;
    if (fail_from >= 0 && n >= fail_from && n < fail_from + fail_count) return fail_with;
    *out = std::malloc(bytes);
    live.insert(*out);
    sizes[*out] = bytes;
    return hipSuccess;
}
hipError_t destroy(void *p) {
    sizes.erase(p);
    if (!live.erase(p)) {
        ++bad_destroys;
        return hipErrorInvalidValue;
    }
    std::free(p);
    return hipSuccess;
}
size_t size_of(void *p) { return sizes.count(p) ? sizes[p] : 0; }
// hipDeviceReset: everything is gone (host memory stays, so that no address comes twice)
void reset() { live.clear(); sizes.clear(); }
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
hipError_t hipMalloc(void **p, size_t bytes) { return rt::create(p, bytes); }
hipError_t hipFree(void *p) { ++rt::frees; return rt::destroy(p); }
hipError_t hipMemPtrGetInfo(void *p, size_t *bytes) { return (*bytes = rt::size_of(p)) ? hipSuccess : hipErrorInvalidValue; }
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
                ContextParts first;                          // (a context leaves a block of the pool's own on the device)
                CHECK(take_parts(&first, 0, 64) == hipSuccess && whole(first), "first");
                destroy_parts(first);
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

static bool alive(const ContextParts &c) {
    return whole(c) && rt::live.count((void *)c.stream) && rt::live.count((void *)c.ev0) && rt::live.count((void *)c.ev1) &&
           rt::live.count(c.counters) && rt::live.count(c.host_counters);
}

// The device is reset while the pool keeps something of it: nothing of that is handed out or destroyed any more.
static void reset_of_the_device() {
    for (bool held : {false, true})                          // a context is open over the reset, or none is
        for (bool trimmed : {false, true}) {                 // sddmm_trim right after it
            rt::fail(-1, 0);
            rt::bad_destroys = 0;
            void *block[3] = {};
            ContextParts old, kept;
            CHECK(take_parts(&old, 0, 64) == hipSuccess && take_parts(&kept, 0, 64) == hipSuccess, "before");
            for (void *&p : block) CHECK(pool_alloc(&p, 8192) == hipSuccess, "before");
            give_parts(kept, true);
            for (void *p : block) pool_free(p, true);
            if (!held) give_parts(old, true);
            rt::reset();
            if (trimmed) pool_trim();
            CHECK(rt::bad_destroys == 0, "trim after a reset destroyed %d things that were gone", rt::bad_destroys);
            ContextParts c, after;
            void *p = nullptr;
            CHECK(take_parts(&c, 0, 64) == hipSuccess && alive(c), "a dead set (%d %d)", held, trimmed);
            CHECK(pool_alloc(&p, 8192) == hipSuccess && rt::live.count(p), "a dead block (%d %d)", held, trimmed);
            if (held) give_parts(old, true);
            CHECK(take_parts(&after, 0, 64) == hipSuccess && alive(after), "a dead set after the old one came back (%d %d)", held, trimmed);
            pool_free(p, true);
            give_parts(c, true);
            give_parts(after, true);
            pool_trim();
            CHECK(rt::live.empty(), "%zu left behind (%d %d)", rt::live.size(), held, trimmed);
            CHECK(rt::bad_destroys == 0, "%d things destroyed that were not there", rt::bad_destroys);
        }
}

// What the pool is for: blocks and parts come back, as far as its limits go.
static void kept_and_bounded() {
    rt::fail(-1, 0);
    ContextParts c, again;
    CHECK(take_parts(&c, 0, 64) == hipSuccess, "parts");
    give_parts(c, true);
    CHECK(take_parts(&again, 0, 64) == hipSuccess && again.stream == c.stream && again.counters == c.counters, "the same set");
    void *p = nullptr, *q = nullptr;
    CHECK(pool_alloc(&p, 100000) == hipSuccess, "block");
    pool_free(p, true);
    CHECK(pool_alloc(&q, 98000) == hipSuccess && q == p, "the same block");
    pool_free(q, true);
    CHECK(pool_alloc(&q, 2 * 100000) == hipSuccess && q != p, "too small");
    pool_free(q, true);
    // more bytes than the limit: the oldest go
    void *big[6];
    for (void *&b : big) CHECK(pool_alloc(&b, POOL_BLOCK_MAX) == hipSuccess, "big");
    for (void *b : big) pool_free(b, true);
    size_t kept = 0;
    for (auto &b : rt::sizes) kept += b.second;
    CHECK(kept <= POOL_BYTES + POOL_WITNESS + 4096, "%zu bytes kept", kept);
    CHECK(!rt::live.count(big[0]) && rt::live.count(big[5]), "the oldest goes first");
    // a block beyond the largest size is not kept
    CHECK(pool_alloc(&p, POOL_BLOCK_MAX + 1) == hipSuccess, "large");
    pool_free(p, true);
    CHECK(!rt::live.count(p), "a large block is kept");
    pool_trim();
    // more blocks than the table keeps, and than it holds
    std::vector<void *> many(2 * POOL_BLOCKS);
    CHECK(take_parts(&c, 0, 64) == hipSuccess, "parts");
    for (void *&b : many) CHECK(pool_alloc(&b, 4096) == hipSuccess, "many");
    for (void *b : many) pool_free(b, true);
    CHECK(device_pool.n <= POOL_BLOCKS * 3 / 4, "%d blocks kept", device_pool.n);
    // more sets than the pool keeps
    ContextParts sets[POOL_CONTEXTS + 3];
    for (ContextParts &s : sets) CHECK(take_parts(&s, 0, 64) == hipSuccess, "set");
    for (ContextParts &s : sets) give_parts(s, true);
    CHECK(device_pool.n_parts == POOL_CONTEXTS, "%d sets kept", device_pool.n_parts);
    // in flight: not kept
    CHECK(pool_alloc(&p, 4096) == hipSuccess, "block");
    give_parts(c, false);
    CHECK(!rt::live.count((void *)c.stream), "a set in flight is kept");
    give_parts(again, true);
    pool_free(p, true);
    pool_trim();
    CHECK(rt::live.empty(), "%zu left behind", rt::live.size());
    CHECK(rt::bad_destroys == 0, "%d things destroyed that were not there", rt::bad_destroys);
}

// The wait is a hipFree of something that is there, whatever fails; without one it says that it could not wait.
static void wait_for_the_device() {
    ContextParts c;
    rt::fail(-1, 0);
    CHECK(take_parts(&c, 0, 64) == hipSuccess, "parts");
    for (int fails : {0, 1000, 1, 0}) {
        rt::fail(fails ? 0 : -1, fails);
        const int before = rt::frees;
        const bool waited = pool_wait();
        CHECK(waited == (rt::frees > before), "waited %d, %d frees", waited, rt::frees - before);
        CHECK(waited || fails, "could not wait");
    }
    rt::fail(-1, 0);
    give_parts(c, true);
    pool_trim();
    CHECK(pool_wait(), "with nothing kept");
    CHECK(rt::live.empty(), "%zu left behind", rt::live.size());
    CHECK(rt::bad_destroys == 0, "%d things destroyed that were not there", rt::bad_destroys);
    // after a reset that no context has noticed yet
    CHECK(take_parts(&c, 0, 64) == hipSuccess && pool_wait(), "parts");
    rt::reset();
    CHECK(!pool_wait() || rt::live.empty(), "what a reset took back was freed for a wait");
    rt::bad_destroys = 0;
    pool_trim();
    CHECK(rt::live.empty() && rt::bad_destroys == 0, "after a reset");
}

int main() {
    parts_that_fail();
    wait_for_the_device();
    reset_of_the_device();
    kept_and_bounded();
    std::printf("%d failed\n", failures);
    return failures != 0;
}
