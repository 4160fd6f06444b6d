// Device memory and the fixed parts of a context (stream, events, counters), kept for the next pattern and the next
// context instead of going back to the driver.
//
// hipMalloc and hipFree cost 5 .. 25 us each, hipFree waits for the device, and a new pattern made about ten of either.
// sddmm_set_csr_device on a pattern of 2.0 M entries 123 -> 39 us and its plan 188 -> 161; a one-shot call on host arrays
// of 783 k entries paid 50 .. 90 us for creating its context and 125 .. 170 for destroying it (2 and 2 now): 1095 -> 840 us.
//
//   bound   POOL_BYTES of free blocks per device, the oldest go first; no block beyond POOL_BLOCK_MAX is kept;
//           POOL_CONTEXTS sets of parts.  sddmm_trim gives all of it back; an allocation that fails gives the free blocks of
//           its device back and is tried once more.  The bound is what is taken from the program's other allocations; a
//           pattern whose arrays exceed it pays for them as without a pool (set, plan and first launch, 12 M entries 285 us,
//           24 M 740; with blocks of 256 MiB and 1 GiB in all 253 and 408).
//   safety  A block that is given back may be handed to any context of the device, so it is kept only when the device is
//           idle (release_*: one wait for all blocks of a pattern, pool_wait); otherwise it goes to hipFree, which waits.
//           One mutex guards the tables.  They have fixed sizes: nothing here allocates host memory or throws; a block
//           that finds no place in them is a plain hipMalloc / hipFree.
//   reset   hipDeviceReset takes back what is kept; the next context finds that out and starts afresh.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <mutex>
#include <utility>

namespace sddmm {

constexpr size_t POOL_BYTES = (size_t)128 << 20, POOL_BLOCK_MAX = (size_t)32 << 20;
constexpr int POOL_BLOCKS = 512, POOL_CONTEXTS = 8, POOL_DEVICES = 16;
constexpr size_t POOL_WITNESS = 19 * 4096 - 16;              // bytes that hardly any other allocation asks for

// what is asked for, rounded up to eighths of its power of two: patterns of about one size share their blocks
inline size_t pool_round(size_t bytes) {
    size_t step = 4096;
    while (step * 16 <= bytes) step *= 2;
    return bytes > POOL_BLOCK_MAX ? bytes : (bytes + step - 1) / step * step;
}

struct ContextParts {
    int device = -1;
    unsigned int life = 0;                                   // of the device (PoolDevice) that they were made in
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    void *counters = nullptr, *host_counters = nullptr;      // device block, pinned landing place
};

// A device that the pool keeps something of.  hipDeviceReset takes all of it back without a word: the witness, a block that
// only the pool knows, is then gone as well (pool_look_after).
struct PoolDevice {
    int device = -1;
    unsigned int life = 0;                                   // resets seen so far
    void *witness = nullptr;
    size_t bytes = 0;                                        // its size, as the runtime tells it
    void *to_free = nullptr;                                 // by the next pool_wait
};

struct DevicePool {
    struct Block {
        void *p;
        size_t bytes;
        uint64_t freed;      // 0: in use, else when it was given back
        int device;
    };
    std::mutex lock;
    Block block[POOL_BLOCKS] = {};
    int n = 0;
    uint64_t clock = 0;
    ContextParts parts[POOL_CONTEXTS];
    int n_parts = 0;
    PoolDevice devices[POOL_DEVICES];
    int n_devices = 0;
};
inline DevicePool device_pool;

// (the lock is held) takes block i out of the table
inline void pool_drop(DevicePool &d, int i) { d.block[i] = d.block[--d.n]; }

// gives the free blocks of a device (-1: of every device) back to the driver
inline void pool_trim_locked(DevicePool &d, int device) {
    for (int i = d.n - 1; i >= 0; --i)
        if (d.block[i].freed && (device < 0 || d.block[i].device == device)) {
            (void)hipFree(d.block[i].p);
            pool_drop(d, i);
        }
}

inline PoolDevice *pool_device(DevicePool &d, int device) {
    for (int i = 0; i < d.n_devices; ++i)
        if (d.devices[i].device == device) return &d.devices[i];
    return nullptr;
}

// (the lock is held) forgets what a reset of the device took back
inline void pool_look_after(DevicePool &d, PoolDevice &v) {
    size_t bytes = 0;
    if (!v.witness || (hipMemPtrGetInfo(v.witness, &bytes) == hipSuccess && bytes == v.bytes)) return;
    (void)hipGetLastError();
    for (int i = d.n - 1; i >= 0; --i)
        if (d.block[i].device == v.device) pool_drop(d, i);
    for (int i = d.n_parts - 1; i >= 0; --i)
        if (d.parts[i].device == v.device) d.parts[i] = d.parts[--d.n_parts];
    v.witness = v.to_free = nullptr;
    ++v.life;
}

// (the lock is held; device is the current one) Before a new context.  nullptr, or no witness: nothing of this device is kept.
inline PoolDevice *pool_open(DevicePool &d, int device) {
    PoolDevice *v = pool_device(d, device);
    if (!v && d.n_devices < POOL_DEVICES) {
        v = &d.devices[d.n_devices++];
        v->device = device;
    }
    if (!v) return nullptr;
    pool_look_after(d, *v);
    if (!v->witness && (hipMalloc(&v->witness, POOL_WITNESS) != hipSuccess || hipMemPtrGetInfo(v->witness, &v->bytes) != hipSuccess)) {
        (void)hipGetLastError();
        if (v->witness) (void)hipFree(v->witness);
        v->witness = nullptr;
    }
    return v;
}

// memory of the current device
inline hipError_t pool_alloc(void **out, size_t bytes) {
    *out = nullptr;
    bytes = pool_round(bytes ? bytes : 16);
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    DevicePool &d = device_pool;
    const std::lock_guard<std::mutex> hold(d.lock);
    int best = -1;                                           // the smallest that holds it, at most a quarter larger
    for (int i = 0; i < d.n; ++i) {
        const DevicePool::Block &b = d.block[i];
        if (b.freed && b.device == device && b.bytes >= bytes && b.bytes <= bytes + bytes / 4 &&
            (best < 0 || b.bytes < d.block[best].bytes)) best = i;
    }
    if (best >= 0) {
        d.block[best].freed = 0;
        *out = d.block[best].p;
        return hipSuccess;
    }
    e = hipMalloc(out, bytes);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        pool_trim_locked(d, device);
        e = hipMalloc(out, bytes);
    }
    if (e != hipSuccess) { *out = nullptr; return e; }
    const PoolDevice *v = pool_device(d, device);
    if (bytes <= POOL_BLOCK_MAX && d.n < POOL_BLOCKS && v && v->witness) d.block[d.n++] = DevicePool::Block{*out, bytes, 0, device};
    return hipSuccess;
}

// Waits for all work of the current device, on whatever stream: false if it could not.  As hipFree does it, by freeing
// something: hipDeviceSynchronize breaks every capture in progress, those of other threads and of relaxed mode too.  A new
// pattern 218 us with it, 213 with hipDeviceSynchronize; 30 .. 80 us more once, after a program's other work.
inline bool pool_wait() {
    DevicePool &d = device_pool;
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess) return false;
    void *p = nullptr;
    {
        const std::lock_guard<std::mutex> hold(d.lock);
        PoolDevice *v = pool_device(d, device);
        if (v) std::swap(p, v->to_free);
    }
    const bool waited = (p || hipMalloc(&p, 16) == hipSuccess) && hipFree(p) == hipSuccess;
    if (waited && hipMalloc(&p, 16) == hipSuccess) {         // the next one, where the last one was: a new place costs 40 us
        const std::lock_guard<std::mutex> hold(d.lock);
        PoolDevice *v = pool_device(d, device);
        if (v && v->witness && !v->to_free) std::swap(p, v->to_free);
        else (void)hipFree(p);
    }
    (void)hipGetLastError();
    return waited;
}

// idle: the caller knows that no work which uses the block is in flight
inline void pool_free(void *p, bool idle) {
    if (!p) return;
    DevicePool &d = device_pool;
    const std::lock_guard<std::mutex> hold(d.lock);
    int at = -1;
    for (int i = 0; i < d.n && at < 0; ++i)
        if (d.block[i].p == p) at = i;
    if (at < 0 || !idle) {
        if (at >= 0) pool_drop(d, at);
        (void)hipFree(p);
        return;
    }
    const int device = d.block[at].device;
    d.block[at].freed = ++d.clock;
    for (;;) {
        size_t kept = 0;
        int oldest = -1;
        for (int i = 0; i < d.n; ++i)
            if (d.block[i].freed && d.block[i].device == device) {
                kept += d.block[i].bytes;
                if (oldest < 0 || d.block[i].freed < d.block[oldest].freed) oldest = i;
            }
        // (a quarter of the table stays free for blocks in use)
        if (oldest < 0 || (kept <= POOL_BYTES && d.n <= POOL_BLOCKS * 3 / 4)) return;
        (void)hipFree(d.block[oldest].p);
        pool_drop(d, oldest);
    }
}

inline void destroy_parts(ContextParts &c) {
    if (c.counters) (void)hipFree(c.counters);
    if (c.host_counters) (void)hipHostFree(c.host_counters);
    if (c.ev0) (void)hipEventDestroy(c.ev0);
    if (c.ev1) (void)hipEventDestroy(c.ev1);
    if (c.stream) (void)hipStreamDestroy(c.stream);
    c = ContextParts{};
}

// device is the current one
inline hipError_t take_parts(ContextParts *out, int device, size_t counter_bytes) {
    unsigned int life = 0;
    {
        DevicePool &d = device_pool;
        const std::lock_guard<std::mutex> hold(d.lock);
        const PoolDevice *v = pool_open(d, device);
        if (v) life = v->life;
        for (int i = d.n_parts - 1; i >= 0; --i)
            if (d.parts[i].device == device) {
                *out = d.parts[i];
                d.parts[i] = d.parts[--d.n_parts];
                return hipSuccess;
            }
    }
    ContextParts c;
    auto make = [&]() {
        c.device = device;
        c.life = life;
        hipError_t e = hipStreamCreate(&c.stream);
        if (e == hipSuccess) e = hipEventCreate(&c.ev0);
        if (e == hipSuccess) e = hipEventCreate(&c.ev1);
        if (e == hipSuccess) e = hipMalloc(&c.counters, counter_bytes);
        if (e == hipSuccess) e = hipHostMalloc(&c.host_counters, counter_bytes, hipHostMallocDefault);
        if (e != hipSuccess) destroy_parts(c);
        return e;
    };
    hipError_t e = make();
    if (e == hipErrorOutOfMemory) {                          // the whole set again, once the free blocks are given back
        (void)hipGetLastError();
        {
            const std::lock_guard<std::mutex> hold(device_pool.lock);
            pool_trim_locked(device_pool, device);
        }
        e = make();
    }
    *out = c;
    return e;
}

// idle: nothing that uses them is in flight
inline void give_parts(ContextParts c, bool idle) {
    DevicePool &d = device_pool;
    if (idle) {
        const std::lock_guard<std::mutex> hold(d.lock);
        const PoolDevice *v = pool_device(d, c.device);
        if (v && v->life != c.life) return;                  // a reset took them back
        if (v && v->witness && d.n_parts < POOL_CONTEXTS) {
            d.parts[d.n_parts++] = c;
            return;
        }
    }
    destroy_parts(c);
}

inline void pool_trim() {
    DevicePool &d = device_pool;
    const std::lock_guard<std::mutex> hold(d.lock);
    for (int i = 0; i < d.n_devices; ++i) pool_look_after(d, d.devices[i]);
    pool_trim_locked(d, -1);
    while (d.n_parts > 0) destroy_parts(d.parts[--d.n_parts]);
    for (int i = 0; i < d.n_devices; ++i) {
        PoolDevice &v = d.devices[i];
        bool used = false;
        for (int k = 0; k < d.n; ++k) used = used || d.block[k].device == v.device;
        if (used || !v.witness) continue;                    // (stays as long as a context has blocks of the table)
        (void)hipFree(v.witness);
        if (v.to_free) (void)hipFree(v.to_free);
        v.witness = v.to_free = nullptr;
    }
}

}  // namespace sddmm
