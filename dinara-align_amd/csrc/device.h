// Device contexts and memory of the library: one stream per GPU, every call ordered on it.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <mutex>
#include <vector>

namespace dinara {

// A block of device memory that holds one batch's buffers, kept by the context for the next batch when it is given back.
// `image` (small blocks only) is as much pinned host memory: a batch's uploads are gathered in it and go in one copy,
// and its results come back in one.
struct Region {
    uint8_t *base = nullptr;
    uint8_t *image = nullptr;
    size_t size = 0;
    bool holds(const void *at, size_t bytes) const {
        const uint8_t *p = static_cast<const uint8_t *>(at);
        return base && p >= base && bytes <= size && (size_t)(p - base) <= size - bytes;
    }
};
// Two sizes, and how many of each a context keeps (144 MiB together): a call's own hipMallocs and hipFrees, about 45 of
// each at 1 us, and as many waits at 10 us as it has uploads and results cost one read 0.55 ms in all, 0.3 of it so.
constexpr size_t REGION_SMALL = size_t(1) << 20, REGION_LARGE = size_t(64) << 20;
constexpr size_t REGIONS_SMALL = 16, REGIONS_LARGE = 2;
// And how many batches may hold at once; a further batch's buffers are allocated one by one.
constexpr size_t REGIONS_SMALL_OUT = 64, REGIONS_LARGE_OUT = 4;

struct DeviceContext {
    int id = 0;
    hipStream_t stream = nullptr;
    hipEvent_t start = nullptr, stop = nullptr, sweep_start = nullptr, sweep_stop = nullptr;
    size_t lds_limit = 0;  // dynamic LDS one workgroup may take
    int compute_units = 0;
    std::vector<hipEvent_t> pool;  // timing events, made as needed
    hipEvent_t event(size_t i);
    // Further streams for launches that may run side by side, forked from and joined back to `stream` by events;
    // made as needed, default priority.
    std::vector<hipStream_t> sides;
    std::vector<hipEvent_t> marks;  // events that only order streams (no timing)
    hipStream_t side(size_t i);
    hipEvent_t mark(size_t i);
    // A free region of at least `bytes`, or none (above REGION_LARGE, or no memory); and one given back, whose device
    // must be done with it: kept, or freed when enough are.
    Region take_region(size_t bytes);
    void give_region(const Region &region);
    void drop_regions();  // frees every region kept
    std::mutex regions_lock;
    std::vector<Region> regions_small, regions_large;
    size_t regions_small_out = 0, regions_large_out = 0;
    std::mutex lock;  // one caller's work on the stream at a time (the events are shared)
    // The unit-cost path's decision arena, lent to each alignment run under `lock` (a run walks its decisions before
    // it returns, so no batch holds it between runs): allocated once, grown when a run wants more, kept until the
    // process ends, so a fresh batch does not pay for mapping tens of gigabytes.
    struct DeviceBuffer *edit_arena = nullptr;
    void *strip_plan = nullptr;  // the strip rounds' plan on the host (batch.hip), used under `lock`
    size_t arena_wanted = 0;  // twice what the last run that left pairs without room had, for runs that may use it
};

// The context of GPU `gpu`, made on first use; null when there is no such GPU.
DeviceContext *device_context(int64_t gpu);
int64_t device_count();

// Makes the context's GPU current for the calling thread, and restores the previous one after.
struct DeviceGuard {
    int previous = -1;
    explicit DeviceGuard(const DeviceContext *ctx);
    ~DeviceGuard();
};

// A fixed device region handed out front to back, 256-byte aligned: the memory of calls that may not allocate.
struct Carve {
    uint8_t *base = nullptr;
    size_t size = 0;
    size_t used = 0;
    bool exhausted = false;    // a reservation found no room
    bool strict = true;        // such a reservation fails; else it is allocated apart
    uint8_t *image = nullptr;  // uploads into the region are gathered here until flush()
    size_t gathered = 0;
    bool flush(DeviceContext *ctx);  // one copy of what was gathered, on the context's stream
    void *take(size_t bytes);  // null (and `exhausted` set) when the region has no room left
};

// While one of these lives on a thread, every DeviceBuffer that thread reserves comes from `carve` and (`strict`) no
// device memory is allocated; such a buffer is never freed (the region outlives it).
struct CarveScope {
    Carve *previous;
    explicit CarveScope(Carve *carve);
    ~CarveScope();
    static bool active();  // on this thread
};

// Gives a batch's region back to its context once nothing on the device uses it (a run that failed may have left work).
void give_back(DeviceContext *ctx, const Region &region);

// Device memory that grows on demand and is freed with its owner.
struct DeviceBuffer {
    void *ptr = nullptr;
    size_t size = 0;
    bool carved = false;  // taken from a Carve: not ours to free
    DeviceBuffer() = default;
    DeviceBuffer(const DeviceBuffer &) = delete;
    DeviceBuffer &operator=(const DeviceBuffer &) = delete;
    ~DeviceBuffer();
    bool reserve(size_t bytes);                                          // at least `bytes`, contents dropped
    void release();                                                      // frees it now
    bool upload(DeviceContext *ctx, const void *host, size_t bytes);     // reserve, copy, wait
    bool write(DeviceContext *ctx, const void *host, size_t bytes);      // copy into what is there, wait
    bool read(DeviceContext *ctx, void *host, size_t bytes) const;       // copy out after the stream's work
};

}  // namespace dinara
