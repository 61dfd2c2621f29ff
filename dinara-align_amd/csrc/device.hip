// Device contexts and memory (see device.h).
#include "device.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

namespace dinara {

namespace {
std::mutex contexts_mutex;
std::vector<DeviceContext *> contexts;
}  // namespace

int64_t device_count() {
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess) return 0;
    return count;
}

DeviceContext *device_context(int64_t gpu) {
    std::lock_guard<std::mutex> lock(contexts_mutex);
    const int64_t count = device_count();
    if (gpu < 0 || gpu >= count) return nullptr;
    if ((int64_t)contexts.size() < count) contexts.resize(count, nullptr);
    if (contexts[gpu]) return contexts[gpu];
    int previous = -1;
    hipGetDevice(&previous);
    if (hipSetDevice((int)gpu) != hipSuccess) return nullptr;
    auto *ctx = new DeviceContext();
    ctx->id = (int)gpu;
    hipDeviceProp_t props;
    bool ok = hipGetDeviceProperties(&props, (int)gpu) == hipSuccess;
    if (ok) {
        // Dynamic LDS up to 64 KiB needs no opt-in attribute for a launch.
        ctx->lds_limit = props.sharedMemPerBlock < 65536 ? props.sharedMemPerBlock : 65536;
        ctx->compute_units = props.multiProcessorCount;
    }
    // Default priority only: one ordinary stream per device.
    ok = ok && hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) == hipSuccess;
    ok = ok && hipEventCreate(&ctx->start) == hipSuccess && hipEventCreate(&ctx->stop) == hipSuccess;
    ok = ok && hipEventCreate(&ctx->sweep_start) == hipSuccess && hipEventCreate(&ctx->sweep_stop) == hipSuccess;
    if (previous >= 0) hipSetDevice(previous);
    if (!ok) {
        delete ctx;
        return nullptr;
    }
    contexts[gpu] = ctx;
    return ctx;
}

hipEvent_t DeviceContext::event(size_t i) {
    while (pool.size() <= i) {
        hipEvent_t e = nullptr;
        if (hipEventCreate(&e) != hipSuccess) return nullptr;
        pool.push_back(e);
    }
    return pool[i];
}

hipStream_t DeviceContext::side(size_t i) {
    while (sides.size() <= i) {
        hipStream_t st = nullptr;
        if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess) return nullptr;
        sides.push_back(st);
    }
    return sides[i];
}

hipEvent_t DeviceContext::mark(size_t i) {
    while (marks.size() <= i) {
        hipEvent_t e = nullptr;
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return nullptr;
        marks.push_back(e);
    }
    return marks[i];
}

DeviceGuard::DeviceGuard(const DeviceContext *ctx) {
    hipGetDevice(&previous);
    if (ctx && ctx->id != previous) hipSetDevice(ctx->id);
}

DeviceGuard::~DeviceGuard() {
    if (previous >= 0) hipSetDevice(previous);
}

namespace {
thread_local Carve *active_carve = nullptr;
}  // namespace

void *Carve::take(size_t bytes) {
    const size_t at = (used + 255) & ~size_t(255);
    if (at > size || bytes > size - at) {
        exhausted = true;
        return nullptr;
    }
    used = at + bytes;
    return base + at;
}

bool Carve::flush(DeviceContext *ctx) {
    const size_t bytes = gathered;
    gathered = 0;
    return bytes == 0 || hipMemcpyAsync(base, image, bytes, hipMemcpyHostToDevice, ctx->stream) == hipSuccess;
}

Region DeviceContext::take_region(size_t bytes) {
    const bool small = bytes <= REGION_SMALL;
    if (bytes > REGION_LARGE) return Region{};
    {
        std::lock_guard<std::mutex> hold(regions_lock);
        std::vector<Region> &kept = small ? regions_small : regions_large;
        size_t &out = small ? regions_small_out : regions_large_out;
        if (out >= (small ? REGIONS_SMALL_OUT : REGIONS_LARGE_OUT)) return Region{};
        ++out;
        if (!kept.empty()) {
            const Region region = kept.back();
            kept.pop_back();
            return region;
        }
    }
    Region region;
    region.size = small ? REGION_SMALL : REGION_LARGE;
    if (hipMalloc(reinterpret_cast<void **>(&region.base), region.size) != hipSuccess) {
        (void)hipGetLastError();
        std::lock_guard<std::mutex> hold(regions_lock);
        --(small ? regions_small_out : regions_large_out);
        return Region{};
    }
    if (small && hipHostMalloc(reinterpret_cast<void **>(&region.image), region.size) != hipSuccess) {
        (void)hipGetLastError();
        region.image = nullptr;
    }
    return region;
}

static void free_region(const Region &region) {
    (void)hipFree(region.base);
    if (region.image) (void)hipHostFree(region.image);
}

void DeviceContext::give_region(const Region &region) {
    {
        std::lock_guard<std::mutex> hold(regions_lock);
        const bool small = region.size == REGION_SMALL;
        std::vector<Region> &kept = small ? regions_small : regions_large;
        --(small ? regions_small_out : regions_large_out);
        if (kept.size() < (small ? REGIONS_SMALL : REGIONS_LARGE)) {
            kept.push_back(region);
            return;
        }
    }
    free_region(region);
}

void DeviceContext::drop_regions() {
    std::vector<Region> dropped;
    {
        std::lock_guard<std::mutex> hold(regions_lock);
        dropped.swap(regions_small);
        dropped.insert(dropped.end(), regions_large.begin(), regions_large.end());
        regions_large.clear();
    }
    for (const Region &region : dropped) free_region(region);
}

void give_back(DeviceContext *ctx, const Region &region) {
    std::lock_guard<std::mutex> serial(ctx->lock);
    DeviceGuard guard(ctx);
    (void)hipDeviceSynchronize();
    ctx->give_region(region);
}

// Frees what the current device's context keeps, for an allocation that found no memory.
static void drop_kept_regions() {
    int id = -1;
    if (hipGetDevice(&id) != hipSuccess) return;
    DeviceContext *ctx = nullptr;
    {
        std::lock_guard<std::mutex> lock(contexts_mutex);
        if (id >= 0 && id < (int)contexts.size()) ctx = contexts[id];
    }
    if (ctx) ctx->drop_regions();
}

CarveScope::CarveScope(Carve *carve) : previous(active_carve) { active_carve = carve; }

CarveScope::~CarveScope() { active_carve = previous; }

bool CarveScope::active() { return active_carve != nullptr; }

DeviceBuffer::~DeviceBuffer() {
    if (ptr && !carved) (void)hipFree(ptr);
}

void DeviceBuffer::release() {
    if (ptr && !carved) (void)hipFree(ptr);
    ptr = nullptr;
    size = 0;
    carved = false;
}

bool DeviceBuffer::reserve(size_t bytes) {
    if (bytes <= size && ptr) return true;
    release();
    if (Carve *carve = active_carve) {
        ptr = carve->take(bytes);
        if (!ptr && carve->strict) return false;  // a call that may not allocate
        if (ptr) {
            carved = true;
            size = bytes;
            return true;
        }
    }
    if (hipMalloc(&ptr, bytes) != hipSuccess) {
        drop_kept_regions();
        if (hipMalloc(&ptr, bytes) != hipSuccess) {
            ptr = nullptr;
            return false;
        }
        (void)hipGetLastError();  // the first try's
    }
    size = bytes;
    return true;
}

bool DeviceBuffer::upload(DeviceContext *ctx, const void *host, size_t bytes) {
    if (!reserve(bytes < 4 ? 4 : bytes)) return false;
    if (bytes == 0) return true;
    if (Carve *carve = active_carve; carve && carve->image && carved) {
        const size_t at = static_cast<uint8_t *>(ptr) - carve->base;
        std::memcpy(carve->image + at, host, bytes);
        carve->gathered = std::max(carve->gathered, at + bytes);
        return true;
    }
    return hipMemcpyAsync(ptr, host, bytes, hipMemcpyHostToDevice, ctx->stream) == hipSuccess &&
           hipStreamSynchronize(ctx->stream) == hipSuccess;
}

bool DeviceBuffer::write(DeviceContext *ctx, const void *host, size_t bytes) {
    if (bytes == 0) return true;
    if (bytes > size) return false;
    return hipMemcpyAsync(ptr, host, bytes, hipMemcpyHostToDevice, ctx->stream) == hipSuccess &&
           hipStreamSynchronize(ctx->stream) == hipSuccess;
}

bool DeviceBuffer::read(DeviceContext *ctx, void *host, size_t bytes) const {
    if (bytes == 0) return true;
    if (bytes > size) return false;
    return hipMemcpyAsync(host, ptr, bytes, hipMemcpyDeviceToHost, ctx->stream) == hipSuccess &&
           hipStreamSynchronize(ctx->stream) == hipSuccess;
}

}  // namespace dinara
