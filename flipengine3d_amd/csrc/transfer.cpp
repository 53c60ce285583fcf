// See transfer.h.
#include "transfer.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

namespace flipmi {

namespace {
// Below this a result is small: one copy into a slab; the ring gains nothing.
constexpr size_t kDirect = (size_t)256 << 10;
// Threads that empty the ring, for copies that are worth starting them (about
// 30 us each).  226 MB of particles in two copies: 59 ms as six pageable copies
// and a loop over the triples, 6.6 ms so (34 GB/s, page faults included).
constexpr size_t kThreaded = (size_t)8 << 20;
constexpr int kCopyThreads = 6;

// Sizes in steps of an eighth of a power of two, 64 KiB at least, so that
// calls of nearly the same sizes share blocks.
size_t block_size(size_t bytes) {
    size_t step = (size_t)8 << 10;
    while (step * 16 <= bytes) step *= 2;
    return std::max((bytes + step - 1) / step * step, (size_t)64 << 10);
}

thread_local PoolScope *t_scope = nullptr;
}  // namespace

// ---------------------------------------------------------------------------
// HostLink
// ---------------------------------------------------------------------------

bool HostLink::ready() {
    if (ring) return true;
    hipError_t e = hipSuccess;
    for (int q = 0; q < kSlots && e == hipSuccess; q++)
        if (!filled[q]) e = hipEventCreateWithFlags(&filled[q], hipEventDisableTiming);
    void *p = nullptr;
    if (e == hipSuccess) e = hipHostMalloc(&p, kChunk * kSlots, hipHostMallocDefault);
    if (e == hipSuccess) ring = static_cast<char *>(p);
    else (void)hipGetLastError();  // plain copies do: no launch is to report it
    return ring != nullptr;
}

void HostLink::release() {
    for (auto *idle : {&pages, &slabs}) {
        for (void *p : *idle) (void)hipHostFree(p);
        idle->clear();
    }
    if (ring) (void)hipHostFree(ring);
    ring = nullptr;
    for (hipEvent_t &e : filled) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
}

hipError_t HostLink::take(std::vector<void *> &idle, size_t bytes, void **p) {
    {
        std::lock_guard<std::mutex> lk(idle_m);
        if (!idle.empty()) {
            *p = idle.back();
            idle.pop_back();
            return hipSuccess;
        }
    }
    const DeviceScope on(device);
    const hipError_t e = hipHostMalloc(p, bytes, hipHostMallocDefault);
    if (e != hipSuccess) (void)hipGetLastError();  // reported here, not by the next launch
    return e;
}

void HostLink::give(std::vector<void *> &idle, size_t most, void *p) {
    {
        std::lock_guard<std::mutex> lk(idle_m);
        if (idle.size() < most) {
            try {
                idle.push_back(p);
                return;
            } catch (...) {
            }
        }
    }
    (void)hipHostFree(p);
}

hipError_t HostLink::to_host(const HostPiece *pieces, int count, hipStream_t s) {
    const DeviceScope on(device);
    // The small pieces go through a slab as far as it reaches; the rest of them,
    // and all without one, are plain copies.
    auto small = [](const HostPiece &p) { return p.bytes > 0 && p.bytes < kDirect; };
    auto room = [](size_t bytes) { return (bytes + 63) & ~(size_t)63; };
    void *block = nullptr;
    bool any = false;
    for (int q = 0; q < count; q++) any |= small(pieces[q]);
    if (any && take(slabs, kSlab, &block) != hipSuccess) block = nullptr;
    char *const slab = static_cast<char *>(block);
    size_t at = 0;
    hipError_t e = hipSuccess;
    for (int q = 0; q < count && e == hipSuccess; q++) {
        const HostPiece &p = pieces[q];
        if (!small(p)) continue;
        const bool staged = slab && at + p.bytes <= kSlab;
        e = hipMemcpyAsync(staged ? (void *)(slab + at) : p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, s);
        if (staged) at += room(p.bytes);
    }
    const hipError_t w = hipStreamSynchronize(s);
    if (e == hipSuccess) e = w;
    at = 0;
    for (int q = 0; q < count && slab && e == hipSuccess; q++) {
        const HostPiece &p = pieces[q];
        if (!small(p) || at + p.bytes > kSlab) continue;
        std::memcpy(p.dst, slab + at, p.bytes);
        at += room(p.bytes);
    }
    if (slab) give(slabs, kSlabs, slab);
    for (int q = 0; q < count && e == hipSuccess; q++) {
        const HostPiece &p = pieces[q];
        if (p.bytes < kDirect) continue;
        std::lock_guard<std::mutex> lk(m);
        if (ready()) {
            e = large(p, s);
        } else {
            e = hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, s);
            const hipError_t done = hipStreamSynchronize(s);
            if (e == hipSuccess) e = done;
        }
    }
    return e;
}

hipError_t HostLink::large(const HostPiece &piece, hipStream_t s) {
    void *const dst = piece.dst;
    const void *const src = piece.src;
    const size_t bytes = piece.bytes;
    const int n = (int)((bytes + kChunk - 1) / kChunk);
    std::atomic<int> queued{0}, failed{0};
    std::atomic<int> emptied[kSlots];  // the last chunk copied out of each slot
    for (auto &e : emptied) e.store(-1);
    auto fill = [&](int c) -> hipError_t {
        const size_t at = (size_t)c * kChunk, len = std::min(kChunk, bytes - at);
        hipError_t e = hipMemcpyAsync(ring + (size_t)(c % kSlots) * kChunk, static_cast<const char *>(src) + at, len,
                                      hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipEventRecord(filled[c % kSlots], s) : e;
    };
    auto empty = [&](int c) {
        hipError_t e = hipEventSynchronize(filled[c % kSlots]);
        if (e != hipSuccess) {
            failed.store((int)e);
            return;
        }
        const size_t at = (size_t)c * kChunk;
        std::memcpy(static_cast<char *>(dst) + at, ring + (size_t)(c % kSlots) * kChunk, std::min(kChunk, bytes - at));
        emptied[c % kSlots].store(c, std::memory_order_release);
    };
    // Worker t empties chunks t, t + nt, ...; this thread fills them, and is
    // worker 0 in between.
    const int want = bytes >= kThreaded ? std::min(kCopyThreads, (int)std::max(1u, std::thread::hardware_concurrency())) : 1;
    std::vector<std::thread> workers;
    std::atomic<int> nt{want};
    std::atomic<bool> go{false};
    auto work = [&](int t) {
        (void)hipSetDevice(device);
        while (!go.load(std::memory_order_acquire)) std::this_thread::yield();
        for (int c = t; c < n; c += nt.load()) {
            while (queued.load(std::memory_order_acquire) <= c && !failed.load()) std::this_thread::yield();
            if (failed.load()) return;
            empty(c);
        }
    };
    try {
        for (int t = 1; t < want; t++) workers.emplace_back(work, t);
    } catch (...) {
        // Fewer threads share the chunks.
    }
    nt.store((int)workers.size() + 1);
    go.store(true, std::memory_order_release);
    hipError_t err = hipSuccess;
    int next = 0, mine = 0;  // next chunk to fill, next of this thread's to empty
    while ((next < n || mine < n) && !failed.load()) {
        if (next < n && (next < kSlots || emptied[next % kSlots].load(std::memory_order_acquire) == next - kSlots)) {
            err = fill(next);
            if (err != hipSuccess) {
                failed.store((int)err);
                break;
            }
            queued.store(++next, std::memory_order_release);
            continue;
        }
        if (mine < next) {
            empty(mine);
            mine += nt.load();
        } else if (next < n) {
            std::this_thread::yield();
        } else {
            break;
        }
    }
    for (std::thread &t : workers) t.join();
    if (failed.load()) {
        (void)hipStreamSynchronize(s);  // no copy into the ring is left behind
        return (hipError_t)failed.load();
    }
    return hipSuccess;
}

// ---------------------------------------------------------------------------
// Device memory of stage calls
// ---------------------------------------------------------------------------

hipError_t DevicePool::get(size_t bytes, void **p, size_t *size) {
    const size_t want = block_size(bytes);
    const DeviceScope on(device);
    {
        std::lock_guard<std::mutex> lk(m);
        auto it = blocks.lower_bound(want);
        if (it != blocks.end() && it->first <= want + want / 4) {
            *p = it->second;
            *size = it->first;
            held -= it->first;
            blocks.erase(it);
            return hipSuccess;
        }
    }
    *size = want;
    hipError_t e = hipMalloc(p, want);
    if (e == hipSuccess) return e;
    release();
    e = hipMalloc(p, want);
    if (e != hipSuccess) {
        *size = bytes;  // the step may be what does not fit
        e = hipMalloc(p, bytes);
    }
    (void)hipGetLastError();  // reported here, not by the next launch
    return e;
}

void DevicePool::put(void *p, size_t size) {
    {
        std::lock_guard<std::mutex> lk(m);
        if (held + size <= kHeld) {
            try {
                blocks.insert({size, p});
                held += size;
                return;
            } catch (...) {
            }
        }
    }
    (void)hipFree(p);
}

void DevicePool::release() {
    std::multimap<size_t, void *> all;
    {
        std::lock_guard<std::mutex> lk(m);
        all.swap(blocks);
        held = 0;
    }
    for (auto &b : all) (void)hipFree(b.second);
}

PoolScope::PoolScope(DevicePool &p, hipStream_t s) : pool(p), stream(s), outer(t_scope) { t_scope = this; }

PoolScope::~PoolScope() {
    t_scope = outer;
    if (back.empty()) return;
    (void)hipStreamSynchronize(stream);  // a call that failed may have left work behind
    for (auto &b : back) pool.put(b.second, b.first);
}

void PoolScope::put(void *p, size_t size) noexcept {
    try {
        back.insert({size, p});
    } catch (...) {
        (void)hipStreamSynchronize(stream);  // its last use may still run
        (void)hipFree(p);
    }
}

PoolScope *PoolScope::current() { return t_scope; }
PoolScope::Off::Off() : was(t_scope) { t_scope = nullptr; }
PoolScope::Off::~Off() { t_scope = was; }

namespace {
std::mutex g_shared_mutex;
std::map<int, std::weak_ptr<DeviceShared>> &all_shared() {
    static std::map<int, std::weak_ptr<DeviceShared>> all;
    return all;
}
}  // namespace

std::shared_ptr<DeviceShared> DeviceShared::of(int device) {
    std::lock_guard<std::mutex> lk(g_shared_mutex);
    std::weak_ptr<DeviceShared> &held = all_shared()[device];
    std::shared_ptr<DeviceShared> p = held.lock();
    if (!p) {
        p = std::make_shared<DeviceShared>(device);
        held = p;
    }
    return p;
}

std::shared_ptr<DeviceShared> DeviceShared::find(int device) {
    std::lock_guard<std::mutex> lk(g_shared_mutex);
    auto it = all_shared().find(device);
    return it == all_shared().end() ? nullptr : it->second.lock();
}

hipError_t device_alloc(void **p, size_t bytes) {
    hipError_t e = hipMalloc(p, bytes);
    int device = 0;
    if (e == hipSuccess || hipGetDevice(&device) != hipSuccess) return e;
    const std::shared_ptr<DeviceShared> shared = DeviceShared::find(device);
    if (shared) {
        shared->pool.release();
        e = hipMalloc(p, bytes);
    }
    (void)hipGetLastError();  // reported here, not by the next launch
    return e;
}

hipError_t PoolScope::get(size_t bytes, void **p, size_t *size) {
    const size_t want = block_size(bytes);
    auto it = back.lower_bound(want);
    if (it != back.end() && it->first <= want + want / 4) {
        *p = it->second;
        *size = it->first;
        back.erase(it);
        return hipSuccess;
    }
    hipError_t e = pool.get(bytes, p, size);
    if (e != hipSuccess && !back.empty()) {
        (void)hipStreamSynchronize(stream);
        for (auto &b : back) (void)hipFree(b.second);
        back.clear();
        e = pool.get(bytes, p, size);
    }
    return e;
}

}  // namespace flipmi
