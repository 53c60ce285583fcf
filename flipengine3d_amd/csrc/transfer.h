// Memory the contexts of a device share: pinned staging for device-to-host
// copies and the device memory that stage calls work in.
#pragma once

#include <hip/hip_runtime.h>

#include <map>
#include <memory>
#include <mutex>
#include <vector>

namespace flipmi {

// Makes a device current while it is alive.
class DeviceScope {
public:
    explicit DeviceScope(int device) {
        changed = hipGetDevice(&was) == hipSuccess && was != device && hipSetDevice(device) == hipSuccess;
    }
    ~DeviceScope() {
        if (changed) (void)hipSetDevice(was);
    }
    DeviceScope(const DeviceScope &) = delete;
    DeviceScope &operator=(const DeviceScope &) = delete;

private:
    int was = 0;
    bool changed = false;
};

// Copies device memory to pageable host memory through a ring of pinned
// chunks: the copy engine fills one chunk while host threads empty others.
// (Straight into pageable memory the runtime reaches 10 to 17 GB/s here,
// most of it spent faulting the caller's fresh pages in on one thread; the
// engine alone moves 55 GB/s.)  Small results are staged in a slab of the
// caller's own.  A caller waits for its stream holding nothing, and for the
// ring only while another's data crosses.  Both are allocated with the first
// copy that uses them.  The caller's current device may be another.
struct HostPiece {
    void *dst;
    const void *src;
    size_t bytes;
};
class HostLink {
public:
    explicit HostLink(int on) : device(on) {}
    HostLink(const HostLink &) = delete;
    HostLink &operator=(const HostLink &) = delete;
    ~HostLink() { release(); }
    // Returns when dst holds the data.  Ordered after the work on s.
    hipError_t to_host(void *dst, const void *src, size_t bytes, hipStream_t s) {
        const HostPiece p{dst, src, bytes};
        return to_host(&p, 1, s);
    }
    // Several results at once: the small ones wait for the device together.
    hipError_t to_host(const HostPiece *pieces, int count, hipStream_t s);
    // Pinned host memory of kPage bytes, for one caller at a time.
    static constexpr size_t kPage = 4096;
    hipError_t get_page(void **p) { return take(pages, kPage, p); }
    void put_page(void *p) { give(pages, kPages, p); }
    void release();

private:
    static constexpr size_t kChunk = (size_t)2 << 20;
    static constexpr int kSlots = 16;
    // A stage call has ten results at most, each under the size that takes the
    // ring when it is small: they all fit one slab.
    static constexpr size_t kSlab = (size_t)5 << 19;
    static constexpr size_t kSlabs = 8, kPages = 64;  // kept idle
    const int device;
    bool ready();
    hipError_t large(const HostPiece &p, hipStream_t s);
    // A block of pinned memory from those kept in `idle`, or a new one.
    hipError_t take(std::vector<void *> &idle, size_t bytes, void **p);
    void give(std::vector<void *> &idle, size_t most, void *p);
    std::mutex m;       // the ring
    std::mutex idle_m;  // the lists below
    char *ring = nullptr;
    hipEvent_t filled[kSlots] = {};
    std::vector<void *> slabs, pages;
};

// Device blocks kept between stage calls, at most kHeld bytes of them; the
// rest goes back to the device, as all of it does when an allocation fails
// here or in device_alloc.  Safe from several threads.
class DevicePool {
public:
    explicit DevicePool(int on) : device(on) {}
    DevicePool(const DevicePool &) = delete;
    DevicePool &operator=(const DevicePool &) = delete;
    ~DevicePool() { release(); }
    hipError_t get(size_t bytes, void **p, size_t *size);
    void put(void *p, size_t size);
    void release();

private:
    static constexpr size_t kHeld = (size_t)1 << 30;
    const int device;
    std::mutex m;
    std::multimap<size_t, void *> blocks;
    size_t held = 0;
};

// While one is alive, the device buffers its thread allocates come from the
// pool.  All their uses are on one stream, so a buffer given back is reused
// within the call as it is; the pool gets it when the stream is idle, and the
// device when an allocation fails.  The scope outlives its buffers.
class PoolScope {
public:
    PoolScope(DevicePool &pool, hipStream_t s);
    ~PoolScope();
    PoolScope(const PoolScope &) = delete;
    PoolScope &operator=(const PoolScope &) = delete;
    static PoolScope *current();
    // While one is alive, buffers are allocated as outside any scope (those
    // that outlive the call).
    class Off {
    public:
        Off();
        ~Off();

    private:
        PoolScope *was;
    };
    hipError_t get(size_t bytes, void **p, size_t *size);
    void put(void *p, size_t size) noexcept;  // from destructors

private:
    DevicePool &pool;
    hipStream_t stream;
    PoolScope *outer;
    std::multimap<size_t, void *> back;
};

// Held by every context of a device, freed with the last of them.
struct DeviceShared {
    explicit DeviceShared(int device) : link(device), pool(device) {}
    HostLink link;
    DevicePool pool;
    static std::shared_ptr<DeviceShared> of(int device);
    // Null where no context holds one.
    static std::shared_ptr<DeviceShared> find(int device);
};

// hipMalloc on the current device, which has what the device's pool holds idle
// before it reports that the memory is out.
hipError_t device_alloc(void **p, size_t bytes);

}  // namespace flipmi
