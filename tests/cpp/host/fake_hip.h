// A HIP runtime without a device, for tests of what the library does on the
// host.  An executable that defines these functions comes before libamdhip64 in
// the symbol search, so libflipmi.so calls them: memory is host memory (zeroed),
// copies are made at once, kernels are noted by name and do nothing.  There are
// two devices; what belongs to one is refused where the other is current, as
// HIP does for launches and event records.
#pragma once

#include <hip/hip_runtime.h>

#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace fake {

struct Runtime {
    std::mutex m;
    std::vector<std::string> launched;    // kernels, in order
    std::map<void *, size_t> device;      // allocations, bytes
    size_t in_use = 0, limit = ~(size_t)0;
    bool pinned_fails = false;
    // After a device-to-host copy of `bytes` to dst.
    std::function<void(void *dst, size_t bytes)> on_download;
    // Before a stream is waited for.
    std::function<void(hipStream_t)> on_stream_wait;
    bool was_launched(const std::string &kernel, size_t since = 0);
};
Runtime &rt();
// The device that holds an allocation, stream or event, or -1.
int device_of(const void *p);

}  // namespace fake
