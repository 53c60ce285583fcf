// See fake_hip.h.
#include "fake_hip.h"

#include <cstdlib>
#include <cstring>
#include <set>

namespace fake {
namespace {
struct Names {
    std::map<const void *, std::string> of;
};
// Filled by the library's constructors, before this file's own statics.
Names &names() {
    static Names *n = new Names();
    return *n;
}
std::map<const void *, int> &owners() {
    static std::map<const void *, int> *o = new std::map<const void *, int>();
    return *o;
}
thread_local int t_device = 0;
thread_local hipError_t t_error = hipSuccess;
thread_local dim3 t_grid, t_block;
thread_local size_t t_lds = 0;
thread_local hipStream_t t_stream = nullptr;

hipError_t done(hipError_t e) {
    if (e != hipSuccess) t_error = e;
    return e;
}
void own(const void *p) {
    std::lock_guard<std::mutex> lk(rt().m);
    owners()[p] = t_device;
}
void *handle() {
    void *p = std::calloc(1, 64);
    own(p);
    return p;
}
void disown(void *p) {
    {
        std::lock_guard<std::mutex> lk(rt().m);
        owners().erase(p);
    }
    std::free(p);
}
}  // namespace

Runtime &rt() {
    static Runtime *r = new Runtime();
    return *r;
}
int device_of(const void *p) {
    std::lock_guard<std::mutex> lk(rt().m);
    auto it = owners().find(p);
    return it == owners().end() ? -1 : it->second;
}
bool Runtime::was_launched(const std::string &kernel, size_t since) {
    std::lock_guard<std::mutex> lk(m);
    for (size_t q = since; q < launched.size(); q++)
        if (launched[q].find(kernel) != std::string::npos) return true;
    return false;
}
}  // namespace fake

using namespace fake;

extern "C" {

void **__hipRegisterFatBinary(const void *) {
    static void *module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    names().of[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    t_grid = grid; t_block = block; t_lds = lds; t_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    *grid = t_grid; *block = t_block; *lds = t_lds; *s = t_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t s) {
    if (s && device_of(s) != t_device) return done(hipErrorInvalidResourceHandle);
    std::lock_guard<std::mutex> lk(rt().m);
    rt().launched.push_back(names().of[f]);
    return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t l, hipStream_t s, hipEvent_t, hipEvent_t,
                              int) {
    return hipLaunchKernel(f, g, b, a, l, s);
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static char symbol[256];
    *p = symbol;
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    if (d < 0 || d > 1) return done(hipErrorInvalidDevice);
    t_device = d;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = t_device;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = t_error;
    t_error = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "fake error"; }

hipError_t hipMalloc(void **p, size_t bytes) {
    {
        std::lock_guard<std::mutex> lk(rt().m);
        if (rt().in_use + bytes > rt().limit) return done(hipErrorOutOfMemory);
    }
    *p = std::calloc(bytes, 1);
    own(*p);
    std::lock_guard<std::mutex> lk(rt().m);
    rt().device[*p] = bytes;
    rt().in_use += bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    {
        std::lock_guard<std::mutex> lk(rt().m);
        auto it = rt().device.find(p);
        if (it == rt().device.end()) std::abort();  // freed twice, or never allocated
        rt().in_use -= it->second;
        rt().device.erase(it);
    }
    disown(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    if (rt().pinned_fails) return done(hipErrorOutOfMemory);
    *p = std::calloc(bytes, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t) {
    std::memcpy(dst, src, bytes);
    if (kind == hipMemcpyDeviceToHost && rt().on_download) rt().on_download(dst, bytes);
    return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind) {
    return hipMemcpyAsync(dst, src, bytes, kind, nullptr);
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = static_cast<hipStream_t>(handle());
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    disown(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    if (rt().on_stream_wait) rt().on_stream_wait(s);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = static_cast<hipEvent_t>(handle());
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) {
    disown(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (s && device_of(e) != device_of(s)) return done(hipErrorInvalidResourceHandle);
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    *g = static_cast<hipGraph_t>(handle());
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *x = static_cast<hipGraphExec_t>(handle());
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    disown(g);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
    disown(x);
    return hipSuccess;
}

}  // extern "C"
