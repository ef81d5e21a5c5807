// The HIP calls backend.cpp makes, on the host, for tests of its ordering and
// of its error paths without a GPU. Streams are queues that run as late as the
// calls allow: work starts only when the host waits for it (or frees memory),
// so whatever the host changes without a wait, the queued work sees changed.
// Device memory is host memory, filled with NaN bits at allocation.
#pragma once
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <deque>
#include <functional>
#include <map>
#include <vector>

#define __device__
#define __align__(n) __attribute__((aligned(n)))
#define HIP_SYMBOL(x) (&(x))

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost, hipMemcpyDeviceToDevice };
enum hipMemoryType { hipMemoryTypeUnregistered, hipMemoryTypeHost, hipMemoryTypeDevice };
enum {
    hipHostMallocDefault = 0,
    hipStreamNonBlocking = 1,
    hipEventDisableTiming = 2,
    hipEventDisableSystemFence = 4,
    hipStreamCaptureModeThreadLocal = 1
};
typedef void *hipDeviceptr_t;
typedef void *hipGraph_t;
typedef void *hipGraphExec_t;
struct hipDeviceProp_t {
    char name[64], gcnArchName[64];
    int multiProcessorCount;
    size_t totalGlobalMem;
};
struct hipPointerAttribute_t {
    hipMemoryType type;
    int device;
    void *devicePointer;
};

namespace host {
struct Stream {
    std::deque<std::function<void()>> work;
    uint64_t queued = 0, done = 0;
    void add(std::function<void()> f) {
        work.push_back(std::move(f));
        ++queued;
    }
    void run(uint64_t upto) {
        while (done < upto) {
            std::function<void()> f = std::move(work.front());
            work.pop_front();
            ++done;
            f();
        }
    }
};
struct Event {
    Stream *stream = nullptr;
    uint64_t at = 0;
};
inline std::vector<Stream *> streams;
inline std::map<char *, size_t> pinned, device;
inline size_t device_bytes = 0, device_limit = ~(size_t)0;
inline void run_all() {
    for (Stream *s : streams) s->run(s->queued);
}
inline const std::pair<char *const, size_t> *find(const std::map<char *, size_t> &m, const void *p) {
    auto it = m.upper_bound((char *)p);
    if (it == m.begin()) return nullptr;
    --it;
    return (char *)p < it->first + it->second ? &*it : nullptr;
}
}  // namespace host
typedef host::Stream *hipStream_t;
typedef host::Event *hipEvent_t;

// Also what synthetic.c allocates pinned host arrays with.
extern "C" inline __attribute__((used)) hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = malloc(n ? n : 1);
    host::pinned[(char *)*p] = n ? n : 1;
    return hipSuccess;
}
extern "C" inline __attribute__((used)) hipError_t hipHostFree(void *p) {
    host::run_all();
    host::pinned.erase((char *)p);
    free(p);
    return hipSuccess;
}
inline hipError_t hipMalloc(void **p, size_t n) {
    if (n > host::device_limit - host::device_bytes) return hipErrorOutOfMemory;
    *p = malloc(n);
    memset(*p, 0xff, n);
    host::device[(char *)*p] = n;
    host::device_bytes += n;
    return hipSuccess;
}
inline hipError_t hipFree(void *p) {
    host::run_all();
    auto it = host::device.find((char *)p);
    if (it == host::device.end()) return hipErrorInvalidValue;
    host::device_bytes -= it->second;
    host::device.erase(it);
    free(p);
    return hipSuccess;
}
inline hipError_t hipMemGetInfo(size_t *free_bytes, size_t *total) {
    *total = host::device_limit;
    *free_bytes = host::device_limit - host::device_bytes;
    return hipSuccess;
}
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    memcpy(d, s, n);
    return hipSuccess;
}
inline hipError_t hipMemset(void *d, int v, size_t n) {
    memset(d, v, n);
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
    st->add([=] { memmove(d, s, n); });
    return hipSuccess;
}
inline hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h,
                                   hipMemcpyKind, hipStream_t st) {
    st->add([=] {
        for (size_t i = 0; i < h; ++i) memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
    });
    return hipSuccess;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    host::streams.push_back(*s = new host::Stream());
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) {
    host::run_all();
    host::streams.erase(std::find(host::streams.begin(), host::streams.end(), s));
    delete s;
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    s->run(s->queued);
    return hipSuccess;
}
inline hipError_t hipDeviceSynchronize() {
    host::run_all();
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = new host::Event();
    return hipSuccess;
}
inline hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    *e = {s, s->queued};
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    if (e->stream) e->stream->run(e->at);
    return hipSuccess;
}
inline hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    const host::Event seen = *e;
    s->add([=] {
        if (seen.stream) seen.stream->run(seen.at);
    });
    return hipSuccess;
}
inline hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}
// Steps are launched eagerly here (PLAMO_HIP_EAGER_DECODE=1): no graphs.
inline hipError_t hipStreamBeginCapture(hipStream_t, int) { return hipErrorInvalidValue; }
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorInvalidValue; }
inline hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, void *, void *, int) {
    return hipErrorInvalidValue;
}
inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorInvalidValue; }
inline hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char *hipGetErrorString(hipError_t) { return "injected error"; }
inline hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->name, "host");
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->totalGlobalMem = 1ull << 38;
    return hipSuccess;
}
inline hipError_t hipGetSymbolAddress(void **p, const void *s) {
    *p = (void *)s;
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    *a = {hipMemoryTypeUnregistered, 0, nullptr};
    if (host::find(host::pinned, p)) *a = {hipMemoryTypeHost, 0, (void *)p};
    if (host::find(host::device, p)) *a = {hipMemoryTypeDevice, 0, (void *)p};
    return hipSuccess;
}
inline hipError_t hipMemGetAddressRange(hipDeviceptr_t *base, size_t *size, hipDeviceptr_t p) {
    auto *r = host::find(host::device, p);
    if (!r) return hipErrorInvalidValue;
    *base = r->first;
    *size = r->second;
    return hipSuccess;
}
