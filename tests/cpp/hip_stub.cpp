// A host stand-in for the HIP calls libtsl.so makes, for CPU tests of its host
// paths: device memory is host memory, kernels do nothing, and an asynchronous
// copy runs only when something waits for it, so that a test can see which
// copies a call left behind.  Loaded with global visibility before libtsl.so;
// what is not defined here stays the runtime's own.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

namespace {

struct Copy {
    void* dst;
    const void* src;
    size_t n;
    const void* host;  // the host side
};

std::recursive_mutex mu;
std::map<const char*, size_t> device, pinned;
std::vector<Copy> queue;
size_t total = (size_t)288 << 30, live = 0;
long launches_left = -1, copies_left = -1;  // launches, asynchronous copies until one fails (-1: none does)
hipError_t last = hipSuccess;
bool no_pinned = false;
int timings = 0, launches = 0;

hipError_t note(hipError_t e)
{
    if (e != hipSuccess) last = e;
    return e;
}

bool inside(const std::map<const char*, size_t>& m, const void* p)
{
    auto it = m.upper_bound(static_cast<const char*>(p));
    if (it == m.begin()) return false;
    --it;
    return static_cast<const char*>(p) < it->first + it->second;
}

void drain()
{
    for (const Copy& c : queue) std::memcpy(c.dst, c.src, c.n);
    queue.clear();
}

}  // namespace

#define LOCK std::lock_guard<std::recursive_mutex> lock(mu)

extern "C" {

size_t stub_live_bytes() { LOCK; return live; }
void stub_set_total(size_t bytes) { LOCK; total = bytes; }
void stub_fail_launch(long after) { LOCK; launches_left = after; last = hipSuccess; }
void stub_fail_copy(long after) { LOCK; copies_left = after; last = hipSuccess; }
void stub_no_pinned(int on) { LOCK; no_pinned = on != 0; }
// event pairs measured since the last call
int stub_timings() { LOCK; const int n = timings; timings = 0; return n; }
// kernels launched since the last call
int stub_launches() { LOCK; const int n = launches; launches = 0; return n; }
// queued copies that read or write the caller's memory
int stub_pending()
{
    LOCK;
    int n = 0;
    for (const Copy& c : queue) n += !inside(pinned, c.host);
    return n;
}

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipGetLastError() { LOCK; const hipError_t e = last; last = hipSuccess; return e; }

hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeWarpSize ? 64 : 1024;
    return hipSuccess;
}

hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    return hipSuccess;
}

hipError_t hipMemGetInfo(size_t* free_bytes, size_t* total_bytes)
{
    LOCK;
    *free_bytes = total - live;
    *total_bytes = total;
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n)
{
    LOCK;
    if (live + n > total) return note(hipErrorOutOfMemory);
    *p = std::calloc(n ? n : 1, 1);
    device[static_cast<char*>(*p)] = n;
    live += n;
    return hipSuccess;
}

hipError_t hipFree(void* p)
{
    LOCK;
    drain();
    auto it = device.find(static_cast<char*>(p));
    if (it == device.end()) return hipSuccess;
    live -= it->second;
    device.erase(it);
    std::free(p);
    return hipSuccess;
}

hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    LOCK;
    if (no_pinned) return note(hipErrorOutOfMemory);
    *p = std::calloc(n ? n : 1, 1);
    pinned[static_cast<char*>(*p)] = n;
    return hipSuccess;
}

hipError_t hipHostFree(void* p)
{
    LOCK;
    drain();
    pinned.erase(static_cast<char*>(p));
    std::free(p);
    return hipSuccess;
}

hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static void* scratch = std::calloc((size_t)64 << 20, 1);
    *p = scratch;
    return hipSuccess;
}

hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t)
{
    LOCK;
    if (copies_left == 0) {
        copies_left = -1;
        return note(hipErrorUnknown);
    }
    if (copies_left > 0) --copies_left;
    if (kind == hipMemcpyDeviceToDevice) {
        drain();
        std::memcpy(dst, src, n);
    } else {
        queue.push_back(Copy{dst, src, n, kind == hipMemcpyHostToDevice ? src : dst});
    }
    return hipSuccess;
}

hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind)
{
    LOCK;
    drain();
    std::memcpy(dst, src, n);
    return hipSuccess;
}

hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t)
{
    LOCK;
    drain();
    std::memset(p, v, n);
    return hipSuccess;
}

hipError_t hipDeviceSynchronize() { LOCK; drain(); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { LOCK; drain(); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = reinterpret_cast<hipStream_t>(std::malloc(1)); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { LOCK; drain(); std::free(s); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = reinterpret_cast<hipEvent_t>(std::malloc(1)); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { LOCK; drain(); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { LOCK; drain(); return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { LOCK; ++timings; *ms = 1.0f; return hipSuccess; }

hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) { std::memset(a, 0, sizeof(*a)); return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return hipSuccess; }

hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s)
{
    *g = *b = dim3();
    *lds = 0;
    *s = nullptr;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t)
{
    LOCK;
    if (launches_left == 0) {
        launches_left = -1;
        return note(hipErrorLaunchFailure);
    }
    if (launches_left > 0) --launches_left;
    ++launches;
    return hipSuccess;
}

}  // extern "C"
