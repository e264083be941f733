// The HIP entry points that libgpunb.so calls, on the CPU, for tests of its
// host paths: device and pinned memory are zeroed heap blocks, copies run when
// they are called, kernels do not run.  Loaded with RTLD_GLOBAL before the
// library, whose calls then come here.
//
// stub_* below: allocations that fail, and what the library did.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>

namespace {

std::mutex mu;
size_t most_device = SIZE_MAX;   // a larger hipMalloc fails
size_t most_pinned = SIZE_MAX;   // a larger hipHostMalloc fails
int fail_uploads = 0;            // that many host-to-device copies fail
int fail_new = -1;               // operator new fails after so many calls
size_t held_device = 0;          // bytes of device memory not freed
int allocations = 0;             // of device and pinned memory
bool graph_running = false;      // launched, and not waited for since
int graph_faults = 0;            // executable graphs destroyed while running
int null_args = 0;               // launches of k_irr_stage without its data
hipError_t last_error = hipSuccess;
std::map<void *, size_t> blocks;
std::map<const void *, std::string> names;
std::map<std::string, int> launches;

void *take(size_t bytes) { return calloc(1, bytes ? bytes : 1); }

// The data pointers of k_irr_stage's argument, as irr.hip declares it.
struct StageHead {
    int nj, nr, ni;
    unsigned bj, bl;
    const double *soa;
    const int *slot;
    void *jp;
    const int *hdr, *flat;
};

hipError_t launched(const void *fn, void **args) {
    std::lock_guard<std::mutex> g(mu);
    const std::string &name = names[fn];
    ++launches[name];
    if (name.find("k_irr_stage") != std::string::npos) {
        const StageHead &s = *(const StageHead *)args[0];
        if (s.nj > 0 && (!s.soa || (uintptr_t)s.soa < 4096)) ++null_args;
        if (s.nr > 0 && (!s.hdr || (uintptr_t)s.hdr < 4096)) ++null_args;
    }
    return hipSuccess;
}

thread_local dim3 cfg_grid, cfg_block;
thread_local size_t cfg_lds;
thread_local hipStream_t cfg_stream;

}  // namespace

extern "C" {

void stub_most_device(size_t bytes) { most_device = bytes; }
void stub_most_pinned(size_t bytes) { most_pinned = bytes; }
void stub_fail_uploads(int n) { fail_uploads = n; }
void stub_fail_new(int n) { fail_new = n; }
size_t stub_held_device() { return held_device; }
int stub_allocations() { return allocations; }
int stub_graph_faults() { return graph_faults; }
int stub_null_args() { return null_args; }
int stub_launches(const char *part) {
    int n = 0;
    for (const auto &l : launches)
        if (l.first.find(part) != std::string::npos) n += l.second;
    return n;
}

void **__hipRegisterFatBinary(const void *) {
    static void *module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *fn, char *, const char *name,
                           unsigned, void *, void *, void *, void *, int *) {
    std::lock_guard<std::mutex> g(mu);
    names[fn] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds,
                                      hipStream_t st) {
    cfg_grid = grid, cfg_block = block, cfg_lds = lds, cfg_stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds,
                                     hipStream_t *st) {
    *grid = cfg_grid, *block = cfg_block, *lds = cfg_lds, *st = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3, dim3, void **args, size_t,
                           hipStream_t) {
    return launched(fn, args);
}

hipError_t hipMalloc(void **p, size_t bytes) {
    std::lock_guard<std::mutex> g(mu);
    ++allocations;
    *p = bytes <= most_device ? take(bytes) : nullptr;
    if (!*p) return last_error = hipErrorOutOfMemory;
    blocks[*p] = bytes;
    held_device += bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> g(mu);
    const auto b = blocks.find(p);
    if (b != blocks.end()) {
        held_device -= b->second;
        blocks.erase(b);
    }
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    ++allocations;
    *p = bytes <= most_pinned ? take(bytes) : nullptr;
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
    free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) {
    *d = h;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes,
                          hipMemcpyKind kind, hipStream_t) {
    {
        std::lock_guard<std::mutex> g(mu);
        if (kind == hipMemcpyHostToDevice && fail_uploads > 0) {
            --fail_uploads;
            return hipErrorUnknown;
        }
    }
    if (bytes) memcpy(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipMemcpyWithStream(void *dst, const void *src, size_t bytes,
                               hipMemcpyKind kind, hipStream_t st) {
    return hipMemcpyAsync(dst, src, bytes, kind, st);
}
hipError_t hipMemsetAsync(void *p, int v, size_t bytes, hipStream_t) {
    memset(p, v, bytes);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *st, unsigned) {
    *st = (hipStream_t)take(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t st) {
    free(st);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    graph_running = false;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *ev) {
    *ev = (hipEvent_t)take(1);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *ev, unsigned) {
    return hipEventCreate(ev);
}
hipError_t hipEventDestroy(hipEvent_t ev) {
    free(ev);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    *g = (hipGraph_t)take(1);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *,
                               char *, size_t) {
    *e = (hipGraphExec_t)take(1);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) {
    graph_running = true;
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    if (graph_running) ++graph_faults;
    free(e);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    free(g);
    return hipSuccess;
}

hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    *p = take(64u << 20);
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int,
                                                        size_t) {
    *n = 4;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) {
    return e == hipErrorOutOfMemory ? "out of memory" : "error";
}

}  // extern "C"

// The library's heap allocations come here too.
void *operator new(size_t bytes) {
    if (fail_new >= 0 && fail_new-- == 0) throw std::bad_alloc();
    void *p = malloc(bytes ? bytes : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }
