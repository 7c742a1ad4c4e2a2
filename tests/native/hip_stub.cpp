// A HIP runtime without a GPU, for tests of the engine's host side: device memory is host memory, copies happen at once,
// streams and events are names, and a kernel launch only leaves a line in a log.  Loaded in front of the engine's library
// (RTLD_GLOBAL), in a process of its own.
#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include <sys/mman.h>

#include <map>
#include <string>

namespace {

size_t g_total = (size_t)288 << 30, g_used = 0, g_peak = 0;
std::map<void *, size_t> g_allocs;
std::map<const void *, std::string> g_kernels;
std::map<std::string, long> g_launches;
std::string g_log; // kernel, grid and block of every launch, a line each
dim3 g_grid, g_block;
long g_uploads = 0, g_replays = 0;
bool g_capturing = false; // launches are being recorded into a graph: nothing may be allocated or waited for

hipError_t map_memory(void **p, size_t bytes)
{
    bytes = (bytes + 4095) & ~(size_t)4095;
    *p = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if(*p == MAP_FAILED)
        return hipErrorOutOfMemory;
    g_allocs[*p] = bytes;
    return hipSuccess;
}

hipError_t unmap_memory(void *p, bool device)
{
    auto it = g_allocs.find(p);
    if(it == g_allocs.end())
        return p ? hipErrorInvalidValue : hipSuccess;
    if(device)
        g_used -= it->second;
    munmap(p, it->second);
    g_allocs.erase(it);
    return hipSuccess;
}

template <typename H> hipError_t new_handle(H *h)
{
    *h = (H) new char;
    return hipSuccess;
}

}  // namespace

extern "C" {

void hipstub_set_memory(size_t total) { g_total = total; }
size_t hipstub_used(void) { return g_used; }
size_t hipstub_peak(void) // since the last question
{
    const size_t p = g_peak;
    g_peak = g_used;
    return p;
}
long hipstub_launches(const char *kernel) // of kernels whose name contains this
{
    long n = 0;
    for(const auto &kv : g_launches)
        if(kv.first.find(kernel) != std::string::npos)
            n += kv.second;
    return n;
}

const char *hipstub_log(void) // since the last question
{
    static std::string last;
    last.swap(g_log);
    g_log.clear();
    return last.c_str();
}
long hipstub_replays(void) { return g_replays; } // launches of graphs
long hipstub_uploads(void) { return g_uploads; } // asynchronous ones

hipError_t hipMalloc(void **p, size_t bytes)
{
    if(g_capturing)
        return hipErrorStreamCaptureUnsupported;
    if(g_used + ((bytes + 4095) & ~(size_t)4095) > g_total)
        return hipErrorOutOfMemory;
    const hipError_t e = map_memory(p, bytes);
    if(e == hipSuccess) {
        g_used += g_allocs[*p];
        g_peak = g_used > g_peak ? g_used : g_peak;
    }
    return e;
}
hipError_t hipFree(void *p) { return unmap_memory(p, true); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return map_memory(p, bytes); }
hipError_t hipHostFree(void *p) { return unmap_memory(p, false); }
hipError_t hipMemGetInfo(size_t *free, size_t *total)
{
    *free = g_total - g_used;
    *total = g_total;
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t bytes)
{
    auto it = g_allocs.find(p);
    if(v == 0 && it != g_allocs.end()) // whole pages go back to being zero without being touched
        return madvise(p, (bytes + 4095) & ~(size_t)4095, MADV_DONTNEED) ? hipErrorInvalidValue : hipSuccess;
    memset(p, v, bytes);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    if(g_capturing)
        return hipErrorStreamCaptureUnsupported;
    memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t)
{
    g_uploads += k == hipMemcpyHostToDevice;
    return hipMemcpy(d, s, n, k);
}

hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 160 << 10 : 0;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof(*p));
    snprintf(p->name, sizeof(p->name), "stub");
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 160 << 10;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "stub error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static char memory[8 << 20];
    *p = memory;
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return new_handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return g_capturing ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s)
{
    *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
    g_capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    g_capturing = false;
    return new_handle(g);
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return new_handle(e); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t)
{
    g_replays++;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return new_handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return new_handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 0;
    return hipSuccess;
}

// what the compiler's host code calls for `kernel<<<...>>>` and for the kernels of a library
void **__hipRegisterFatBinary(const void *)
{
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    g_kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t)
{
    g_grid = grid;
    g_block = block;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    *g = g_grid;
    *b = g_block;
    *lds = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **, size_t, hipStream_t)
{
    if(g_log.size() < (1 << 20))
        g_log += g_kernels[f] + " " + std::to_string(grid.x) + " " + std::to_string(block.x) + "\n";
    g_launches[g_kernels[f]]++;
    return hipSuccess;
}

}  // extern "C"
