// The HIP runtime calls of the library on the host alone: device memory is host memory with a
// limit, kernels are counted and not run.  Loaded globally before the library, it takes the place
// of the runtime, so that host paths (allocation, launch shapes, tuning) run without a GPU.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

std::map<void*, size_t> allocs;
size_t used = 0, limit = (size_t)-1;
long to_host = 0;
hipError_t last = hipSuccess;
struct Call {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} call{};
std::map<const void*, std::string> names;
struct Seen {
    long launches = 0;
    unsigned block = 0;
};
std::map<std::string, Seen> seen;
alignas(256) char symbol[(size_t)8 << 20];

hipError_t give(hipError_t e)
{
    if (e != hipSuccess) last = e;
    return e;
}
void* handle() { return std::malloc(16); }
void copied(void* d, const void* s, size_t n, hipMemcpyKind k)
{
    std::memcpy(d, s, n);
    to_host += k == hipMemcpyDeviceToHost;
}

}  // namespace

extern "C" {

// ---- what a test sets and asks
size_t host_used() { return used; }
void host_limit(size_t bytes) { limit = bytes; }
long host_copies_to_host() { return to_host; }
long host_launches(const char* kernel)
{
    long n = 0;
    for (auto& s : seen)
        if (s.first.find(kernel) != std::string::npos) n += s.second.launches;
    return n;
}
// threads per block of the last launch of a kernel whose name holds this text; 0 for none
unsigned host_block(const char* kernel)
{
    for (auto& s : seen)
        if (s.first.find(kernel) != std::string::npos && s.second.launches) return s.second.block;
    return 0;
}
void host_forget() { seen.clear(); }

// ---- the runtime
hipError_t hipMalloc(void** p, size_t n)
{
    *p = nullptr;
    if (n > limit || used > limit - n) return give(hipErrorOutOfMemory);
    *p = std::malloc(n ? n : 1);
    allocs[*p] = n;
    used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    if (!p) return hipSuccess;
    auto i = allocs.find(p);
    if (i == allocs.end()) return give(hipErrorInvalidValue);
    used -= i->second;
    allocs.erase(i);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return (*p = std::malloc(n ? n : 1)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t)
{
    *t = limit;
    *f = limit - used;
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k)
{
    copied(d, s, n, k);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t)
{
    copied(d, s, n, k);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n)
{
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    *p = symbol;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    *p = hipDeviceProp_tR0600{};
    std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "host"; }
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    *s = (hipStream_t)handle();
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e)
{
    *e = (hipEvent_t)handle();
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
    *g = (hipGraph_t)handle();
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    *x = (hipGraphExec_t)handle();
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g)
{
    std::free(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x)
{
    std::free(x);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3, dim3 block, void**, size_t, hipStream_t)
{
    Seen& s = seen[names[f]];
    s.launches += 1;
    s.block = block.x;
    return hipSuccess;
}

// ---- what compiled launches call
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    call = Call{grid, block, lds, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream)
{
    *grid = call.grid;
    *block = call.block;
    *lds = call.lds;
    *stream = call.stream;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*)
{
    static void* h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*)
{
    names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

}  // extern "C"
