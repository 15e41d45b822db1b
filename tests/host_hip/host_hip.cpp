// A HIP runtime without a device, for tests of the library's host code: device
// memory is host memory, kernels are noted and not run, every event is complete
// when it is recorded and events lie 1 ms apart for each kernel between them.
// hh_fail(name, n, times) makes the n-th call from now of that function fail, and
// as many in all as `times` says.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

std::map<const void*, std::string> names;   // kernels by the address they are launched by
std::string launches, hostmallocs;
std::map<std::string, std::pair<int, int>> failing;   // calls until the first that fails, calls that fail
float clock_ms = 0;
int allocs = 0;

hipError_t status(const char* name)
{
    auto f = failing.find(name);
    if (f == failing.end() || --f->second.first > 0) return hipSuccess;
    if (--f->second.second <= 0) failing.erase(f);
    return hipErrorUnknown;
}

struct Dims {
    dim3 grid, block;
    size_t lds = 0;
    hipStream_t stream = nullptr;
} dims;

} // namespace

extern "C" {

// "name gridx blockx lds" of each launch, a line each, since the last call
const char* hh_launches()
{
    static std::string s;
    s.swap(launches);
    launches.clear();
    return s.c_str();
}
// "bytes flags" of each hipHostMalloc
const char* hh_hostmallocs() { return hostmallocs.c_str(); }
void hh_fail(const char* name, int n, int times) { failing[name] = {n, times}; }
int hh_allocs() { return allocs; }

void** __hipRegisterFatBinary(const void*)
{
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, uint3*, uint3*, dim3*, dim3*,
                           int*)
{
    names[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    dims = {grid, block, lds, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream)
{
    *grid = dims.grid;
    *block = dims.block;
    *lds = dims.lds;
    *stream = dims.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t lds, hipStream_t)
{
    launches += names[f] + " " + std::to_string(grid.x) + " " + std::to_string(block.x) + " " + std::to_string(lds) + "\n";
    clock_ms += 1;
    return hipSuccess;
}
hipError_t hipGetLastError() { return status("hipLaunchKernel"); }
const char* hipGetErrorString(hipError_t) { return "planted"; }

hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 160 << 10 : 0;
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*)
{
    *a = hipFuncAttributes{};
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static double scratch[(16 << 20) / sizeof(double)];
    *p = scratch;
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n)
{
    const hipError_t e = status("hipMalloc");
    if (e != hipSuccess) return e;
    ++allocs;
    *p = std::malloc(n);
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    --allocs;
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned flags)
{
    hostmallocs += std::to_string(n) + " " + std::to_string(flags) + "\n";
    ++allocs;
    *p = std::calloc(n, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipHostGetDevicePointer(void** d, void* p, unsigned)
{
    *d = p;
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return status("hipMemcpyAsync");
}
hipError_t hipMemset(void* d, int v, size_t n)
{
    std::memset(d, v, n);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    *s = reinterpret_cast<hipStream_t>(1);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return status("hipStreamSynchronize"); }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
    *g = reinterpret_cast<hipGraph_t>(1);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* g, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    *g = reinterpret_cast<hipGraphExec_t>(1);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t)
{
    launches += "graph 0 0 0\n";
    clock_ms += 1;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = reinterpret_cast<hipEvent_t>(new float(0));
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    delete reinterpret_cast<float*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    *reinterpret_cast<float*>(e) = clock_ms;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return status("hipEventQuery"); }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b)
{
    *ms = *reinterpret_cast<float*>(b) - *reinterpret_cast<float*>(a);
    return hipSuccess;
}

} // extern "C"
