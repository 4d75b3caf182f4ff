// hip_stub.cpp -- the part of the HIP runtime that libCReaDDyGPU.so calls, on
// the CPU: memory is host memory (zeroed), copies are done at once, streams and
// events do nothing and kernels are not run, only recorded.  Loaded ahead of
// the library (globally), it lets a test follow the host code: which kernels
// are launched with which sizes and pointers, how often steps are captured,
// and what a call leaves behind after an allocation or a copy failed.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Launch {
    std::string name;
    dim3 grid, block;
    size_t lds;
    std::vector<void*> arg;      // the first arguments' first 8 bytes (pointers where they are pointers)
};
std::map<const void*, std::string> kernels;
std::vector<Launch> launches;
std::map<char*, size_t> blocks;
long captures, graph_launches, mallocs, copies, fail_malloc_at = -1, fail_copy_at = -1;
struct Config { dim3 grid, block; size_t lds; hipStream_t stream; };
std::vector<Config> pushed;

hipError_t record(const void* f, dim3 grid, dim3 block, void** args, size_t lds)
{
    Launch l;
    l.name = kernels.count(f) ? kernels[f] : "?";
    l.grid = grid; l.block = block; l.lds = lds;
    // the force kernels' pointers (eleven before the first number but one)
    if (l.name.find("k_force_update") != std::string::npos)
        for (int i = 0; i < 11; ++i) {
            void* v = nullptr;
            memcpy(&v, args[i], i == 9 ? sizeof(int) : sizeof(void*));
            l.arg.push_back(v);
        }
    launches.push_back(l);
    return hipSuccess;
}

hipError_t allocate(void** p, size_t n)
{
    *p = nullptr;
    if (mallocs++ == fail_malloc_at) return hipErrorOutOfMemory;
    *p = calloc(n ? n : 1, 1);
    blocks[(char*)*p] = n;
    return hipSuccess;
}

hipError_t copy(void* d, const void* s, size_t n)
{
    if (copies++ == fail_copy_at) return hipErrorUnknown;
    memmove(d, s, n);
    return hipSuccess;
}
}  // namespace

extern "C" {
// ---- for the test ----
void stub_reset() { launches.clear(); captures = graph_launches = mallocs = copies = 0; fail_malloc_at = fail_copy_at = -1; }
void stub_fail_malloc(long k) { mallocs = 0; fail_malloc_at = k; }
void stub_fail_copy(long k) { copies = 0; fail_copy_at = k; }
long stub_mallocs() { return mallocs; }
long stub_copies() { return copies; }
long stub_captures() { return captures; }
long stub_graph_launches() { return graph_launches; }
long stub_launches() { return (long)launches.size(); }
const char* stub_name(long i) { return launches[i].name.c_str(); }
void stub_dims(long i, long* out)
{
    const Launch& l = launches[i];
    out[0] = l.grid.x; out[1] = l.block.x; out[2] = (long)l.lds;
}
void* stub_arg(long i, int k) { return k < (int)launches[i].arg.size() ? launches[i].arg[k] : nullptr; }
long stub_size(void* p) { auto it = blocks.find((char*)p); return it == blocks.end() ? -1 : (long)it->second; }

// ---- the runtime ----
hipError_t hipMalloc(void** p, size_t n) { return allocate(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) { return allocate(p, n); }
hipError_t hipFree(void* p)
{
    if (p && !blocks.erase((char*)p)) return hipErrorInvalidValue;
    free(p);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return copy(d, s, n); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return copy(d, s, n); }
hipError_t hipMemset(void* d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static void* scratch = calloc((size_t)64 << 20, 1);
    *p = scratch;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    memset(p, 0, sizeof(*p));
    strcpy(p->name, "stub");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 4; return hipSuccess; }

static char handle;
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) { *s = (hipStream_t)&handle; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned int) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)&handle; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned int) { *e = (hipEvent_t)&handle; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { ++captures; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = (hipGraph_t)&handle; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    *e = (hipGraphExec_t)&handle;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { ++graph_launches; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

void** __hipRegisterFatBinary(const void*) { static void* m[1]; return m; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned int, void*, void*, dim3*, dim3*, int*)
{
    kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s)
{
    pushed.push_back({ grid, block, lds, s });
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s)
{
    const Config c = pushed.back();
    pushed.pop_back();
    *grid = c.grid; *block = c.block; *lds = c.lds; *s = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t)
{
    return record(f, grid, block, args, lds);
}
hipError_t hipExtLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t, hipEvent_t,
                              hipEvent_t, int)
{
    return record(f, grid, block, args, lds);
}
}
