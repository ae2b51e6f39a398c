// A HIP runtime without a GPU, for the host side of libmgh (dispatch, plans, context buffers): device
// memory is host memory that is never read, launches are recorded by kernel name and grid, and
// allocations past a limit fail. Loaded with RTLD_GLOBAL before libmgh, whose HIP symbols then
// resolve here. No kernel runs, so copies move bytes and outputs mean nothing.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cstdio>
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
};
std::map<const void*, std::string> g_names;
std::vector<Launch> g_launches;
std::map<void*, size_t> g_allocs;
size_t g_used = 0, g_limit = (size_t)-1;
hipError_t g_last = hipSuccess;
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} g_cfg;
hipError_t ret(hipError_t e) {
    if (e != hipSuccess) g_last = e;
    return e;
}
}  // namespace

extern "C" {

// ---- the test's side
void fake_limit(size_t bytes) { g_limit = bytes; }
size_t fake_used() { return g_used; }
int fake_launches() { return (int)g_launches.size(); }
void fake_clear() { g_launches.clear(); }
void fake_launch(int i, char* name, int cap, unsigned dims[6]) {
    const Launch& l = g_launches.at(i);
    std::snprintf(name, cap, "%s", l.name.c_str());
    dims[0] = l.grid.x, dims[1] = l.grid.y, dims[2] = l.grid.z;
    dims[3] = l.block.x, dims[4] = l.block.y, dims[5] = l.block.z;
}

// ---- registration and launches
void** __hipRegisterFatBinary(const void*) {
    static void* h;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    g_names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    g_cfg = Config{g, b, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = g_cfg.grid, *b = g_cfg.block, *lds = g_cfg.lds, *s = g_cfg.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t lds, hipStream_t) {
    auto it = g_names.find(f);
    // (threads per dimension fit 32 bits, as the runtime requires)
    const bool wide = (uint64_t)g.x * b.x >> 32 || (uint64_t)g.y * b.y >> 32 || (uint64_t)g.z * b.z >> 32;
    if (it == g_names.end() || wide || !g.x || !g.y || !g.z || g.y > 65535 || g.z > 65535 || b.x * b.y * b.z > 1024 || lds > 65536)
        return ret(hipErrorInvalidConfiguration);
    g_launches.push_back(Launch{it->second, g, b, lds});
    return hipSuccess;
}

// ---- device, memory, streams, events, graphs
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    std::snprintf(p->name, sizeof p->name, "no GPU");
    std::snprintf(p->gcnArchName, sizeof p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (n > g_limit || g_used > g_limit - n) return ret(hipErrorOutOfMemory);
    *p = std::aligned_alloc(256, (n + 255) / 256 * 256);
    if (!*p) return ret(hipErrorOutOfMemory);
    g_allocs[*p] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    auto it = g_allocs.find(p);
    if (it == g_allocs.end()) return ret(hipErrorInvalidValue);
    g_used -= it->second;
    g_allocs.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = (hipStream_t)std::malloc(8), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return std::free((void*)s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t)std::malloc(8), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free((void*)e), hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return *g = (hipGraph_t)std::malloc(8), hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return *e = (hipGraphExec_t)std::malloc(8), hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return std::free((void*)e), hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return std::free((void*)g), hipSuccess; }
}
