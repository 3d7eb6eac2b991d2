// A HIP runtime for tests of the engines' host side on a machine without a GPU: loaded ahead of libtllm_stack_engine.so, it takes the
// place of the 20 runtime calls that the library makes, and ahead of libnvinfer_plugin_tensorrt_llm.so of those of a LLaMA session on one GPU, its step graph included.  Device memory is host memory within a budget, launches are recorded and compute
// nothing, but that wanted rows land: all of them zeros.  Launch limits are the runtime's documented ones: fewer than 2^32 threads per grid dimension, 65535 workgroups in y and z.
#include <hip/hip_runtime_api.h>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace
{
struct Config
{
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
std::vector<Config> g_configs;
std::map<void*, size_t> g_device, g_pinned;
std::map<const void*, std::string> g_names;
std::string g_launched, *g_captured = nullptr; // (a graph is the names of its kernels)
size_t g_live = 0, g_budget = ~size_t(0), g_pinned_budget = ~size_t(0), g_largest = 0;
int g_host_mallocs = 0, g_syncs = 0, g_stream_syncs = 0, g_event_syncs = 0, g_event_records = 0, g_graphs = 0, g_fail_launches = 0;
hipError_t g_last = hipSuccess;

hipError_t done(hipError_t e)
{
    if (e != hipSuccess)
        g_last = e;
    return e;
}
hipError_t release(std::map<void*, size_t>& from, void* p)
{
    if (!p)
        return hipSuccess;
    auto it = from.find(p);
    if (it == from.end())
        return done(hipErrorInvalidValue);
    if (&from == &g_device)
        g_live -= it->second;
    from.erase(it);
    std::free(p);
    return hipSuccess;
}
} // namespace

extern "C" {
// what the tests ask
void stub_budget(size_t bytes) { g_budget = bytes; }
void stub_pinned_budget(size_t bytes) { g_pinned_budget = bytes; } // of one allocation
size_t stub_live() { return g_live; }
size_t stub_largest() { return g_largest; } // allocation on the device so far
int stub_has_allocation(size_t bytes)
{
    for (auto& a : g_device)
        if (a.second == bytes)
            return 1;
    return 0;
}
int stub_host_mallocs() { return g_host_mallocs; }
int stub_device_syncs() { return g_syncs; }
int stub_stream_syncs() { return g_stream_syncs; }
int stub_event_syncs() { return g_event_syncs; }
int stub_event_records() { return g_event_records; }
void stub_fail_launches(int on) { g_fail_launches = on; }
int stub_graphs() { return g_graphs; } // instantiated so far
size_t stub_pinned_bytes()
{
    size_t n = 0;
    for (auto& a : g_pinned)
        n += a.second;
    return n;
}
const char* stub_launched() { return g_launched.c_str(); } // kernel names since the last stub_forget, a line each
void stub_forget() { g_launched.clear(); }

hipError_t hipMalloc(void** p, size_t n)
{
    if (n > g_budget || g_live > g_budget - n)
        return done(hipErrorOutOfMemory);
    *p = std::calloc(1, n ? n : 1); // (large ones are mapped on demand: nothing computes on them)
    g_device[*p] = n;
    g_live += n;
    g_largest = g_largest < n ? n : g_largest;
    return hipSuccess;
}
hipError_t hipFree(void* p) { return release(g_device, p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int)
{
    if (n > g_pinned_budget)
        return done(hipErrorOutOfMemory);
    ++g_host_mallocs;
    *p = std::calloc(1, n ? n : 1);
    g_pinned[*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { return release(g_pinned, p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return std::memmove(d, s, n), hipSuccess; }
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(new int(0)), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<int*>(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return ++g_event_records, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return ++g_event_syncs, hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; } // (all kernels are as quick)
hipError_t hipDeviceSynchronize() { return ++g_syncs, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return ++g_stream_syncs, hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) { return *s = reinterpret_cast<hipStream_t>(new int(0)), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return delete reinterpret_cast<int*>(s), hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return g_captured = new std::string, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
    *g = reinterpret_cast<hipGraph_t>(g_captured);
    g_captured = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t)
{
    ++g_graphs;
    *e = reinterpret_cast<hipGraphExec_t>(new std::string(*reinterpret_cast<std::string*>(g)));
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete reinterpret_cast<std::string*>(g), hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return delete reinterpret_cast<std::string*>(e), hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) { return g_launched += *reinterpret_cast<std::string*>(e), hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : e == hipSuccess ? "no error" : "invalid configuration"; }
hipError_t hipGetLastError()
{
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t)
{
    auto it = g_names.find(f);
    if (it != g_names.end() && it->second.find("deliver_kernel") != std::string::npos)
        std::memset(*static_cast<void**>(args[1]), 0, (size_t) grid.x * grid.y * 8); // every part's choice
    (g_captured ? *g_captured : g_launched) += (it == g_names.end() ? std::string("?") : it->second) + "\n";
    const bool fits = !g_fail_launches && grid.x && grid.y && grid.z && (uint64_t) grid.x * block.x < (1ull << 32) && grid.y <= 65535 && grid.z <= 65535;
    return done(fits ? hipSuccess : hipErrorInvalidConfiguration);
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream)
{
    g_configs.push_back({grid, block, shared, stream});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream)
{
    const Config c = g_configs.back();
    g_configs.pop_back();
    *grid = c.grid;
    *block = c.block;
    *shared = c.shared;
    *stream = c.stream;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*)
{
    static void* module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned int, void*, void*, void*, void*, int*) { g_names[host] = name; }
}
