// A stand-in for the HIP runtime that runs no kernel: device memory is host memory, every call is written down, and the
// clock of the events advances by a cost per kernel launch. With it loaded first (RTLD_GLOBAL), libswmi.so's host side
// runs on a machine without a GPU, and a test reads which kernels it launched, on which streams and in which order, or
// makes a call fail. Used by test_host_path.py only.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <utility>
#include <vector>

namespace
{
    struct Event { double at = 0.0; int id = 0; };
    struct Graph { std::vector<std::string> lines; double cost = 0.0; };

    std::string text;
    std::map<const void*, std::string> kernels;
    std::vector<std::pair<std::string, double>> costs;   // substring of the kernel's name -> microseconds
    std::string failing;                                 // name of the call that fails
    size_t fail_from = 0;                                // (allocations: those of at least this many bytes)
    double now = 0.0;
    int ids = 0;
    Graph* capturing = nullptr;
    dim3 cfg_grid, cfg_block;
    size_t cfg_lds = 0;
    hipStream_t cfg_stream = nullptr;

    long Id(const void* p) { return static_cast<long>(reinterpret_cast<intptr_t>(p)); }
    void Note(const std::string& s) { (capturing ? capturing->lines.emplace_back(s), text += "captured " : text) += s + "\n"; }
    hipError_t Maybe(const char* name) { return failing == name ? hipErrorUnknown : hipSuccess; }
}

extern "C" {

// ---- the test's side ----
const char* rec_take()
{
    static std::string out;
    out.swap(text);
    text.clear();
    return out.c_str();
}
void rec_fail(const char* name, size_t from)
{
    failing = name;
    fail_from = from;
}
void rec_cost(const char* part, double us) { costs.insert(costs.begin(), {part, us}); }

// ---- the runtime's side ----
void** __hipRegisterFatBinary(const void*)
{
    static void* handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { kernels[host] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    cfg_grid = grid;
    cfg_block = block;
    cfg_lds = lds;
    cfg_stream = stream;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream)
{
    *grid = cfg_grid;
    *block = cfg_block;
    *lds = cfg_lds;
    *stream = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 grid, dim3 block, void**, size_t lds, hipStream_t stream)
{
    const std::string& name = kernels[fn];
    double us = 1.0;
    for (const auto& c : costs)
        if (name.find(c.first) != std::string::npos)
        {
            us = c.second;
            break;
        }
    (capturing ? capturing->cost : now) += us;
    char line[64];
    std::snprintf(line, sizeof line, " grid %u block %u lds %zu stream %ld", grid.x, block.x, lds, Id(stream));
    Note("launch " + name + line);
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t* p, int)
{
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "failed by the test"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    static std::vector<char> memory(64u << 20);
    return *p = memory.data(), hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n)
{
    if (failing == "hipMalloc" && n >= fail_from)
        return hipErrorOutOfMemory;
    return *p = std::calloc(n, 1), hipSuccess;
}
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>(static_cast<intptr_t>(++ids)), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    Note("wait stream " + std::to_string(Id(s)) + " event " + std::to_string(reinterpret_cast<Event*>(e)->id));
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
    if (const hipError_t e = Maybe("hipStreamBeginCapture"))
        return e;
    return capturing = new Graph, hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
    *g = reinterpret_cast<hipGraph_t>(capturing);
    capturing = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t)
{
    if (const hipError_t e = Maybe("hipGraphInstantiate"))
        return e;
    return *x = reinterpret_cast<hipGraphExec_t>(new Graph(*reinterpret_cast<Graph*>(g))), hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return delete reinterpret_cast<Graph*>(g), hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return delete reinterpret_cast<Graph*>(x), hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t)
{
    for (const auto& l : reinterpret_cast<Graph*>(x)->lines)
        Note(l);
    now += reinterpret_cast<Graph*>(x)->cost;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    auto* ev = new Event;
    ev->id = ++ids;
    return *e = reinterpret_cast<hipEvent_t>(ev), hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete reinterpret_cast<Event*>(e), hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    reinterpret_cast<Event*>(e)->at = now;
    Note("record event " + std::to_string(reinterpret_cast<Event*>(e)->id) + " stream " + std::to_string(Id(s)));
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b)
{
    *ms = static_cast<float>((reinterpret_cast<Event*>(b)->at - reinterpret_cast<Event*>(a)->at) * 1e-3);
    return hipSuccess;
}
}
