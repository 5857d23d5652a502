// A stand-in for the HIP runtime on a machine without a device: memory is host memory, copies are memcpy, kernels
// are recorded and not run.  Loaded with global symbols before libmset_amd.so, it takes the place of libamdhip64 for
// that library, so the host logic (buffers, captures, grids, routes) runs and can be looked at.  Built and driven by
// tests/fake_hip.py.
#define __HIP_PLATFORM_AMD__ 1
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>

namespace {

std::map<void*, size_t> g_live;                     // device allocations
size_t g_bytes = 0, g_peak = 0, g_total = (size_t)288 << 30, g_fail = 0;
std::map<const void*, std::string> g_names;         // kernels by host function
std::map<std::string, int> g_occ;                   // workgroups per CU by a part of the name
std::map<const void*, void*> g_vars;
std::string g_log;                                  // "name grid block captured" per launch
bool g_capturing = false;
int g_captures = 0, g_replays = 0, g_stale_replays = 0;

// an executable graph is stale once any allocation that was live when it was made has been freed
struct Exec {
    bool stale = false;
};
std::set<Exec*> g_exec;

struct Call {
    dim3 grid, block;
};
Call g_call;

}  // namespace

extern "C" {

// ---- what a test reads and sets
void fake_reset() {
    g_log.clear();
    g_captures = g_replays = g_stale_replays = 0;
    g_peak = g_bytes;
}
const char* fake_log() { return g_log.c_str(); }
const char* fake_kernels() {                              // every kernel of the library, one a line
    static std::string all;
    all.clear();
    for (const auto& kv : g_names) all += kv.second + "\n";
    return all.c_str();
}
int fake_captures() { return g_captures; }
int fake_replays() { return g_replays; }
int fake_stale_replays() { return g_stale_replays; }
size_t fake_bytes() { return g_bytes; }
size_t fake_peak() { return g_peak; }
void fake_fail_malloc(size_t bytes) { g_fail = bytes; }   // allocations of exactly this size fail (0: none)
void fake_device_memory(size_t bytes) { g_total = bytes; }   // allocations beyond it fail
void fake_occupancy(const char* part, int per_cu) { g_occ[part] = per_cu; }

// ---- the runtime
hipError_t hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if ((g_fail && n == g_fail) || g_bytes + n > g_total) return hipErrorOutOfMemory;
    *p = calloc(1, n ? n : 1);
    g_live[*p] = n;
    g_bytes += n;
    if (g_bytes > g_peak) g_peak = g_bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    auto it = g_live.find(p);
    if (it == g_live.end()) return hipErrorInvalidValue;
    g_bytes -= it->second;
    g_live.erase(it);
    free(p);
    for (Exec* e : g_exec) e->stale = true;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (!g_capturing) memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    *f = g_total - g_bytes;
    *t = g_total;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* s) {
    void*& v = g_vars[s];
    if (!v) v = calloc(1, 64);
    *p = v;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = (hipStream_t)calloc(1, 64);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = (hipEvent_t)calloc(1, 8);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0.f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    g_capturing = true;
    ++g_captures;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    g_capturing = false;
    *g = (hipGraph_t)calloc(1, 8);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    free(g);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    Exec* x = new Exec;
    g_exec.insert(x);
    *e = (hipGraphExec_t)x;
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    g_exec.erase((Exec*)e);
    delete (Exec*)e;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    ++g_replays;
    if (((Exec*)e)->stale) ++g_stale_replays;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int, size_t) {
    const std::string& name = g_names[f];
    *n = 2;
    for (const auto& kv : g_occ)
        if (name.find(kv.first) != std::string::npos) *n = kv.second;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t, hipStream_t) {
    g_log += g_names[f] + "|" + std::to_string(grid.x) + "|" + std::to_string(grid.y) + "|" + std::to_string(block.x) + "|" +
             (g_capturing ? "1" : "0") + "\n";
    return hipSuccess;
}

// ---- registration of the library's kernels
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    int st = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    g_names[host] = d ? d : name;
    free(d);
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
    g_call = Call{grid, block};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* st) {
    *grid = g_call.grid;
    *block = g_call.block;
    *shared = 0;
    *st = nullptr;
    return hipSuccess;
}

}  // extern "C"
