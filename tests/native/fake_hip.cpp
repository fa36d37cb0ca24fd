// fake_hip.cpp -- a stand-in for the HIP runtime under the library's host code, for CPU tests of its call order and
// error paths.  Device memory is host memory, kernels are logged and not run (three small ones, whose effect the
// host code goes on from, are done here).  Linked with the library's own objects by tests/native/Makefile.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

std::map<const void*, std::string> g_kernels;      // host function -> device name
std::map<char*, size_t> g_live;                     // allocations
std::vector<std::string> g_log;
std::string g_fail;                                 // function to fail, ...
int g_fail_in = 0;                                  // ... at its n-th call from now
int g_cus = 256, g_occ = 2;
hipError_t g_error = hipSuccess;
struct Launch { std::string line; };
std::vector<Launch> g_captured;
bool g_capturing = false;
std::map<uintptr_t, std::vector<Launch>> g_graphs;
uintptr_t g_next = 0x1000;
struct Config { dim3 g, b; size_t lds; hipStream_t s; };
std::vector<Config> g_config;

void note(const std::string& s) { g_log.push_back(s); }
std::string hex(const void* p)
{
    char b[32];
    snprintf(b, sizeof b, "%p", p);
    return b;
}
hipError_t fails(const char* f)
{
    if (g_fail != f || --g_fail_in > 0) return hipSuccess;
    g_fail.clear();
    note(std::string("failed ") + f);
    return g_error = hipErrorUnknown;
}
#define TRY(f) if (hipError_t e_ = fails(f)) return e_

}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
    g_kernels[f] = name;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    g_config.push_back({g, b, lds, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s)
{
    const Config c = g_config.back();
    g_config.pop_back();
    *g = c.g; *b = c.b; *lds = c.lds; *s = c.s;
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n)
{
    TRY("hipMalloc");
    char* q = (char*)malloc(n ? n : 1);
    memset(q, 0xa5, n);   // device memory comes with what was there
    g_live[q] = n;
    *p = q;
    note("malloc " + hex(q) + " " + std::to_string(n));
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    note("free " + hex(p));
    if (g_live.erase((char*)p)) free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    TRY("hipHostMalloc");
    return hipMalloc(p, n);
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemset(void* p, int v, size_t n)
{
    TRY("hipMemset");
    note("memset " + hex(p) + " null-stream");   // not waited for: the memory has it at the next wait
    memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s)
{
    TRY("hipMemsetAsync");
    note("memset " + hex(p) + " " + hex(s));
    memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
    TRY("hipMemcpy");
    note("memcpy " + hex(d) + " " + hex(s));
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t)
{
    TRY("hipMemcpyAsync");
    note("memcpy " + hex(d) + " " + hex(s));
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s)
{
    TRY("hipStreamSynchronize");
    note("sync " + hex(s));
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void)
{
    note("sync device");
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)(g_next += 16); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)(g_next += 16); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* t, hipEvent_t, hipEvent_t) { *t = 1.0f; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = nullptr; return hipErrorInvalidSymbol; }
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) { memset(a, 0, sizeof *a); return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipGetLastError(void)
{
    const hipError_t e = g_error;
    g_error = hipSuccess;
    return e;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? g_cus : 100000;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t)
{
    *n = g_occ;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { g_capturing = true; g_captured.clear(); return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
    g_capturing = false;
    g_graphs[g_next += 16] = g_captured;
    *g = (hipGraph_t)g_next;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t)
{
    TRY("hipGraphInstantiate");
    *x = (hipGraphExec_t)g;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t)
{
    if (!x) return hipErrorInvalidValue;
    for (const Launch& l : g_graphs[(uintptr_t)x]) note(l.line);
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void** args, size_t, hipStream_t s)
{
    TRY("hipLaunchKernel");
    const std::string name = g_kernels.count(f) ? g_kernels[f] : "?";
    std::string line = "launch " + name + " grid " + std::to_string(g.x) + " stream " + hex(s);
    const bool publish = name.find("publish_u64") != std::string::npos, clear = name.find("clear_u64") != std::string::npos;
    const bool control = name.find("ens_ctl") != std::string::npos;
    if (publish || clear) line += " p " + hex(*(void**)args[0]);
    if (publish) line += " host " + hex(*(void**)args[1]);
    if (name.find("ens_march") != std::string::npos) {   // EnsLaunch: boxes, tiles, total
        const char* a = (const char*)args[0];
        line += " boxes " + hex(*(void* const*)a) + " tiles " + hex(*(void* const*)(a + 8)) + " total " +
                std::to_string(*(const int*)(a + 16));
    }
    if (g_capturing) {
        g_captured.push_back({line});
        return hipSuccess;
    }
    note(line);
    if (publish) {
        unsigned long long* slot = *(unsigned long long**)args[0];
        **(unsigned long long**)args[1] = *slot;
        if (*(int*)args[2]) *slot = 0;
    } else if (clear) {
        memset(*(void**)args[0], 0, 8 * (size_t) * (int*)args[1]);
    } else if (control) {
        **(int**)args[9] = (int)(++**(long long**)args[4] + 1) & 1;   // the sweep number, and the buffers' parity
    }
    return hipSuccess;
}

// the tests' side
void fh_reset(int cus, int occ) { g_log.clear(); g_fail.clear(); g_cus = cus; g_occ = occ; g_error = hipSuccess; }
void fh_fail(const char* f, int nth) { g_fail = f; g_fail_in = nth; }
int fh_log_size(void) { return (int)g_log.size(); }
const char* fh_log(int i) { return g_log[i].c_str(); }
long fh_live(const char* p)   // bytes of the allocation, -1: freed
{
    auto it = g_live.find((char*)p);
    return it == g_live.end() ? -1 : (long)it->second;
}

}  // extern "C"
