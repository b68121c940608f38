// A HIP runtime without a device, for tests of the library's host code on the
// CPU: loaded with RTLD_GLOBAL ahead of libter_hip.so it takes the place of
// libamdhip64.  Device memory is host memory, kernels do not run (done_kernel
// writes its number), and every call that matters to a test is a line of
// fake_log().
#include <cxxabi.h>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

struct Dim3 {
    uint32_t x, y, z;
};

namespace {
std::map<const void*, std::string> g_names;
std::string g_log, g_fail;
int g_device = 0, g_last = 0;
struct {
    Dim3 grid, block;
    size_t lds;
    void* st;
} g_call;

const char* name_of(const void* fn) { return g_names[fn].c_str(); }
void note(const char* what, const std::string& rest = "") { g_log += std::string(what) + " " + rest + "\n"; }
void* host(size_t n) { return aligned_alloc(4096, (n + 4095) / 4096 * 4096); }
}  // namespace

extern "C" {
// ---- the test's side
const char* fake_log() { return g_log.c_str(); }
void fake_reset() { g_log.clear(); }
void fake_device(int d) { g_device = d; }
void fake_fail(const char* kernel) { g_fail = kernel; }  // launches of kernels whose name contains it fail

// ---- the runtime's side
void** __hipRegisterFatBinary(const void*) {
    static void* h;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* fn, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    int rc = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &rc);
    g_names[fn] = d ? d : name;
    free(d);
}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t lds, void* st) {
    g_call = {grid, block, lds, st};
    return 0;
}
int __hipPopCallConfiguration(Dim3* grid, Dim3* block, size_t* lds, void** st) {
    *grid = g_call.grid;
    *block = g_call.block;
    *lds = g_call.lds;
    *st = g_call.st;
    return 0;
}
int hipLaunchKernel(const void* fn, Dim3 grid, Dim3 block, void** args, size_t lds, void*) {
    const std::string n = name_of(fn);
    if (!g_fail.empty() && n.find(g_fail) != std::string::npos) {
        note("failed", n);
        return g_last = 719;
    }
    note("launch", std::to_string(g_device) + " " + std::to_string(grid.x) + " " + std::to_string(block.x) + " " +
                       std::to_string(lds) + " " + n);
    if (n.find("done_kernel") != std::string::npos) **static_cast<uint32_t**>(args[0]) = *static_cast<uint32_t*>(args[1]);
    return 0;
}
int hipGetLastError() {
    const int e = g_last;
    g_last = 0;
    return e;
}
const char* hipGetErrorString(int) { return "fake error"; }
int hipGetDevice(int* d) {
    *d = g_device;
    return 0;
}
int hipSetDevice(int d) {
    g_device = d;
    return 0;
}
int hipDeviceGetAttribute(int* v, int, int) {
    *v = 256;  // the CU count
    return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void*) {
    note("sync");
    return 0;
}
int hipFuncSetAttribute(const void* fn, int, int v) {
    note("attribute", std::to_string(g_device) + " " + std::to_string(v) + " " + name_of(fn));
    return 0;
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t lds) {
    *n = lds > 163840 ? 0 : (lds > 81920 ? 1 : 2);
    return 0;
}
int hipMalloc(void** p, size_t n) {
    *p = host(n);
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
int hipHostGetDevicePointer(void** d, void* h, unsigned) {
    *d = h;
    return 0;
}
int hipFree(void* p) {
    free(p);
    return 0;
}
int hipHostFree(void* p) { return hipFree(p); }
int hipMemcpy(void* d, const void* s, size_t n, int) {
    memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
    note("copy");
    memcpy(d, s, n);
    return 0;
}
int hipMemset(void* d, int v, size_t n) {
    memset(d, v, n);
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) { return hipMemset(d, v, n); }
int hipGetSymbolAddress(void** p, const void*) {
    *p = host(4096);
    return 0;
}
}
