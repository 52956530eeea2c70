// A stand-in for the HIP runtime that records the launches a host makes instead of making them.  Linked with the library's
// sources compiled for the host alone (tests/recorder.py), it shows, without a GPU, which kernel an entry point takes for a
// shape, with which grid, workgroup and LDS, and what it is given: the rules of the launchers can then be tested over sizes no
// test would allocate.  Pointers are never followed.
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>
#include <vector>

#include <hip/hip_runtime_api.h>

namespace {
struct Launch {
    std::string name; // mangled
    unsigned shape[7]; // grid, workgroup, LDS bytes
    std::vector<uint64_t> args;
};
std::map<const void*, std::string>& names() {
    static std::map<const void*, std::string> m; // (filled by the registrations of objects constructed before this file's)
    return m;
}
std::vector<Launch> g_launches;
int g_args = 0, g_cus = 256;
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
std::vector<Config> g_configs;
} // namespace

extern "C" {

// ---- what the tests read ----
void rec_start(int args) { // args: words of each launch's arguments to keep, for kernels whose arguments are 64-bit words
    g_launches.clear();
    g_args = args;
}
void rec_cus(int cus) { g_cus = cus; }
int rec_count() { return (int)g_launches.size(); }
const char* rec_name(int i) { return g_launches[i].name.c_str(); }
void rec_shape(int i, unsigned* out) { memcpy(out, g_launches[i].shape, sizeof(g_launches[i].shape)); }
uint64_t rec_arg(int i, int k) { return g_launches[i].args[k]; }

// ---- the runtime ----
char __hip_fatbin[16] = {}; // (the device code the objects name: none)
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) { names()[host] = name; }
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
    g_configs.push_back(Config{grid, block, lds, stream});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
    const Config c = g_configs.back();
    g_configs.pop_back();
    *grid = c.grid, *block = c.block, *lds = c.lds, *stream = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* kernel, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t) {
    Launch l{names()[kernel], {grid.x, grid.y, grid.z, block.x, block.y, block.z, (unsigned)lds}, {}};
    for (int k = 0; k < g_args; ++k) {
        uint64_t v;
        memcpy(&v, args[k], sizeof(v));
        l.args.push_back(v);
    }
    g_launches.push_back(l);
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "(recorded)"; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) { // (the header names the runtime's current form of it)
    memset(p, 0, sizeof(*p));
    p->multiProcessorCount = g_cus;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return posix_memalign(p, 256, n < 256 ? 256 : n) ? hipErrorOutOfMemory : hipSuccess; }
hipError_t hipFree(void* p) {
    free(p);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
    *p = const_cast<void*>(symbol);
    return hipSuccess;
}

} // extern "C"
