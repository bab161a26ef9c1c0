// The HIP runtime's entry points without a device, for tests of what the
// engine does on the host: memory is host memory (zeroed, optionally limited),
// copies are memcpy, events are always complete, and a kernel launch is
// recorded (name, grid, block, dynamic LDS) instead of run.  Loaded with
// RTLD_GLOBAL before libqfe.so, whose calls it then takes.
#include <hip/hip_runtime.h>

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
std::map<const void*, std::string> names;
std::vector<Launch> launches;
std::map<void*, size_t> live;
size_t used = 0, limit = ~(size_t)0, symbol_bytes = 0;
dim3 cfg_grid, cfg_block;
size_t cfg_lds = 0;
hipStream_t cfg_stream = nullptr;
hipError_t last = hipSuccess;

hipError_t done(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
hipError_t take(void** p, size_t bytes, bool device) {
    if (device && (bytes > limit || used > limit - bytes)) return done(hipErrorOutOfMemory);
    *p = std::calloc(1, bytes ? bytes : 1);
    if (!*p) return done(hipErrorOutOfMemory);
    if (device) {
        live[*p] = bytes;
        used += bytes;
    }
    return hipSuccess;
}
}  // namespace

extern "C" {

// ---- for the tests --------------------------------------------------------------
void host_limit(size_t bytes) { limit = bytes; }
size_t host_used() { return used; }
size_t host_launches() { return launches.size(); }
const char* host_launch(size_t i, unsigned* shape7) {
    const Launch& l = launches[i];
    const unsigned v[7] = {l.grid.x, l.grid.y, l.grid.z, l.block.x, l.block.y, l.block.z, (unsigned)l.lds};
    std::memcpy(shape7, v, sizeof(v));
    return l.name.c_str();
}
void host_forget() { launches.clear(); }

// ---- registration and launches -----------------------------------------------------
void** __hipRegisterFatBinary(const void*) {
    static void* handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device_name, unsigned, uint3*, uint3*, dim3*, dim3*, int*) {
    names[host] = device_name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t size, int, int) { symbol_bytes = size > symbol_bytes ? size : symbol_bytes; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) {
    cfg_grid = grid;
    cfg_block = block;
    cfg_lds = lds;
    cfg_stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* st) {
    *grid = cfg_grid;
    *block = cfg_block;
    *lds = cfg_lds;
    *st = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t lds, hipStream_t) {
    launches.push_back(Launch{names[f], grid, block, lds});
    // what a device takes: 2^31 - 1 blocks in x, 65535 in y and z
    const bool ok = grid.x && grid.y && grid.z && grid.x < (1u << 31) && grid.y <= 65535 && grid.z <= 65535;
    return ok ? hipSuccess : done(hipErrorInvalidConfiguration);
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }

// ---- memory ------------------------------------------------------------------------
hipError_t hipMalloc(void** p, size_t bytes) { return take(p, bytes, true); }
hipError_t hipFree(void* p) {
    auto it = live.find(p);
    if (it != live.end()) {
        used -= it->second;
        live.erase(it);
    }
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return take(p, bytes, false); }
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* symbol = nullptr;
    if (!symbol) symbol = std::calloc(1, symbol_bytes);
    *p = symbol;
    return hipSuccess;
}

// ---- device, streams, events ---------------------------------------------------------
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 160 << 10;  // the engine asks for the LDS of a block
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error of the host runtime"; }

}  // extern "C"
