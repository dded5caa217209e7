// A stand-in for the HIP runtime under libsgemm.so, for tests of its host side without a GPU: device memory is addresses
// that nobody reads, and a launch is a line in a list.  Loaded with RTLD_GLOBAL in front of the library (launch_recorder.py),
// whose calls then resolve here.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>
#include <unistd.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
struct Launch { const char* kernel; unsigned grid, threads; size_t lds; void* stream; unsigned long thread; };
struct Call { dim3 grid, block; size_t lds; hipStream_t stream; };
std::mutex g_lock;
std::map<const void*, std::string> g_names;   // host stub -> kernel
std::vector<Launch> g_launches;
size_t g_next = 1ul << 40, g_largest = ~(size_t)0;
int g_pause_us = 0, g_capturing = 0, g_allocations = 0;
thread_local Call t_call;
}  // namespace

extern "C" {
// ---- what a test asks for
void rec_clear() { std::lock_guard<std::mutex> l(g_lock); g_launches.clear(); }
int rec_count() { std::lock_guard<std::mutex> l(g_lock); return (int)g_launches.size(); }
void rec_get(int i, Launch* out) { std::lock_guard<std::mutex> l(g_lock); *out = g_launches[(size_t)i]; }
void rec_pause(int us) { g_pause_us = us; }              // every launch takes that long to return
void rec_largest_allocation(size_t bytes) { g_largest = bytes; }
void rec_capturing(int on) { g_capturing = on; }         // every stream is being captured
int rec_allocations() { std::lock_guard<std::mutex> l(g_lock); return g_allocations; }

// ---- what hipcc's host code calls
void** __hipRegisterFatBinary(const void*) { static void* handle; return &handle; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device_name, unsigned, void*, void*, void*, void*, int*) {
    int status = 0;
    char* plain = abi::__cxa_demangle(device_name, nullptr, nullptr, &status);
    std::lock_guard<std::mutex> l(g_lock);
    g_names[host] = status == 0 ? plain : device_name;
    free(plain);
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
    t_call = {grid, block, lds, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
    *grid = t_call.grid; *block = t_call.block; *lds = t_call.lds; *stream = t_call.stream;
    return hipSuccess;
}

// ---- the runtime
hipError_t hipLaunchKernel(const void* host, dim3 grid, dim3 block, void**, size_t lds, hipStream_t stream) {
    {
        std::lock_guard<std::mutex> l(g_lock);
        g_launches.push_back({g_names[host].c_str(), grid.x, block.x, lds, stream, (unsigned long)pthread_self()});
    }
    if (g_pause_us) usleep((useconds_t)g_pause_us);
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::mutex> l(g_lock);
    if (bytes > g_largest) return hipErrorOutOfMemory;
    g_allocations++;
    *p = reinterpret_cast<void*>(g_next);
    g_next += (bytes + 4095) & ~(size_t)4095;
    return hipSuccess;
}
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = reinterpret_cast<void*>(1ul << 39); return hipSuccess; }
hipError_t hipGetDevice(int* device) { *device = 0; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* prop, int) {
    memset(prop, 0, sizeof *prop);
    prop->multiProcessorCount = 256;
    prop->sharedMemPerBlock = 64 * 1024;
    strcpy(prop->gcnArchName, "gfx950:sramecc+:xnack-");
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "an error of the stand-in"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = reinterpret_cast<hipStream_t>(0x1000); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }
}
