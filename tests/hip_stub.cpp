// A HIP runtime without a device, for tests of the host side on the CPU: the
// library's host sources are linked against it instead of libamdhip64.  Every
// pointer counts as device memory, modules and kernels do nothing, and each
// launch is recorded with its grid and arguments.  As by the runtime, a launch
// of 2^32 or more work-items in a dimension is refused, and so are allocations
// and synchronisations while a stream is captured.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../pto-wsp_amd/csrc/device/ptowsp_launch.h"
#include "noalloc.hpp"

namespace {
struct Launch {
    std::string entry;
    unsigned long long blocks, threads;
    ptowsp::LaunchArgs args;
};
std::vector<Launch>& log() {
    static std::vector<Launch> l;
    return l;
}
bool capturing = false;
std::vector<void*> freed;
hipError_t uncaptured() { return capturing ? hipErrorStreamCaptureUnsupported : hipSuccess; }
}  // namespace

extern "C" {

// Recorded launches, for the tests.
int stub_num_launches() { return static_cast<int>(log().size()); }
void stub_clear() { log().clear(); }
void stub_capture(int on) { capturing = on != 0; }
int stub_freed(void* p) {  // whether p has been given back since it was last allocated
    for (void* f : freed)
        if (f == p) return 1;
    return 0;
}
const char* stub_entry(int i) { return log()[i].entry.c_str(); }
unsigned long long stub_blocks(int i) { return log()[i].blocks; }
unsigned long long stub_threads(int i) { return log()[i].threads; }
void* stub_base(int i, int p) { return log()[i].args.base[p]; }
long long stub_s3(int i, int p) { return log()[i].args.s3[p]; }
long long stub_s4(int i, int p) { return log()[i].args.s4[p]; }
long long stub_coef(int i, int p, int v) { return log()[i].args.coef[p][v]; }

const char* hipGetErrorString(hipError_t e) { return e == hipErrorInvalidValue ? "invalid argument" : "stub error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 160 * 1024;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return uncaptured(); }
hipError_t hipStreamSynchronize(hipStream_t) { return uncaptured(); }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) {
    if (capturing) return uncaptured();
    *p = std::malloc(n);
    for (size_t i = freed.size(); i-- > 0;)
        if (freed[i] == *p) freed.erase(freed.begin() + static_cast<long>(i));
    return hipSuccess;
}
hipError_t hipFree(void* p) { return freed.push_back(p), std::free(p), uncaptured(); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::calloc(1, n), uncaptured(); }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemset(void* p, int v, size_t n) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) { return a->type = hipMemoryTypeDevice, hipSuccess; }
hipError_t hipModuleLoadData(hipModule_t* m, const void*) { return *m = nullptr, uncaptured(); }
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) {
    *f = reinterpret_cast<hipFunction_t>(new std::string(name));
    return hipSuccess;
}
hipError_t hipFuncGetAttribute(int* v, hipFunction_attribute, hipFunction_t) { return *v = 0, hipSuccess; }
hipError_t hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(int* n, hipFunction_t, int, size_t) { return *n = 1, hipSuccess; }
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned, unsigned, unsigned bx, unsigned, unsigned, unsigned, hipStream_t,
                                 void** params, void**) {
    if (static_cast<unsigned long long>(gx) * bx >= 1ull << 32) return hipErrorInvalidValue;
    log().push_back({*reinterpret_cast<std::string*>(f), gx, bx, *static_cast<const ptowsp::LaunchArgs*>(params[0])});
    return hipSuccess;
}

}  // extern "C"

namespace ptowsp {
void noalloc_prepare(hipStream_t) {}
void* noalloc_scratch() {
    static void* p = std::calloc(1, kNoAllocScratchBytes);
    return p;
}
void noalloc_zero(void* p, size_t n, hipStream_t) { std::memset(p, 0, n); }
}  // namespace ptowsp
