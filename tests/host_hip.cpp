// A stand-in for the HIP runtime under the library's host code, for tests of its dispatch without a
// device: device memory is numbers, nothing runs, and every launch is written down by its kernel's name.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstring>
#include <map>
#include <set>
#include <string>

namespace {

std::set<std::string> names;                 // hipFunction_t is the address of a name here
std::string launches;                        // "<kernel> <grid x> <y> <z> <block>\n" each
std::map<uintptr_t, size_t> memory;          // live allocations
uintptr_t next_address = 1ull << 40;
size_t largest = SIZE_MAX;                   // allocations above it fail
int own_capture = 0, other_capture = 0;      // the context's stream, another stream (global mode)
int broken_captures = 0;
hipError_t last_error = hipSuccess;
hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;

hipError_t fail(hipError_t e) { return last_error = e; }

// calls that a capture in progress anywhere forbids to threads that have not relaxed their mode
bool forbidden() {
    if (!(other_capture || own_capture) || mode == hipStreamCaptureModeRelaxed) return false;
    ++broken_captures;
    return true;
}

}  // namespace

extern "C" {

void host_hip_reset() {
    launches.clear();
    largest = SIZE_MAX;
    own_capture = other_capture = broken_captures = 0;
    last_error = hipSuccess;
}
const char *host_hip_launches() { return launches.c_str(); }
void host_hip_largest(size_t n) { largest = n; }
void host_hip_capture(int own, int other) { own_capture = own, other_capture = other; }
int host_hip_broken_captures() { return broken_captures; }
int host_hip_last_error() { return (int) last_error; }
size_t host_hip_allocations() { return memory.size(); }

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) { return std::memset(p, 0, sizeof(*p)), hipSuccess; }
hipError_t hipDeviceGetName(char *name, int len, hipDevice_t) { return std::strncpy(name, "host", (size_t) len), hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipFuncGetAttribute(int *v, hipFunction_attribute, hipFunction_t) { return *v = 256, hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}

hipError_t hipMalloc(void **p, size_t n) {
    if (forbidden()) return fail(hipErrorStreamCaptureUnsupported);
    if (n > largest) return fail(hipErrorOutOfMemory);
    memory[next_address] = n;
    *p = (void *) next_address;
    next_address += (n + 4095) / 4096 * 4096 + 4096;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (forbidden()) return fail(hipErrorStreamCaptureUnsupported);
    return memory.erase((uintptr_t) p) ? hipSuccess : fail(hipErrorInvalidValue);
}
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t) 16, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    if (own_capture) return fail(hipErrorStreamCaptureUnsupported);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = own_capture ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) {
    const hipStreamCaptureMode was = mode;
    mode = *m;
    *m = was;
    return hipSuccess;
}

hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t) 16, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }

hipError_t hipModuleLoad(hipModule_t *m, const char *) { return *m = (hipModule_t) 16, hipSuccess; }
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
hipError_t hipModuleGetGlobal(hipDeviceptr_t *p, size_t *n, hipModule_t, const char *) {
    *p = (void *) (1ull << 39);
    *n = 8u << 20;
    return hipSuccess;
}
hipError_t hipModuleGetFunction(hipFunction_t *f, hipModule_t, const char *name) {
    *f = (hipFunction_t) &*names.insert(name).first;
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned, unsigned,
                                 unsigned, hipStream_t, void **, void **) {
    launches += *(const std::string *) f;
    for (unsigned v : {gx, gy, gz, bx}) launches += " " + std::to_string(v);
    launches += "\n";
    return hipSuccess;
}

}  // extern "C"
