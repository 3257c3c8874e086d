// The HIP functions that the library calls, on host memory of a set capacity,
// for host tests linked against the library: the executable's definitions come
// before the runtime's.  Kernels do not run; each launch is handed to
// on_launch with the kernel's name.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

extern "C" {
size_t fake_capacity = (size_t)1 << 40, fake_used = 0;
void on_launch(const char* kernel, void** args);
}

namespace {
std::map<const void*, std::string>& names() {
    static std::map<const void*, std::string> m;
    return m;
}
std::map<char*, size_t>& live() {
    static std::map<char*, size_t> m;
    return m;
}
std::map<char*, size_t>::iterator find(const void* p) {
    auto it = live().upper_bound((char*)p);
    if (it == live().begin()) return live().end();
    --it;
    return (char*)p < it->first + it->second ? it : live().end();
}
}  // namespace

extern "C" {
int fake_is_live(const void* p) { return find(p) != live().end(); }

void** __hipRegisterFatBinary(const void*) {
    static void* h;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    names()[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
    on_launch(names()[f].c_str(), args);
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
    if (fake_used + n > fake_capacity) return hipErrorOutOfMemory;
    *p = aligned_alloc(256, (n + 255) / 256 * 256);
    memset(*p, 0xff, n);
    live()[(char*)*p] = n;
    fake_used += n;
    return hipSuccess;
}
// freed addresses are not handed out again
hipError_t hipFree(void* p) {
    auto it = live().find((char*)p);
    if (it == live().end()) return p ? hipErrorInvalidValue : hipSuccess;
    fake_used -= it->second;
    live().erase(it);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* free_b, size_t* total) {
    *total = fake_capacity;
    *free_b = fake_capacity - fake_used;
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
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    memset(a, 0, sizeof *a);
    if (!fake_is_live(p)) return hipErrorInvalidValue;
    a->type = hipMemoryTypeDevice;
    return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p) {
    auto it = find(p);
    if (it == live().end()) return hipErrorInvalidValue;
    *base = it->first;
    *size = it->second;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static char* scratch = (char*)calloc(1, 64 << 20);
    *p = scratch;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = (hipStream_t)&fake_used;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = (hipEvent_t)&fake_used;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1;
    return hipSuccess;
}
}
