// fake_hip.h — a HIP runtime without a device, for programs that link librocketnpu's objects on a
// machine without a GPU: device memory is host memory, kernels are recorded and not run, a stream is
// always done, and a switch makes it look captured. Included by one source file of a program.
#pragma once

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <set>
#include <string>
#include <vector>

namespace fake {

struct State {
    bool capturing = false;
    size_t limit = (size_t)-1;             // a larger allocation fails
    std::map<char *, size_t> live;         // device allocations
    int allocs = 0, frees = 0, syncs = 0;
    std::vector<std::string> launches;     // kernel names, in order
    std::map<const void *, std::string> names;
    dim3 grid, block;
    size_t lds = 0;
    hipStream_t stream = nullptr;
};
inline State &st()
{
    static State *s = new State;   // (the modules register before main)
    return *s;
}
inline int count(const char *part)
{
    int n = 0;
    for (const auto &l : st().launches) n += l.find(part) != std::string::npos;
    return n;
}

}  // namespace fake

extern "C" {

void **__hipRegisterFatBinary(const void *)
{
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    fake::st().names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    auto &f = fake::st();
    f.grid = g, f.block = b, f.lds = lds, f.stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    auto &f = fake::st();
    *g = f.grid, *b = f.block, *lds = f.lds, *s = f.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3, dim3, void **, size_t, hipStream_t)
{
    fake::st().launches.push_back(fake::st().names[fn]);
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n)
{
    auto &f = fake::st();
    if (f.capturing || n > f.limit) return hipErrorOutOfMemory;
    char *m = nullptr;
    if (posix_memalign(reinterpret_cast<void **>(&m), 256, n)) return hipErrorOutOfMemory;
    f.live[m] = n;
    f.allocs++;
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    auto &f = fake::st();
    if (!p) return hipSuccess;
    if (!f.live.erase(static_cast<char *>(p))) return hipErrorInvalidValue;
    f.frees++;
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned)
{
    *d = h;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static char array[16 << 20];
    *p = array;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    memset(a, 0, sizeof *a);
    for (const auto &m : fake::st().live)
        if (p >= m.first && p < m.first + m.second) {
            a->type = hipMemoryTypeDevice;
            return hipSuccess;
        }
    return hipErrorInvalidValue;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = reinterpret_cast<hipStream_t>(0x10);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c)
{
    *c = fake::st().capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return fake::st().capturing ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t)
{
    auto &f = fake::st();
    f.syncs++;
    return f.capturing ? hipErrorStreamCaptureUnsupported : hipSuccess;
}

}  // extern "C"
