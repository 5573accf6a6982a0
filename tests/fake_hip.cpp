// A HIP runtime for host-side tests: memory is the host's, launches are only
// recorded, and a flag says whether the stream is "being captured".  Loaded
// with global symbols before libokf_quant.so (fakehip.py), so that the
// library's host code runs whole on a machine without a GPU.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Alloc {
    void *p;
    size_t n;
    bool freed;
};
std::map<const void *, std::string> kernels;  // host stub -> device name
std::vector<std::string> launches;            // "name gx gy gz bx by bz lds"
std::vector<Alloc> allocs;                    // in order; a freed one is kept, so no address comes back
int capturing, fail_above;                    // fail_above: KiB from which hipMalloc fails (0: never)
dim3 cfg_grid, cfg_block;
size_t cfg_lds;
hipStream_t cfg_stream;
}  // namespace

extern "C" {
void fake_capture(int on) { capturing = on; }
void fake_fail_above(int kib) { fail_above = kib; }
int fake_launches() { return (int)launches.size(); }
const char *fake_launch(int i) { return launches[i].c_str(); }
int fake_allocs() { return (int)allocs.size(); }
unsigned long long fake_alloc_bytes(int i) { return allocs[i].n; }
int fake_alloc_freed(int i) { return allocs[i].freed; }

void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    cfg_grid = g, cfg_block = b, cfg_lds = lds, cfg_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
    *g = cfg_grid, *b = cfg_block, *lds = cfg_lds, *s = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t lds, hipStream_t) {
    char t[160];
    snprintf(t, sizeof(t), " %u %u %u %u %u %u %zu", g.x, g.y, g.z, b.x, b.y, b.z, lds);
    launches.push_back(kernels[f] + t);
    return hipSuccess;
}
hipError_t hipLaunchCooperativeKernel(const void *f, dim3 g, dim3 b, void **a, unsigned lds, hipStream_t s) {
    return hipLaunchKernel(f, g, b, a, lds, s);
}
hipError_t hipMalloc(void **p, size_t n) {
    if (fail_above && n >= (size_t)fail_above << 10) return *p = nullptr, hipErrorOutOfMemory;
    *p = malloc(n);
    allocs.push_back({*p, n, false});
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
    for (auto &a : allocs)
        if (a.p == p) a.freed = true;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = calloc(1, n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) {
    *s = (hipStream_t)&capturing;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return capturing ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static char area[16];
    *p = area;
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) {
    memset(a, 0, sizeof(*a));
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 1;
    return hipSuccess;
}
// an MI355X: 256 CUs, 160 KB of LDS a workgroup
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 163840 : 0;
    return hipSuccess;
}
}
