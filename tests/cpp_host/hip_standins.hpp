// The HIP calls of a hierarchy's build, on the host: memory of the heap, kernels as nothing. A program
// that defines them and exports its symbols has the library call them. fail_at: the allocation that fails.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>

static std::map<void*, size_t> live;  // sizes
static size_t held_bytes = 0, peak_bytes = 0;
static long long calls = 0, fail_at = -1;
static hipError_t take(void** p, size_t n) {
    if (calls++ == fail_at) return hipErrorOutOfMemory;
    live[*p = std::calloc(n, 1)] = n;
    held_bytes += n;
    peak_bytes = held_bytes > peak_bytes ? held_bytes : peak_bytes;
    return hipSuccess;
}
static hipError_t give(void* p) {
    if (!p) return hipSuccess;
    const auto it = live.find(p);
    if (it == live.end()) return hipErrorInvalidValue;
    held_bytes -= it->second;
    live.erase(it);
    std::free(p);
    return hipSuccess;
}
extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return take(p, n); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return take(p, n); }
hipError_t hipFree(void* p) { return give(p); }
hipError_t hipHostFree(void* p) { return give(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    *g = *b = dim3(1);
    *m = 0;
    *s = nullptr;
    return hipSuccess;
}
}
