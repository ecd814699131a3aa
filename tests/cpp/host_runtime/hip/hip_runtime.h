// A runtime of several devices on the host, for checks of the code around the
// kernels: allocations belong to the device that was current, kernels run as
// loops on the calling thread and count for its current device, and both kinds
// of allocation can be made to fail.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <map>
#include <mutex>

using hipError_t = int;
using hipStream_t = void*;
using hipEvent_t = void*;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidDevice = 101, hipErrorOutOfMemory = 2;
constexpr unsigned hipHostMallocPortable = 1, hipHostMallocMapped = 2, hipEventDisableTiming = 2;
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };

namespace host_runtime {
constexpr int kDevices = 3;
struct state {
    std::mutex mu;
    std::map<void*, std::pair<int, size_t>> blocks;  // device blocks: device, bytes
    std::map<void*, size_t> pinned;
    size_t device_bytes = 0, pinned_bytes = 0, largest_pinned = 0, allocations = 0;
    size_t device_limit = ~size_t(0), pinned_limit = ~size_t(0);
    uint64_t launches[kDevices] = {};
};
inline state& rt() {
    static state s;
    return s;
}
inline thread_local int device = 0;
struct dim3_ {
    unsigned x;
};
inline thread_local dim3_ thread_idx, block_idx;
}  // namespace host_runtime

#define __global__
#define __device__
#define __host__
#define __launch_bounds__(...)
#define threadIdx host_runtime::thread_idx
#define blockIdx host_runtime::block_idx

struct float2 {
    float x, y;
};
struct alignas(16) uint4 {
    uint32_t x, y, z, w;
};
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return {x, y, z, w}; }
struct dim3 {
    unsigned x;
    explicit dim3(unsigned n = 1) : x(n) {}
};
using std::max;
using std::min;

inline const char* hipGetErrorString(hipError_t e) {
    return e == hipSuccess ? "success" : e == hipErrorOutOfMemory ? "out of memory" : "error";
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) {
    *d = host_runtime::device;
    return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
    if (d < 0 || d >= host_runtime::kDevices) return hipErrorInvalidDevice;
    host_runtime::device = d;
    return hipSuccess;
}
template <typename T>
hipError_t hipMalloc(T** p, size_t n) {
    auto& s = host_runtime::rt();
    std::lock_guard<std::mutex> lk(s.mu);
    if (s.device_bytes + n > s.device_limit) return hipErrorOutOfMemory;
    // backed lazily: checks of sizes ask for more than a host has
    void* q = std::malloc(n);
    if (q == nullptr) return hipErrorOutOfMemory;
    s.blocks[q] = {host_runtime::device, n};
    s.device_bytes += n;
    ++s.allocations;
    *p = static_cast<T*>(q);
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    auto& s = host_runtime::rt();
    std::lock_guard<std::mutex> lk(s.mu);
    auto it = s.blocks.find(p);
    if (it == s.blocks.end()) return p == nullptr ? hipSuccess : hipErrorInvalidDevice;
    s.device_bytes -= it->second.second;
    s.blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
template <typename T>
hipError_t hipHostMalloc(T** p, size_t n, unsigned = 0) {
    auto& s = host_runtime::rt();
    std::lock_guard<std::mutex> lk(s.mu);
    if (s.pinned_bytes + n > s.pinned_limit) return hipErrorOutOfMemory;
    void* q = std::aligned_alloc(256, (n + 255) / 256 * 256);
    s.pinned[q] = n;
    s.pinned_bytes += n;
    s.largest_pinned = std::max(s.largest_pinned, n);
    *p = static_cast<T*>(q);
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    auto& s = host_runtime::rt();
    std::lock_guard<std::mutex> lk(s.mu);
    s.pinned_bytes -= s.pinned[p];
    s.pinned.erase(p);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::copy_n(static_cast<const char*>(s), n, static_cast<char*>(d));
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
    return hipMemcpy(d, s, n, k);
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }

template <typename K, typename... A>
void host_launch(K kernel, dim3 grid, dim3 block, A... args) {
    ++host_runtime::rt().launches[host_runtime::device];
    for (unsigned b = 0; b < grid.x; ++b) {
        for (unsigned t = 0; t < block.x; ++t) {
            host_runtime::block_idx = {b};
            host_runtime::thread_idx = {t};
            kernel(args...);
        }
    }
}
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) host_launch(kernel, grid, block, __VA_ARGS__)
