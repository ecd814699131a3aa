// Handles of the C ABI shared by the CKF and the fitter runtimes: device
// buffers, the per-call result block cache, and the device-resident
// detector, events and track candidates.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <map>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

#include "../common/device.hpp"
#include "../common/errors.hpp"
#include "traccc_amd/ckf.h"
#include "../core/geometry.hpp"

namespace tamd {

// A device block of the cache: its own size, and the device it is on.
struct device_block {
    void* p = nullptr;
    size_t size = 0;
    int device = 0;
};

// Process-wide cache of device blocks for per-call results: freed blocks are
// kept by device and size and handed out again, so a steady stream of operator
// calls does not call hipMalloc / hipFree.  At most kMaxHeld bytes are kept: for
// a returned block the ones that have waited longest go (pruned calls of 64 x
// 60,000 pions after plain ones, whose blocks are twice as large: 47.8 ms, 49.0
// where those stayed and every call allocated its own).  release() frees them all
// (ckf_release_cached_memory), and so does an allocation that finds the device full.
//
// New blocks are a power of two up to kGrain, then an eighth larger than asked
// for up to kMedium and a sixteenth up to kLarge, in steps of a sixteenth of the
// power of two below: the next event's result, a few percent larger, finds them
// then.  (First call on other events, us: seeding of 10,000 muons 2,600, 2,650
// where it allocates; fit and resolution of 2 x 60,000 pions 5,650 and 6,200.)
// From kLarge on they are what is asked for: rounded up to a power of two, the fit
// of 37 million states took 16 GiB for records of 9.6.  A request is served by the
// smallest free block that holds it and is at most twice what a new one would be.
struct block_cache {
    static constexpr size_t kMaxHeld = size_t(4) << 30;
    static constexpr size_t kGrain = size_t(2) << 20;
    static constexpr size_t kMedium = size_t(256) << 20;
    static constexpr size_t kLarge = size_t(1) << 30;
    std::mutex mu;
    struct waiting {
        void* p;
        uint64_t since;
    };
    std::map<std::pair<int, size_t>, std::vector<waiting>> free_blocks;  // (device, size); none empty
    size_t held = 0;
    uint64_t puts = 0;
    static size_t block_size(size_t bytes) {
        size_t c = 256;
        while (c < bytes) c <<= 1;
        if (c <= kGrain) return c;
        const size_t step = c > kLarge ? kGrain : c / 32;
        if (bytes <= kLarge) bytes += bytes <= kMedium ? bytes / 8 : bytes / 16;
        return (bytes + step - 1) / step * step;
    }
    // A block on the calling thread's current device, `device`.
    device_block get(size_t bytes, int device) {
        const size_t c = block_size(bytes);
        std::unique_lock<std::mutex> lk(mu);
        const auto it = free_blocks.lower_bound({device, bytes});
        if (it != free_blocks.end() && it->first.first == device && it->first.second <= 2 * c) {
            const device_block b{it->second.back().p, it->first.second, device};
            it->second.pop_back();
            held -= b.size;
            if (it->second.empty()) free_blocks.erase(it);
            return b;
        }
        lk.unlock();
        return {allocate(c), c, device};
    }
    // Back to the cache, from whichever thread.
    void put(const device_block& b) {
        if (b.p == nullptr) return;
        std::lock_guard<std::mutex> lk(mu);
        if (b.size > kMaxHeld) {
            (void)hipFree(b.p);
            return;
        }
        while (held + b.size > kMaxHeld) drop_oldest();
        free_blocks[{b.device, b.size}].push_back({b.p, puts++});
        held += b.size;
    }
    // Of each size the first one has waited longest.
    void drop_oldest() {
        auto oldest = free_blocks.end();
        for (auto it = free_blocks.begin(); it != free_blocks.end(); ++it) {
            if (oldest == free_blocks.end() || it->second.front().since < oldest->second.front().since) oldest = it;
        }
        (void)hipFree(oldest->second.front().p);
        oldest->second.erase(oldest->second.begin());
        held -= oldest->first.second;
        if (oldest->second.empty()) free_blocks.erase(oldest);
    }
    // hipMalloc; where the device is full, once more without the cached blocks.
    void* allocate(size_t bytes) {
        void* p = nullptr;
        hipError_t e = hipMalloc(&p, bytes);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            release();
            e = hipMalloc(&p, bytes);
        }
        hip_check(e, "hipMalloc");
        return p;
    }
    void release() {
        std::lock_guard<std::mutex> lk(mu);
        for (auto& kv : free_blocks) {
            for (const waiting& w : kv.second) (void)hipFree(w.p);
        }
        free_blocks.clear();
        held = 0;
    }
};

block_cache& result_cache();

// Device memory that is no result: the cached results' make room for it.
inline void* device_alloc(size_t bytes) { return result_cache().allocate(bytes); }

// Device allocation that grows by doubling and is reused across calls.
struct dbuf {
    void* p = nullptr;
    size_t bytes = 0;
    void ensure(size_t need) {
        if (need <= bytes) {
            return;
        }
        if (p != nullptr) {
            tamd::hip_check(hipFree(p), "hipFree");
            p = nullptr;
        }
        size_t nb = std::max<size_t>(need, bytes * 2);
        bytes = 0;  // of nothing, should the allocation fail
        nb = (nb + 255) & ~size_t(255);
        p = device_alloc(nb);
        bytes = nb;
    }
    void release() {
        if (p != nullptr) {
            (void)hipFree(p);
        }
        p = nullptr;
        bytes = 0;
    }
    template <typename T>
    T* as() const {
        return static_cast<T*>(p);
    }
};

// A result's device block, from the result cache and back to it.  Contents are
// whatever the block held before: the kernels of a result write all of it.
struct rbuf {
    void* p = nullptr;
    rbuf() = default;
    rbuf(const rbuf&) = delete;
    rbuf& operator=(const rbuf&) = delete;
    ~rbuf() { result_cache().put(block_); }
    void take(size_t need, int device) {
        result_cache().put(block_);
        block_ = {};
        block_ = result_cache().get(need, device);
        p = block_.p;
    }
    template <typename T>
    T* as() const {
        return static_cast<T*>(p);
    }

private:
    device_block block_;
};

// Surface index -> identifier, made once per detector and held by its results.
using id_table = std::shared_ptr<const std::vector<uint64_t>>;

template <typename T>
T* dev_copy(const T* src, size_t n) {
    T* d = static_cast<T*>(device_alloc(std::max<size_t>(n, 1) * sizeof(T)));
    if (n > 0 && src != nullptr) {
        tamd::hip_check(hipMemcpy(d, src, n * sizeof(T), hipMemcpyHostToDevice), "hipMemcpy H2D");
    }
    return d;
}

}  // namespace tamd

struct ckf_device_detector {
    std::vector<ckf_surface> h_sfs;
    std::vector<ckf_layer> h_layers;
    tamd::id_table ids;
    ckf_bfield field{};
    ckf_surface* d_sfs = nullptr;
    ckf_layer* d_layers = nullptr;
    // the navigator's layer groups (tamd::build_layer_groups)
    std::vector<tamd::layer_group> h_groups;
    tamd::layer_group* d_groups = nullptr;
    float* d_map = nullptr;
    ~ckf_device_detector() {
        if (d_sfs) (void)hipFree(d_sfs);
        if (d_groups) (void)hipFree(d_groups);
        if (d_layers) (void)hipFree(d_layers);
        if (d_map) (void)hipFree(d_map);
    }
};

struct ckf_device_event {
    uint32_t n_events = 0, n_meas = 0, n_seeds = 0, n_surfaces = 0;
    std::vector<uint32_t> meas_off, seed_off;  // [n_events + 1]
    float2* d_pos = nullptr;
    float2* d_var = nullptr;
    uint32_t* d_info = nullptr;
    uint32_t* d_ranges = nullptr;
    uint32_t* d_seed_event = nullptr;
    uint32_t* d_seed_surface = nullptr;
    float* d_seed_vec = nullptr;
    float* d_seed_cov = nullptr;
    uint32_t* d_meas_off = nullptr;
    uint32_t* d_meas_sf = nullptr;  // surface index of every measurement
    float* d_win_var = nullptr;     // per event: largest loc0 variance, or -1 (no window search)
    ~ckf_device_event() {
        void* ps[] = {d_pos, d_var, d_info, d_ranges, d_seed_event, d_seed_surface,
                      d_seed_vec, d_seed_cov, d_meas_off, d_meas_sf, d_win_var};
        for (void* p : ps) {
            if (p) (void)hipFree(p);
        }
    }
};

// Fitted tracks in HBM (ckf_fit_tracks): per-track columns, the
// candidates' constituents (event-relative measurement indices) and the
// per-state filtered / smoothed records.
struct ckf_device_fitted {
    uint32_t n_tracks = 0, n_states = 0;
    int device = tamd::current_device();
    tamd::id_table ids;
    std::vector<uint32_t> ev_track_off;   // [n_events + 1] tracks of each event
    tamd::rbuf outcome, surface, vec, cov, ndf, chi2, pval, nholes, offsets, cons, flt, smt, flags,
        state_sf;
};

struct ckf_device_tracks {
    uint32_t n_events = 0, n_tracks = 0, n_const = 0;
    int device = tamd::current_device();
    std::vector<uint32_t> ev_track_off, ev_const_off;
    tamd::id_table ids;
    uint16_t* outcome = nullptr;
    uint32_t* surface = nullptr;
    float* vec = nullptr;
    float* cov = nullptr;
    float* ndf = nullptr;
    float* chi2 = nullptr;
    float* pval = nullptr;
    uint32_t* nholes = nullptr;
    uint32_t* offsets = nullptr;
    uint32_t* cons = nullptr;
    tamd::device_block blocks[10];  // of the columns, in that order
    ~ckf_device_tracks() {
        for (const tamd::device_block& b : blocks) tamd::result_cache().put(b);
    }
};

