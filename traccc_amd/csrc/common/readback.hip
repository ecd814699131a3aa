// Read-back of results: one kernel writes all columns of a result, in the
// layout of the host arrays, into pinned host memory, and the host copies them
// on from there.
//
// What bounds it: the link (57 GB/s) and the host's copy (31 GB/s with one
// thread).  A copy of its own for each column costs 11 us at 64 bytes, 33 us at
// 64 KiB and 110 us at 256 KiB, because the caller's pages are not pinned, and
// 3.8 ms for 64 MiB, because the transfer and the host's copy out of the
// runtime's staging take turns.  Here a result's 11 to 19 columns cost one
// launch; from 2 MiB on they pass in chunks, so that the link and the host work
// at the same time, and from 6 MiB on four threads copy (64 MiB out of pinned
// memory: 2.0 ms with one thread, 0.85 with four; starting them takes 40 us).
#include "readback.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

#include "device.hpp"
#include "errors.hpp"

namespace tamd {

size_t pinned_cache::size_class(size_t bytes) {
    size_t c = 4096;
    while (c < bytes) c <<= 1;
    return c;
}

void* pinned_cache::get(size_t bytes) {
    if (bytes > kMaxBlock) return nullptr;
    const size_t c = size_class(bytes);
    {
        std::lock_guard<std::mutex> lk(mu);
        auto it = free_blocks.find(c);
        if (it != free_blocks.end() && !it->second.empty()) {
            void* p = it->second.back();
            it->second.pop_back();
            held -= c;
            return p;
        }
    }
    void* p = nullptr;
    if (hipHostMalloc(&p, c, hipHostMallocPortable | hipHostMallocMapped) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return p;
}

void pinned_cache::put(void* p, size_t bytes) {
    if (p == nullptr) return;
    const size_t c = size_class(bytes);
    std::lock_guard<std::mutex> lk(mu);
    if (held + c > kMaxHeld) {
        (void)hipHostFree(p);
        return;
    }
    free_blocks[c].push_back(p);
    held += c;
}

void pinned_cache::release() {
    std::lock_guard<std::mutex> lk(mu);
    for (auto& kv : free_blocks) {
        for (void* p : kv.second) (void)hipHostFree(p);
    }
    free_blocks.clear();
    held = 0;
}

pinned_cache& staging_cache() {
    static pinned_cache* c = new pinned_cache();  // never destroyed: outlives the HIP runtime's exit
    return *c;
}

namespace {

struct pinned_scope {
    void* const p;
    const size_t bytes;
    explicit pinned_scope(size_t n) : p(staging_cache().get(n)), bytes(n) {}
    pinned_scope(const pinned_scope&) = delete;
    pinned_scope& operator=(const pinned_scope&) = delete;
    ~pinned_scope() { staging_cache().put(p, bytes); }
};

enum : uint8_t { kPlain = 0, kWords = 1, kSymmetric = 2, kMasked = 3 };

// A column's part of one chunk.  `src` and `only_if` are at the item of the
// part's first word, `phase` is that word's place in its item.
struct part {
    const uint32_t* src;
    const uint16_t* only_if;
    uint32_t begin, end;  // words of the chunk
    uint32_t phase, stride, base, width;
    uint16_t value;
    uint8_t kind;
};

struct chunk {
    part parts[readback::kMaxColumns];
    uint32_t n_parts;
    uint32_t n_words;
};

constexpr int kPackBlock = 256;

__device__ uint32_t packed_word(const part& q, uint32_t w) {
    if (q.kind == kPlain) return q.src[w];
    if (q.kind == kMasked) return q.only_if[w] == q.value ? q.src[w] : 0xffffffffu;
    const uint32_t g = q.phase + w, item = g / q.width, k = g - item * q.width;
    uint32_t f = k;
    if (q.kind == kSymmetric) {
        // upper triangle by rows: (i, j), i <= j, is word 6 i - i (i - 1) / 2 + j - i
        const uint32_t r = k / 6u, c = k - 6u * r, i = min(r, c), j = max(r, c);
        f = 6u * i - (i * (i - 1u)) / 2u + j - i;
    }
    return q.src[size_t(item) * q.stride + q.base + f];
}

// Four words of the chunk per thread, written as one 16-byte piece.  Columns
// start on 16 bytes of the chunk, so a piece belongs to one column.
__global__ void __launch_bounds__(kPackBlock) k_pack(chunk C, uint4* __restrict__ out) {
    const uint32_t piece = blockIdx.x * kPackBlock + threadIdx.x, w0 = 4u * piece;
    if (w0 >= C.n_words) return;
    uint32_t v[4] = {0u, 0u, 0u, 0u};
    for (uint32_t c = 0; c < C.n_parts; ++c) {
        const part& q = C.parts[c];
        if (w0 < q.begin || w0 >= q.end) continue;
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) {
            if (w0 + k < q.end) v[k] = packed_word(q, w0 + k - q.begin);
        }
    }
    out[piece] = make_uint4(v[0], v[1], v[2], v[3]);
}

}  // namespace

void readback::add(column c) {
    if (c.dst == nullptr || c.bytes == 0u) return;
    if (n_ == kMaxColumns) throw ckf_error(CKF_ERR_INTERNAL, "read-back columns");
    c.offset = total_;
    total_ += (c.bytes + 15u) & ~size_t(15);
    cols_[n_++] = c;
}

void readback::bytes(void* dst, const void* src, size_t bytes) {
    add({dst, src, nullptr, nullptr, bytes, 0, 1, 0, 1, 0, kPlain});
}

void readback::words(void* dst, const void* src, size_t n, uint32_t stride, uint32_t base, uint32_t width) {
    add({dst, src, nullptr, nullptr, 4u * n * width, 0, stride, base, width, 0, kWords});
}

void readback::symmetric(float* dst, const void* src, size_t n, uint32_t stride, uint32_t base) {
    add({dst, src, nullptr, nullptr, 144u * n, 0, stride, base, 36, 0, kSymmetric});
}

void readback::identifiers(uint64_t* dst, const uint32_t* src, size_t n, const std::vector<uint64_t>& ids,
                           const uint16_t* only_if, uint16_t value) {
    add({dst, src, only_if, &ids, 4u * n, 0, 1, 0, 1, value, only_if != nullptr ? kMasked : kPlain});
}

// Staged bytes [begin, end) on the device into `staged`.
hipError_t readback::launch(void* staged, size_t begin, size_t end) const {
    chunk C{};
    for (uint32_t c = 0; c < n_; ++c) {
        const column& k = cols_[c];
        const size_t words = (k.bytes + 3u) / 4u;
        const size_t b = std::max(begin, k.offset), e = std::min(end, k.offset + 4u * words);
        if (b >= e) continue;
        const size_t first = (b - k.offset) / 4u, item = first / k.width;
        part& q = C.parts[C.n_parts++];
        q.src = static_cast<const uint32_t*>(k.src) + item * k.stride;
        q.only_if = k.only_if != nullptr ? k.only_if + item : nullptr;
        q.begin = static_cast<uint32_t>((b - begin) / 4u);
        q.end = static_cast<uint32_t>((e - begin) / 4u);
        q.phase = static_cast<uint32_t>(first - item * k.width);
        q.stride = k.stride;
        q.base = k.base;
        q.width = k.width;
        q.value = k.value;
        q.kind = k.kind;
    }
    C.n_words = static_cast<uint32_t>((end - begin) / 4u);
    const uint32_t pieces = (C.n_words + 3u) / 4u;
    hipLaunchKernelGGL(k_pack, dim3((pieces + kPackBlock - 1) / kPackBlock), dim3(kPackBlock), 0, nullptr, C,
                       static_cast<uint4*>(staged));
    return hipGetLastError();
}

// Staged bytes [begin, end), at `staged`, into the host arrays.
void readback::deliver(const char* staged, size_t begin, size_t end) const {
    for (uint32_t c = 0; c < n_; ++c) {
        const column& k = cols_[c];
        const size_t b = std::max(begin, k.offset), e = std::min(end, k.offset + k.bytes);
        if (b >= e) continue;
        const char* src = staged + (b - begin);
        if (k.ids == nullptr) {
            std::memcpy(static_cast<char*>(k.dst) + (b - k.offset), src, e - b);
            continue;
        }
        const uint32_t* sf = reinterpret_cast<const uint32_t*>(src);
        uint64_t* dst = static_cast<uint64_t*>(k.dst) + (b - k.offset) / 4u;
        const uint64_t* ids = k.ids->data();
        const size_t n_ids = k.ids->size();
        for (size_t i = 0, m = (e - b) / 4u; i < m; ++i) dst[i] = sf[i] < n_ids ? ids[sf[i]] : ~0ull;
    }
}

// Without pinned memory: each chunk through a device block, copied as the runtime
// copies to any memory.
void readback::run_pageable() {
    const size_t block = std::min(total_, kChunk);
    const std::unique_ptr<char[]> host(new char[block]);
    void* dev = nullptr;
    hip_check(hipMalloc(&dev, block), "hipMalloc");
    hipError_t e = hipSuccess;
    for (size_t begin = 0; begin < total_ && e == hipSuccess; begin += block) {
        const size_t end = std::min(total_, begin + block);
        e = launch(dev, begin, end);
        if (e == hipSuccess) e = hipMemcpy(host.get(), dev, end - begin, hipMemcpyDeviceToHost);
        if (e == hipSuccess) deliver(host.get(), begin, end);
    }
    (void)hipFree(dev);
    hip_check(e, "download");
}

void readback::run() {
    if (total_ == 0u) return;
    const device_scope on(device_);
    hip_check(on.status, "hipSetDevice");
    const size_t n_chunks = (total_ + kChunk - 1u) / kChunk;
    const size_t slots = std::min<size_t>(n_chunks, kSlots);
    const size_t block = n_chunks == 1u ? total_ : slots * kChunk;
    const pinned_scope held(block);
    if (held.p == nullptr) {
        run_pageable();
        return;
    }
    char* const staged = static_cast<char*>(held.p);
    auto begin = [&](size_t c) { return c * kChunk; };
    auto end = [&](size_t c) { return std::min(total_, (c + 1u) * kChunk); };
    auto slot = [&](size_t c) { return staged + (c % slots) * kChunk; };

    if (n_chunks == 1u) {
        hipError_t e = launch(staged, 0, total_);
        const hipError_t w = hipStreamSynchronize(nullptr);
        if (e == hipSuccess) e = w;
        if (e == hipSuccess) deliver(staged, 0, total_);
        hip_check(e, "download");
        return;
    }

    // This thread makes every HIP call; the helpers only copy: of each chunk
    // that has arrived, thread j copies the j-th part.
    const uint32_t helpers = total_ >= kManyBytes ? kThreads - 1u : 0u;
    std::atomic<size_t> arrived{0};
    std::atomic<bool> stop{false};
    std::vector<std::atomic<size_t>> copied(helpers);  // chunks each helper has finished
    for (auto& c : copied) c.store(0);
    std::vector<std::thread> threads;
    uint32_t n_threads = 1u;
    std::atomic<uint32_t> share{0};  // threads that copy, once known
    auto copy = [&](size_t c, uint32_t j, uint32_t of) {
        const size_t n = end(c) - begin(c), piece = ((n + of - 1u) / of + 15u) & ~size_t(15);
        const size_t lo = std::min(n, j * piece), hi = std::min(n, lo + piece);
        if (lo < hi) deliver(slot(c) + lo, begin(c) + lo, begin(c) + hi);
    };
    auto help = [&](uint32_t j) {
        for (size_t c = 0; c < n_chunks; ++c) {
            while (arrived.load(std::memory_order_acquire) <= c) {
                if (stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            copy(c, j + 1u, share.load(std::memory_order_relaxed));
            copied[j].store(c + 1u, std::memory_order_release);
        }
    };

    std::vector<hipEvent_t> done(slots, nullptr);
    threads.reserve(helpers);
    hipError_t e = hipSuccess;
    for (auto& v : done) {
        if (e == hipSuccess) e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
    }
    auto start = [&](size_t c) {
        if (e == hipSuccess) e = launch(slot(c), begin(c), end(c));
        if (e == hipSuccess) e = hipEventRecord(done[c % slots], nullptr);
    };
    for (size_t c = 0; c < slots; ++c) start(c);
    try {
        for (uint32_t j = 0; j < helpers && e == hipSuccess; ++j, ++n_threads) threads.emplace_back(help, j);
    } catch (...) {
        // no thread to be had: those there are share the work
    }
    share.store(n_threads, std::memory_order_relaxed);
    for (size_t c = 0; c < n_chunks && e == hipSuccess; ++c) {
        e = hipEventSynchronize(done[c % slots]);
        if (e != hipSuccess) break;
        arrived.store(c + 1u, std::memory_order_release);
        copy(c, 0u, n_threads);
        for (uint32_t j = 0; j + 1u < n_threads; ++j) {
            while (copied[j].load(std::memory_order_acquire) <= c) std::this_thread::yield();
        }
        if (c + slots < n_chunks) start(c + slots);
    }
    stop.store(true, std::memory_order_relaxed);
    for (auto& t : threads) t.join();
    for (auto& v : done) {
        if (v != nullptr) (void)hipEventDestroy(v);
    }
    if (e != hipSuccess) (void)hipStreamSynchronize(nullptr);
    hip_check(e, "download");
}

}  // namespace tamd
