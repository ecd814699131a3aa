// Host harness: result blocks and read-backs on the host runtime's devices.
#include <cstring>

#include "ckf/handles.hpp"
#include "common/readback.hpp"

namespace tamd {
block_cache& result_cache() {
    static block_cache c;
    return c;
}
std::string& last_error() {
    static thread_local std::string s;
    return s;
}
}  // namespace tamd

using host_runtime::rt;

// Blocks returned on one device are handed out on that one only, whichever
// device the thread that returns or takes them is on.  0, or a step's number.
extern "C" int cache_keeps_devices_apart() {
    using namespace tamd;
    (void)hipSetDevice(1);
    void* first = nullptr;
    {
        rbuf b;
        b.take(1000, current_device());
        first = b.p;
        if (rt().blocks[first].first != 1) return 1;
        (void)hipSetDevice(0);  // the block goes back from here
    }
    {
        rbuf b;
        b.take(1000, current_device());
        if (b.p == first || rt().blocks[b.p].first != 0) return 2;
    }
    (void)hipSetDevice(1);
    {
        rbuf b;
        b.take(1000, current_device());
        if (b.p != first) return 3;
    }
    ckf_device_tracks* t = new ckf_device_tracks();
    t->blocks[2] = result_cache().get(5000, current_device());
    t->vec = static_cast<float*>(t->blocks[2].p);
    void* vec = t->vec;
    (void)hipSetDevice(2);
    delete t;
    const device_block other = result_cache().get(5000, current_device());
    if (other.p == vec || rt().blocks[other.p].first != 2) return 4;
    result_cache().put(other);
    (void)hipSetDevice(0);
    result_cache().release();
    return rt().blocks.empty() ? 0 : 5;
}

// A result of n records (6 words, a triangle of 21, flags, identifiers) on
// `device`, read back by a thread on device 0.  0, or what is wrong.
extern "C" int read_back_from(int device, uint32_t n) {
    using namespace tamd;
    (void)hipSetDevice(device);
    rbuf rec, flag, surface;
    rec.take(128u * size_t(n), current_device());
    flag.take(size_t(n) + 3u, current_device());
    surface.take(4u * size_t(n), current_device());
    for (size_t i = 0; i < 32u * size_t(n); ++i) rec.as<uint32_t>()[i] = static_cast<uint32_t>(i * 2654435761u);
    for (uint32_t i = 0; i < n; ++i) {
        flag.as<uint8_t>()[i] = static_cast<uint8_t>(i * 7u);
        surface.as<uint32_t>()[i] = i % 5u;
    }
    const std::vector<uint64_t> ids = {11, 22, 33, 44};
    (void)hipSetDevice(0);
    uint64_t before[host_runtime::kDevices];
    std::memcpy(before, rt().launches, sizeof(before));
    std::vector<float> vec(6u * size_t(n)), cov(36u * size_t(n));
    std::vector<uint8_t> flags(n);
    std::vector<uint64_t> links(n);
    readback rb(device);
    rb.words(vec.data(), rec.p, n, 32u, 0u, 6u);
    rb.symmetric(cov.data(), rec.p, n, 32u, 6u);
    rb.bytes(flags.data(), flag.p, n);
    rb.identifiers(links.data(), surface.as<uint32_t>(), n, ids);
    rb.run();
    if (host_runtime::device != 0) return 1;  // the caller's device is his own
    for (int d = 0; d < host_runtime::kDevices; ++d) {
        if ((rt().launches[d] > before[d]) != (d == device)) return 2;
    }
    const uint32_t* r = rec.as<uint32_t>();
    for (uint32_t i = 0; i < n; ++i) {
        if (std::memcmp(&vec[6u * size_t(i)], r + 32u * size_t(i), 24u) != 0) return 3;
        for (uint32_t a = 0, k = 0; a < 6u; ++a) {
            for (uint32_t b = a; b < 6u; ++b, ++k) {
                const uint32_t* want = r + 32u * size_t(i) + 6u + k;
                if (std::memcmp(&cov[36u * size_t(i) + 6u * a + b], want, 4u) != 0) return 4;
                if (std::memcmp(&cov[36u * size_t(i) + 6u * b + a], want, 4u) != 0) return 5;
            }
        }
        if (flags[i] != static_cast<uint8_t>(i * 7u)) return 6;
        if (links[i] != (i % 5u < 4u ? ids[i % 5u] : ~0ull)) return 7;
    }
    return 0;
}

// Device bytes that a result's blocks take beyond what it needs.
extern "C" uint64_t bytes_over(const uint64_t* need, uint32_t n) {
    using namespace tamd;
    result_cache().release();
    const size_t before = rt().device_bytes;
    uint64_t sum = 0;
    std::vector<rbuf> blocks(n);
    for (uint32_t i = 0; i < n; ++i) {
        blocks[i].take(need[i], current_device());
        sum += need[i];
    }
    return rt().device_bytes - before - sum;
}

// Allocations of `calls` results one after another, their sizes around `bytes`.
extern "C" uint64_t allocations_of(uint64_t bytes, uint32_t calls) {
    using namespace tamd;
    result_cache().release();
    const size_t before = rt().allocations;
    uint32_t r = 12345u;
    for (uint32_t k = 0; k < calls; ++k) {
        r = r * 1664525u + 1013904223u;
        rbuf a, b;
        a.take(bytes * 8 / 10 + bytes * 4 / 10 * (r >> 16) / 65536, current_device());
        b.take(bytes / 3, current_device());
    }
    result_cache().release();
    return rt().allocations - before;
}

// On a device that holds `limit` bytes: a result of `idle` bytes goes to the cache,
// then a result and a work buffer of `want` bytes each are asked for.
// 0, or the step that fails.
extern "C" int room_from_the_cache(uint64_t limit, uint64_t idle, uint64_t want) {
    using namespace tamd;
    result_cache().release();
    rt().device_limit = rt().device_bytes + limit;
    int step = 0;
    dbuf work;
    try {
        {
            rbuf b;
            b.take(idle, current_device());
        }
        step = 1;
        {
            rbuf b;
            b.take(want, current_device());
        }
        step = 2;
        work.ensure(want);
        step = 3;
        rbuf b;
        b.take(limit, current_device());  // does not fit beside it
        step = 4;
    } catch (const ckf_error& e) {
        if (step == 3 && e.code == CKF_ERR_OUT_OF_MEMORY) step = 0;
    }
    work.release();
    result_cache().release();
    rt().device_limit = ~size_t(0);
    return step;
}

// Blocks for transfers of `bytes` from a pool that may pin `limit` bytes more; the
// result: the largest block pinned since the last call.
extern "C" uint64_t staging(uint64_t bytes, uint64_t limit) {
    using namespace tamd;
    staging_cache().release();
    rt().pinned_limit = rt().pinned_bytes + limit;
    rt().largest_pinned = 0;
    {
        const staging_block b(bytes);
        std::memset(b.p, 7, bytes);
    }
    rt().pinned_limit = ~size_t(0);
    return rt().largest_pinned;
}

extern "C" int read_back_without_pinned_memory(uint32_t n) {
    using namespace tamd;
    staging_cache().release();
    rt().pinned_limit = rt().pinned_bytes;
    const int r = read_back_from(1, n);
    rt().pinned_limit = ~size_t(0);
    return r;
}

// Allocations of `calls` results of two blocks after one call's blocks of `stale`
// bytes in all have gone to the cache.
extern "C" uint64_t allocations_after(uint64_t stale, uint64_t bytes, uint32_t calls) {
    using namespace tamd;
    result_cache().release();
    {
        rbuf a, b;
        a.take(stale / 4 * 3, current_device());
        b.take(stale / 4, current_device());
    }
    const size_t before = rt().allocations;
    for (uint32_t k = 0; k < calls; ++k) {
        rbuf a, b;
        a.take(bytes, current_device());
        b.take(bytes / 10, current_device());
    }
    const bool bounded = result_cache().held <= block_cache::kMaxHeld;
    result_cache().release();
    return bounded ? rt().allocations - before : ~uint64_t(0);
}

// A work buffer whose growth failed holds nothing: a smaller request allocates.
extern "C" int buffer_after_a_failed_growth() {
    using namespace tamd;
    result_cache().release();
    dbuf b;
    b.ensure(3 << 20);
    rt().device_limit = rt().device_bytes + (1 << 20);
    int step = 1;
    try {
        b.ensure(50 << 20);
    } catch (const ckf_error& e) {
        step = e.code == CKF_ERR_OUT_OF_MEMORY ? 2 : 3;
    }
    rt().device_limit = ~size_t(0);
    b.ensure(2 << 20);
    const bool there = b.p != nullptr && b.bytes >= (2 << 20);
    b.release();
    return step == 2 && there ? 0 : step;
}
