// Reading results back to the caller's host arrays: every column of a result
// leaves the device in one pass.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <map>
#include <memory>
#include <mutex>
#include <vector>

namespace tamd {

// Process-wide pool of pinned host blocks, in power-of-two size classes.  At
// most kMaxHeld bytes are kept (a returned block beyond that is freed);
// release() frees them all (ckf_release_cached_memory).  get() gives none above
// kMaxBlock, which would be pinned and freed again by every call (a 128 MiB
// block: 10 ms of an estimation of 3 million seeds), nor where none is to be had.
struct pinned_cache {
    static constexpr size_t kMaxHeld = size_t(64) << 20;
    static constexpr size_t kMaxBlock = size_t(32) << 20;
    std::mutex mu;
    std::map<size_t, std::vector<void*>> free_blocks;
    size_t held = 0;
    static size_t size_class(size_t bytes);
    void* get(size_t bytes);
    void put(void* p, size_t bytes);
    void release();
};

pinned_cache& staging_cache();

// A host block for transfers: a pinned one from the pool and back to it, or
// ordinary memory, which a copy takes as well (a kernel does not).  Whoever lets
// a transfer use it waits for the transfer before the block goes.
struct staging_block {
    void* const pinned;
    const size_t bytes;
    explicit staging_block(size_t n)
        : pinned(staging_cache().get(n)), bytes(n), pageable_(pinned == nullptr ? new char[n] : nullptr),
          p(pinned != nullptr ? pinned : pageable_.get()) {}
    staging_block(const staging_block&) = delete;
    staging_block& operator=(const staging_block&) = delete;
    ~staging_block() { staging_cache().put(pinned, bytes); }

private:
    const std::unique_ptr<char[]> pageable_;

public:
    void* const p;
};

// One read-back: the columns are declared, then run() fills the host arrays.
// A column whose host array is null, or that is empty, is left out.
//
// Sources start on 16 bytes and are read in whole 4-byte words: an allocation
// of a multiple of four bytes is needed, which every device block here is.
class readback {
public:
    // `device`: where the sources are (the caller's thread may be on another one)
    explicit readback(int device) : device_(device) {}
    // `bytes` bytes as they are
    void bytes(void* dst, const void* src, size_t bytes);
    // words [base, base + width) of every record of `stride` words
    void words(void* dst, const void* src, size_t n, uint32_t stride, uint32_t base, uint32_t width);
    // the 6x6 matrix of the 21 words from `base` of every record of `stride` words
    void symmetric(float* dst, const void* src, size_t n, uint32_t stride, uint32_t base);
    // ids[src[i]], or all ones past the table, or where `only_if` (one value per
    // item, may be null) is not `value`
    void identifiers(uint64_t* dst, const uint32_t* src, size_t n, const std::vector<uint64_t>& ids,
                     const uint16_t* only_if = nullptr, uint16_t value = 0);
    // On the device's null stream; returns when every host array is written.
    void run();

    static constexpr uint32_t kMaxColumns = 20;
    // A chunk's bytes, and how many chunks are on their way at most.
    static constexpr size_t kChunk = size_t(2) << 20;
    static constexpr uint32_t kSlots = 8;
    // Results from here on are copied out of the pinned blocks by kThreads threads.
    static constexpr size_t kManyBytes = size_t(6) << 20;
    static constexpr uint32_t kThreads = 4;

private:
    struct column {
        void* dst;
        const void* src;
        const uint16_t* only_if;
        const std::vector<uint64_t>* ids;
        size_t bytes;   // staged bytes that reach the host array
        size_t offset;  // of the first staged byte
        uint32_t stride, base, width;
        uint16_t value;
        uint8_t kind;
    };
    void add(column c);
    void deliver(const char* staged, size_t begin, size_t end) const;
    hipError_t launch(void* staged, size_t begin, size_t end) const;
    void run_pageable();
    const int device_;
    column cols_[kMaxColumns];
    uint32_t n_ = 0;
    size_t total_ = 0;
};

}  // namespace tamd
