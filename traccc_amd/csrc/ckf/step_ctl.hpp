// The step control block: what the kernels of a step hand each other and the
// step loop, how a compaction splits its items, and the advance to the next step.
// Plain code for the device and for the host's checks.
#pragma once

#include <cstdint>

#include "../core/defs.hpp"

namespace tamd {

constexpr int kTickets = 9;  // work queues of the control block
constexpr uint32_t kCtlXcds = 8u;

// A counter alone on its 128-byte cache line.  The work-queue counters take
// an atomic per partition from every wave of a grid; counters sharing a line
// (with each other, or with the fields every wave reads at kernel start) are
// served one after another by that line's L2 channel.
struct alignas(128) line_u32 {
    uint32_t v;
};
struct alignas(128) line_u64 {
    uint64_t v;
};
static_assert(sizeof(line_u32) == 128 && sizeof(line_u64) == 128, "one counter per line");

// Step control block in device memory; the step loop reads and advances it
// without host round trips.  The fields every wave reads at kernel start
// share the first line; each counter that waves hammer with atomics has its
// own.
struct step_ctl {
    uint32_t step;        // current CKF step
    uint32_t epoch;       // tag of this step's look-back descriptors
    uint32_t n_in;        // inputs of this step
    uint32_t link_base;   // global index of this step's first link
    uint32_t n_links;     // links made this step (written by find), 0 from its advance on
    uint32_t n_live;      // inputs of the next step (written by propagate)
    uint32_t n_tips;      // tips recorded before this step
    uint32_t n_tips_step; // tips recorded this step (written by propagate)
    uint32_t overflow;    // bit 0 links, bit 1 per-step states, bit 2 filtered, bit 3 tips, bit 4 inputs
    uint32_t done;
    uint32_t n_steps_run;
    uint32_t n_tracks;
    uint32_t n_constituents;
    uint32_t prev_link_base;  // global index of the previous step's first link
    uint32_t emit_links;  // n_links for k_prop_emit: written by find, left alone by the advance
    uint64_t n_links_total;
    uint64_t n_scored;        // scorer rows of the finished steps
    uint64_t n_deferred;      // propagations of the finished steps that asked to be deferred
    line_u32 ticket[kTickets];  // work-queue tickets: [0] progressive filter, [1] votes /
                                // progressive filter, [2] free, [3] build, [4] find emit,
                                // [5] propagate emit, [6] free, [7] resume, [8] free
    line_u32 exit_count;  // partitions that k_prop_emit has written this step
    line_u32 n_rows;      // scorer rows scored this step (added up by k_score_update)
    line_u64 n_props;     // propagations so far
    line_u32 n_defer;     // links whose propagation k_propagate_resume continues (this step)
    line_u32 xcd_ticket[4][kCtlXcds];  // per-XCD work queues (one counter per XCD): find,
                                       // scorer list, propagate, dedup mark
};

// Overflow bits raised by k_find (links, filtered states).  Later kernels of
// the step only read these: the bits k_propagate raises itself must not change
// the partition count its waves see mid-kernel.
constexpr uint32_t kFindOverflow = 1u | 4u;

// Links of this step that exist: a step whose find kernel overflowed a buffer
// is abandoned (the host regrows and re-runs), so nothing walks missing links.
// For kernels between k_find_emit and k_prop_emit; k_prop_emit, in which the
// control block advances, has emit_extent.
TAMD_HD uint32_t step_links(const step_ctl& ctl, uint32_t state_cap, uint32_t link_cap) {
    if ((ctl.overflow & kFindOverflow) != 0u) {
        return 0u;
    }
    uint32_t n = ctl.n_links;
    n = n < state_cap ? n : state_cap;
    const uint32_t room = link_cap > ctl.link_base ? link_cap - ctl.link_base : 0u;
    return n < room ? n : room;
}

// Chunks of kEmitBlock items per partition for n items: one until there are
// `parts` partitions, then more, at most kEmitChunks.  A look-back round trip
// covers 64 partitions, so that many keep its chain at a round (k_prop_emit,
// 200,000 links: 12 us, 24 with 512); k_find_emit, whose items cost more than
// the chain, takes two for every CU (with duplicate lists to make, 160,000
// inputs: 38 us, 60 with 64).
constexpr uint32_t kEmitBlock = 256;
constexpr uint32_t kEmitChunks = 4;
constexpr uint32_t kLightParts = 64u, kHeavyParts = 512u;
TAMD_HD uint32_t emit_chunks(uint32_t n, uint32_t parts) {
    const uint32_t c = n / (kEmitBlock * parts);
    return c < 1u ? 1u : (c > kEmitChunks ? kEmitChunks : c);
}

// What a block of k_prop_emit goes by: the step's links, chunks per partition
// and partitions (none in a step abandoned by an overflow).
//
// The block that writes the step's last partition advances the control block, so
// a block that starts late may see any mixture of the step's words and the next
// step's.  The extent comes from words that the advance leaves alone (emit_links,
// and the overflow bits of the find, which only earlier kernels raise), so every
// block of the launch has the same one and a late block finds done or the spent
// queue, which k_find_emit clears in the next step.  From n_links and link_base
// it could not: with one of them advanced and the other not, the clamp to the
// link buffer gives fewer links, which may make more partitions (32,768 links
// are 64 partitions, 32,767 are 128), and a block would wait for ever for the
// predecessor of a partition that does not exist.  No clamp is needed: links
// past a buffer raise an overflow bit.
struct emit_extent {
    uint32_t n, chunks, parts;
};
TAMD_HD emit_extent emit_extent_of(const step_ctl& ctl) {
    const uint32_t n = (ctl.overflow & kFindOverflow) != 0u ? 0u : ctl.emit_links;
    const uint32_t chunks = emit_chunks(n, kLightParts);
    const uint32_t part = kEmitBlock * chunks;
    return {n, chunks, (n + part - 1u) / part};
}

// Step advance: move the control block to the next step.  Run by one lane once
// the step's propagation and its compaction have finished; `overflow` is the
// word as other blocks of the same kernel have left it.
TAMD_HD void advance_ctl(step_ctl* ctl, uint32_t max_cands, uint32_t overflow) {
    const uint32_t n_links = ctl->n_links;
    ctl->n_links_total += n_links;
    ctl->n_tips += ctl->n_tips_step;
    ctl->n_tips_step = 0u;
    ctl->prev_link_base = ctl->link_base;
    ctl->link_base += n_links;
    ctl->n_in = ctl->n_live;
    ctl->n_live = 0u;
    ctl->n_links = 0u;
    ctl->n_scored += ctl->n_rows.v;
    ctl->n_rows.v = 0u;
    ctl->step += 1u;
    ctl->n_steps_run = ctl->step;
    ctl->epoch += 1u;
    for (int k = 0; k < kTickets; ++k) {
        if (k != 5) ctl->ticket[k].v = 0u;  // [5] is still being taken from: see emit_extent
    }
    ctl->n_deferred += ctl->n_defer.v;
    ctl->n_defer.v = 0u;
    for (int q = 0; q < 4; ++q) {
        for (uint32_t x = 0; x < kCtlXcds; ++x) ctl->xcd_ticket[q][x].v = 0u;
    }
    if (ctl->n_in == 0u || ctl->step >= max_cands || overflow != 0u) {
        ctl->done = 1u;
    }
}

}  // namespace tamd
