// Host harness: what a block of k_prop_emit that starts while the control block
// advances goes by, for every mixture of the words before and after.
#include <cstring>

#include "ckf/step_ctl.hpp"

// Returns the number of mixtures in which the block would take its step for a
// different one: another number of partitions than the launch's other blocks
// have, with the queue spent at theirs.
extern "C" uint32_t torn_extents(uint32_t n_links, uint32_t link_base, uint32_t link_cap, uint32_t n_live,
                                 uint32_t tips, uint32_t max_cands, uint32_t raised, uint32_t* n_mixtures) {
    using namespace tamd;
    static step_ctl before, after, torn;
    std::memset(&before, 0, sizeof(before));
    before.step = 3u;
    before.epoch = 77u;
    before.n_in = n_links;
    before.link_base = link_base;
    before.n_links = before.emit_links = n_links;
    before.n_tips = 1000u;
    before.n_tips_step = tips;
    before.n_live = n_live;
    before.overflow = raised;  // by blocks of the same kernel
    const uint32_t parts = emit_extent_of(before).parts;
    before.ticket[5].v = parts;
    after = before;
    advance_ctl(&after, max_cands, raised);

    // the words of the first lines that the advance changes
    constexpr uint32_t kWords = 32u;
    uint32_t a[kWords], b[kWords], changed[kWords], n = 0u;
    std::memcpy(a, &before, sizeof(a));
    std::memcpy(b, &after, sizeof(b));
    for (uint32_t w = 0; w < kWords; ++w) {
        if (a[w] != b[w]) changed[n++] = w;
    }
    uint32_t wrong = 0u;
    *n_mixtures = 1u << n;
    for (uint32_t m = 0; m < *n_mixtures; ++m) {
        uint32_t w[kWords];
        std::memcpy(w, a, sizeof(w));
        for (uint32_t k = 0; k < n; ++k) {
            if ((m >> k) & 1u) w[changed[k]] = b[changed[k]];
        }
        std::memcpy(static_cast<void*>(&torn), &after, sizeof(torn));
        std::memcpy(static_cast<void*>(&torn), w, sizeof(w));
        if (torn.done != 0u) continue;
        const emit_extent e = emit_extent_of(torn);
        // a ticket below e.parts, or (without partitions) a second advance
        if (torn.ticket[5].v < e.parts || e.parts != parts) ++wrong;
    }
    return wrong;
}

extern "C" uint32_t emit_parts(uint32_t n) {
    tamd::step_ctl ctl{};
    ctl.emit_links = n;
    return tamd::emit_extent_of(ctl).parts;
}
