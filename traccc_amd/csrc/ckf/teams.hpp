// How many lanes take one chain of work together, by how many chains there are.
// Plain code for the host: the rules that choose a call's launches.
#pragma once

#include <algorithm>
#include <cstdint>

namespace tamd {

// One launch of k_propagate: `team` lanes per link (1, 2, 4, 8 or 16; 0: no
// launch) for steps of [from, below) links.
struct prop_launch {
    uint32_t team, from, below, blocks;
};

// k_propagate's registers allow two waves per SIMD, four SIMDs per CU
constexpr uint32_t kPropWavesPerCu = 8u;

// Inputs that a step of a call is first given room for.
inline uint64_t input_bound(uint32_t n_seeds, uint32_t per_surface, uint32_t per_seed) {
    const uint64_t branchy = std::min<uint64_t>(per_seed, uint64_t(per_surface) * per_surface);
    return uint64_t(n_seeds) * std::max<uint64_t>(branchy, 1u);
}

// Links that a step of this call can have: with one branch per surface as many as
// seeds, otherwise what its first buffers hold; all that the buffers hold
// (state_cap) once the call has outgrown those.  The buffers alone say nothing
// about the call: they are as large as the largest one before it.
inline uint64_t step_bound(uint32_t n_seeds, uint32_t per_surface, uint32_t per_seed, uint32_t state_cap,
                           bool regrown) {
    if (per_surface == 1u) return n_seeds;
    if (regrown) return state_cap;
    return std::min<uint64_t>(state_cap, input_bound(n_seeds, per_surface, per_seed) * per_surface);
}

// The launches of k_propagate in a step, by how many links a step of this call
// can have (`bound`).  lanes = what the chip holds (two waves per SIMD, what the
// kernel's registers allow): a team is worth its redundant steps while its waves
// all run at once.  us per step (1 without deferral / 2 / 4 / 8 / 16 lanes):
// 285,989 links 268 / 416 / 518 / 693 / 1011; 84,815 124 / 156 / 188 / 288 /
// 416; 54,417 117 / 106 / 131 / 187 / 264; 29,559 107 / 93 / 75 / 107 / 176;
// 11,089 89 / 86 / 60 / 54 / 68; 3,435 93 / 79 / 55 / 44 / 40; 335 66 / 73 /
// 48 / 36 / 30.  A call whose steps all fit one team's range runs one launch
// (a second one costs ~3 us a step to find that it has nothing to do).
// `fixed`: that team for every step (diagnostics), 0 by the rule.
inline void propagate_launches(uint32_t n_cu, uint64_t bound, uint32_t fixed, prop_launch (&out)[2]) {
    const uint64_t lanes = uint64_t(n_cu) * kPropWavesPerCu * 64u;
    const uint32_t max_blocks = n_cu * kPropWavesPerCu / 4u;
    auto entry = [&](int k, uint32_t team, uint32_t from, uint32_t below) {
        const uint64_t most = std::min<uint64_t>(bound, below);
        const uint64_t blocks = (most * team + 255u) / 256u;
        out[k] = prop_launch{team, from, below, static_cast<uint32_t>(std::max<uint64_t>(
                                                    1u, std::min<uint64_t>(blocks, max_blocks)))};
    };
    constexpr uint32_t kAll = 0xffffffffu;
    out[0] = out[1] = prop_launch{};
    if (fixed != 0u) {
        entry(0, fixed, 0u, kAll);
    } else if (bound * 16u <= lanes * 5u / 8u) {
        entry(0, 16u, 0u, kAll);
    } else if (bound * 8u <= lanes) {
        entry(0, 8u, 0u, kAll);
    } else if (bound * 4u <= lanes) {
        const uint32_t t = static_cast<uint32_t>(lanes / 16u);  // 8,192 on 256 CUs
        entry(0, 4u, t, kAll);
        entry(1, 16u, 0u, t);
    } else {
        const uint32_t t = static_cast<uint32_t>(lanes * 27u / 128u);  // 27,648 on 256 CUs
        entry(0, bound * 2u <= lanes * 7u / 8u ? 2u : 1u, t, kAll);
        entry(1, 8u, 0u, t);
    }
}

// Lanes that take one chain together in a kernel without steps (the fit's forward
// pass: a candidate's propagations and updates one after another; the progressive
// filter: a seed's walk through the detector): few chains are bound by the chain,
// which a team's navigation shortens (a propagation takes ~100 us on one lane
// alone, 55 on 8, 40 on 16), many by the lanes, which a team spends on redundant
// steps.  So the lines lie at chains per CU.  Whole calls, us, with 1 / 8 / 16
// lanes on 256 CUs:
//                fit of candidates         progressive filter of seeds
//    5,000   1,084 /   795 /   724       787 /   394 /   388
//   10,000   1,263 /   998 / 1,026       875 /   490 /   529
//   28,000   2,115 / 1,935 / 2,078     1,003 /   858 / 1,014
//   36,000   2,477 / 2,450 / 2,601     1,016 /   903 / 1,125
//   56,000   3,431 / 3,488 / 3,805     1,121 / 1,292 / 1,568
inline uint32_t chain_team(uint64_t n, uint32_t n_cu) {
    if (n <= uint64_t(n_cu) * 20u) return 16u;  // 5,120 on 256 CUs
    return n <= uint64_t(n_cu) * 112u ? 8u : 1u;  // 28,672
}

}  // namespace tamd
