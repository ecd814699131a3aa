// Host harness: the rules that choose a call's launches.
#include "ckf/teams.hpp"

extern "C" void propagate_launches(uint32_t n_cu, uint64_t bound, uint32_t fixed, uint32_t out[8]) {
    tamd::prop_launch l[2];
    tamd::propagate_launches(n_cu, bound, fixed, l);
    for (int k = 0; k < 2; ++k) {
        out[4 * k] = l[k].team;
        out[4 * k + 1] = l[k].from;
        out[4 * k + 2] = l[k].below;
        out[4 * k + 3] = l[k].blocks;
    }
}

extern "C" uint64_t step_bound(uint32_t n_seeds, uint32_t per_surface, uint32_t per_seed, uint32_t state_cap,
                               int regrown) {
    return tamd::step_bound(n_seeds, per_surface, per_seed, state_cap, regrown != 0);
}

extern "C" uint32_t chain_team(uint64_t n, uint32_t n_cu) { return tamd::chain_team(n, n_cu); }
