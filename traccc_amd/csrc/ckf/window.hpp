// The measurements of a surface that can pass the chi2 cut, by a team of lanes.
#pragma once

#include "device_types.hpp"

namespace tamd {

// Measurements a lane reads per round, all loads issued before the arithmetic.
constexpr int kBatch = 4;

// A superset [lo, up) of the surface's measurements whose loc0 can lie in
// [a, b], for measurements sorted by loc0: cooperative 16-ary narrowing by the
// team (kT lanes x kBatch probes per round) of the first index >= a and of the
// first index > b, both in every round: a round costs one memory latency, which
// bounds the search, whichever of the two still has to go on.
template <int kT>
__device__ inline void window_range(const ckf_params& P, float a, float b, uint32_t tl,
                                    uint32_t& lo, uint32_t& up) {
    constexpr uint32_t kProbes = kT * kBatch;
    uint32_t La = lo, Ha = up, Lb = lo, Hb = up;  // the wanted indices lie in [L, H]
    while (Ha - La > kProbes || Hb - Lb > kProbes) {
        const uint32_t sa = Ha - La, sb = Hb - Lb;
        float va[kBatch], vb[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const uint32_t k = static_cast<uint32_t>(u * kT) + tl;
            va[u] = sa > kProbes ? P.meas_pos[La + ((k + 1u) * sa) / (kProbes + 1u)].x : 0.f;
            vb[u] = sb > kProbes ? P.meas_pos[Lb + ((k + 1u) * sb) / (kProbes + 1u)].x : 0.f;
        }
        uint32_t below = 0u;  // of a in the low half, of b in the high half
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            below += (va[u] < a ? 1u : 0u) + (!(vb[u] > b) ? 0x10000u : 0u);
        }
#pragma unroll
        for (int d = kT / 2; d >= 1; d >>= 1) below += __shfl_xor(below, d, kT);
        // probes are sorted: so many of them precede the wanted index
        const uint32_t na = below & 0xffffu, nb = below >> 16;
        if (sa > kProbes) {
            const uint32_t L = La;
            La = na == 0u ? L : L + (na * sa) / (kProbes + 1u) + 1u;
            Ha = na == kProbes ? Ha : L + ((na + 1u) * sa) / (kProbes + 1u);
        }
        if (sb > kProbes) {
            const uint32_t L = Lb;
            Lb = nb == 0u ? L : L + (nb * sb) / (kProbes + 1u) + 1u;
            Hb = nb == kProbes ? Hb : L + ((nb + 1u) * sb) / (kProbes + 1u);
        }
    }
    lo = La;
    up = Hb;
}

// Narrow [lo, up) to what can pass the cut: chi2 >= r0^2 / R00 for any 2 x 2
// SPD R, so a measurement that passes has r0^2 <= chi2_max (P00 + V00).
// win_var: the event's largest loc0 variance, below 0 where its surfaces are
// not sorted by loc0 (nothing is narrowed then).
template <int kT>
__device__ inline void narrow_to_window(const ckf_params& P, float win_var, float x0, float p00, uint32_t tl,
                                        uint32_t& lo, uint32_t& up) {
    if (win_var >= 0.f && up - lo > static_cast<uint32_t>(kT * kBatch)) {
        const float w = sqrtf(P.chi2_max * (p00 + win_var)) * 1.01f + 1e-3f;
        if (w == w) {
            window_range<kT>(P, x0 - w, x0 + w, tl, lo, up);
        }
    }
}

}  // namespace tamd
