// CKF step kernels for CDNA (gfx950).
//
// Per step (counts live in the device step control block):
//   k_find        two lanes per input branch: chi2 over the surface's
//                 measurements, best-N selection by (chi2, measurement index),
//                 gain-matrix update, hole links; links are compacted in input
//                 order with a wave scan + decoupled look-back
//                 (traccc host: details/combinatorial_kalman_filter.hpp:174-364)
//   k_dedup_mark  duplicate removal grouped by latest measurements (the groups'
//                 lists are made where the links are, in k_find_emit)
//                 (traccc host :371-488)
//   k_propagate   one lane or a team per link: per-seed cap, hole limits, RK4 transport
//                 to the next sensitive surface, tips; next-step inputs and
//                 tips compacted with ballots + look-back (traccc host :493-627)
//   k_advance     one lane: advances the control block
// build_tracks after the loop (traccc host :637-715).
//
// Work distribution: every kernel is a persistent grid whose waves take
// 64-item partitions from an atomic ticket (device work queue), so uneven
// per-branch cost (measurements per surface, RK steps per crossing) balances
// across the chip.
#include <hip/hip_runtime.h>

#include <cfloat>

#include "device_types.hpp"
#include "kalman_device.hpp"
#include "features.hpp"
#include "kernels.hpp"
#include "../scorer/mlp_device.hpp"
#include "state_io.hpp"
#include "wave.hpp"
#include "window.hpp"

namespace tamd {

namespace {

constexpr int kBlock = 256;

__device__ inline void set_overflow(step_ctl* ctl, uint32_t bit) { atomicOr(&ctl->overflow, bit); }

__device__ inline dlink load_link(const ckf_params& P, uint32_t g) { return P.links[g]; }

}  // namespace

// ---------------------------------------------------------------------------
// find_tracks
// ---------------------------------------------------------------------------
// A team of kT lanes handles one input branch: the lanes split the
// surface's measurements, reduce the best (chi2, index) candidate with
// shuffles, and run the gain update redundantly (so the team stays uniform);
// the team leader writes.  A wave holds kWave / kT inputs.  Each lane reads
// kBatch measurements per round with all loads issued before the chi2
// arithmetic, so a round costs one memory latency.  The plain find runs
// two-lane teams (its gain updates are redundant over the team, and the loc0
// window leaves few measurements to split); the scorer list, which updates
// nothing, runs four-lane teams.
static_assert(sizeof(line_u32) == kXcdCounterStride * 4u &&
                  sizeof(step_ctl::xcd_ticket[0]) == kXcds * sizeof(line_u32),
              "per-XCD counters: one per XCD, 128 B apart");
constexpr int kFindTeam = 2;
constexpr int kListTeam = 4;
// scorer lists: up to kListTeam * kListSlots candidates per input
constexpr int kListSlots = 4;

// One pass of a team over the surface's measurements [lo, up): the best
// (chi2, index) candidate after (last_c, last_m) (every candidate when
// !have_last) that passes the cut and the step-0 rule.  kInvalid when none.
// With count_pass, n_pass receives the number of measurements passing the cut
// (on every lane of the team).
template <int kT>
__device__ inline void scan_next(const ckf_params& P, const float* x, const float* c, uint32_t lo,
                                 uint32_t up, bool rule0, bool have_last, float last_c,
                                 uint32_t last_m, uint32_t tl, bool count_pass, float& best_c,
                                 uint32_t& best_m, uint32_t& n_pass) {
    best_c = 0.f;
    best_m = kInvalid;
    uint32_t np = 0u;
    for (uint32_t m0 = lo + tl; m0 < up; m0 += kT * kBatch) {
        meas_data mb[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const uint32_t m = m0 + static_cast<uint32_t>(u * kT);
            mb[u] = load_meas(P.meas_pos, P.meas_var, P.meas_info, m < up ? m : lo);
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const uint32_t m = m0 + static_cast<uint32_t>(u * kT);
            const float chi2 = predicted_chi2(mb[u], x, c);
            // outside the cut (a NaN never yields a link either)
            bool take = m < up && chi2 <= P.chi2_max && chi2 >= 0.f;
            take = take && !(rule0 && chi2 != 0.f);
            np += take ? 1u : 0u;
            take = take && !(have_last && (chi2 < last_c || (chi2 == last_c && m <= last_m)));
            if (take && (best_m == kInvalid || chi2 < best_c || (chi2 == best_c && m < best_m))) {
                best_c = chi2;
                best_m = m;
            }
        }
    }
    // team minimum of (chi2, index); kInvalid sorts last
#pragma unroll
    for (int d = kT / 2; d >= 1; d >>= 1) {
        const float oc = __shfl_xor(best_c, d, kT);
        const uint32_t om = __shfl_xor(best_m, d, kT);
        const bool take = (om != kInvalid) &&
                          (best_m == kInvalid || oc < best_c || (oc == best_c && om < best_m));
        if (take) {
            best_c = oc;
            best_m = om;
        }
    }
    if (count_pass) {
#pragma unroll
        for (int d = kT / 2; d >= 1; d >>= 1) np += __shfl_xor(np, d, kT);
        n_pass = np;
    }
}

// The input branch a team works on at this step: its predicted state, its
// previous link's bookkeeping and the surface's measurement range.
struct find_input {
    float x[6], c[21];
    uint32_t sf, seed, prev_g, skip, consec, ndf_prev, in_slot, lo, up;
    float chi2_prev;
    float win_var;  // the event's largest loc0 variance, < 0: no window search
    bool rule0;
};

// Candidates of one input in (chi2, index) order from a single pass over the
// surface's measurements (its loc0 window when the event allows one): every
// lane keeps the kLaneKeep best passing candidates of its share in registers
// (sorted), and next() merges the team's lists with one team minimum per
// candidate.  When some lane of the team saw more passing candidates than it
// keeps, the stream falls back to one scan_next pass over the same range per
// candidate (the order is the same either way).
template <int kLaneKeep, int kT>
struct cand_stream {
    static constexpr int kKeep = kLaneKeep;
    static constexpr int kTeamSize = kT;
    float lc[kLaneKeep];
    uint32_t lm[kLaneKeep];
    uint32_t lo, up;    // the measurements searched (the loc0 window when taken)
    uint32_t head;      // next own list entry
    uint32_t n_pass;    // team: measurements passing the cut
    bool fallback;      // team-uniform
    bool have_last;
    float last_c;
    uint32_t last_m;
};

template <typename Stream>
__device__ __forceinline__ void stream_init(const ckf_params& P, const find_input& in, uint32_t tl,
                                   Stream& S) {
    constexpr int kLaneKeep = Stream::kKeep;
    constexpr int kT = Stream::kTeamSize;
    const float inf = __int_as_float(0x7f800000);
#pragma unroll
    for (int j = 0; j < kLaneKeep; ++j) {
        S.lc[j] = inf;
        S.lm[j] = kInvalid;
    }
    uint32_t np = 0u;
    // on a dense surface sorted by loc0 only the window of measurements that
    // can pass is read
    uint32_t lo = in.lo, up = in.up;
    narrow_to_window<kT>(P, in.win_var, in.x[e_loc0], in.c[sym_idx(0, 0)], tl, lo, up);
    for (uint32_t m0 = lo + tl; m0 < up; m0 += kT * kBatch) {
        meas_data mb[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const uint32_t m = m0 + static_cast<uint32_t>(u * kT);
            mb[u] = load_meas(P.meas_pos, P.meas_var, P.meas_info, m < up ? m : lo);
        }
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
            const uint32_t m = m0 + static_cast<uint32_t>(u * kT);
            const float chi2 = predicted_chi2(mb[u], in.x, in.c);
            bool take = m < up && chi2 <= P.chi2_max && chi2 >= 0.f;
            take = take && !(in.rule0 && chi2 != 0.f);
            if (take) {
                ++np;
                // insertion into the list sorted by (chi2, index)
                float cc = chi2;
                uint32_t cm = m;
#pragma unroll
                for (int j = 0; j < kLaneKeep; ++j) {
                    if (cc < S.lc[j] || (cc == S.lc[j] && cm < S.lm[j])) {
                        const float tc = S.lc[j];
                        const uint32_t tm = S.lm[j];
                        S.lc[j] = cc;
                        S.lm[j] = cm;
                        cc = tc;
                        cm = tm;
                    }
                }
            }
        }
    }
    uint32_t over = np > static_cast<uint32_t>(kLaneKeep) ? 1u : 0u;
#pragma unroll
    for (int d = kT / 2; d >= 1; d >>= 1) {
        np += __shfl_xor(np, d, kT);
        over |= __shfl_xor(over, d, kT);
    }
    S.n_pass = np;
    S.lo = lo;
    S.up = up;
    S.fallback = over != 0u;
    S.head = 0u;
    S.have_last = false;
    S.last_c = 0.f;
    S.last_m = 0u;
}

template <typename Stream>
__device__ __forceinline__ void stream_next(const ckf_params& P, const find_input& in, uint32_t tl,
                                   Stream& S, float& best_c, uint32_t& best_m) {
    constexpr int kLaneKeep = Stream::kKeep;
    constexpr int kT = Stream::kTeamSize;
    if (S.fallback) {
        uint32_t unused = 0u;
        scan_next<kT>(P, in.x, in.c, S.lo, S.up, in.rule0, S.have_last, S.last_c, S.last_m, tl,
                  false, best_c, best_m, unused);
    } else {
        // own head: a select chain keeps the list in registers
        float c = S.lc[kLaneKeep - 1];
        uint32_t m = S.lm[kLaneKeep - 1];
#pragma unroll
        for (int j = kLaneKeep - 2; j >= 0; --j) {
            if (S.head == static_cast<uint32_t>(j)) {
                c = S.lc[j];
                m = S.lm[j];
            }
        }
        if (S.head >= static_cast<uint32_t>(kLaneKeep)) {
            m = kInvalid;
        }
        best_c = c;
        best_m = m;
        // team minimum of (chi2, index); kInvalid sorts last
#pragma unroll
        for (int d = kT / 2; d >= 1; d >>= 1) {
            const float oc = __shfl_xor(best_c, d, kT);
            const uint32_t om = __shfl_xor(best_m, d, kT);
            const bool take = (om != kInvalid) &&
                              (best_m == kInvalid || oc < best_c || (oc == best_c && om < best_m));
            if (take) {
                best_c = oc;
                best_m = om;
            }
        }
        if (best_m != kInvalid && best_m == m) {
            ++S.head;  // the owner moves to its next entry
        }
    }
    if (best_m != kInvalid) {
        S.have_last = true;
        S.last_c = best_c;
        S.last_m = best_m;
    }
}

// kRanges = false (the scored update, which scans nothing) skips the
// event's measurement range and window lookups.
template <bool kRanges = true>
__device__ inline void load_input(const ckf_params& P, uint32_t step, uint32_t i,
                                  uint32_t prev_base, find_input& in) {
    const uint32_t in_par = (step + 1u) & 1u;
    in.prev_g = kInvalid;
    in.skip = in.consec = in.ndf_prev = in.in_slot = 0u;
    in.chi2_prev = 0.f;
    if (step == 0u) {
        in.seed = i;
        load_seed(P, i, in.x, in.c, in.sf);
    } else {
        in.in_slot = P.live[i];
        in.prev_g = prev_base + in.in_slot;
        const dlink L = load_link(P, in.prev_g);
        in.seed = L.seed;
        in.skip = link_skipped(L);
        in.consec = link_consec(L);
        in.chi2_prev = L.chi2_sum;
        in.ndf_prev = L.ndf_sum;
        load_soa(P.state[in_par], P.state_cap, in.in_slot, in.x, in.c, in.sf);
    }
    in.lo = in.up = 0u;
    in.win_var = -1.f;
    if constexpr (kRanges) {
        const uint32_t ev = P.seed_event[in.seed];
        const uint32_t* rg = P.meas_ranges + static_cast<size_t>(ev) * (P.n_surfaces + 1u);
        in.lo = rg[in.sf];
        in.up = rg[in.sf + 1u];
        in.win_var = P.event_win_var[ev];
    }
    in.rule0 = (step == 0u) && !(P.sfs[in.sf].thickness_x0 > 0.f);
}

// Link bookkeeping handed from k_find to k_find_emit (see stage_head).
__device__ inline stage_head make_stage_head(const find_input& in, uint32_t step, uint32_t i) {
    stage_head h;
    h.prev = in.prev_g;
    h.seed = in.seed;
    h.hist = in.skip | (in.consec << 8);
    h.hole_ref = (step == 0u) ? ((kRefSeed << kRefKindShift) | i)
                              : ((kRefInput << kRefKindShift) | in.in_slot);
    h.chi2_sum = in.chi2_prev;
    h.ndf_sum = in.ndf_prev;
    h.pad[0] = h.pad[1] = 0u;
    return h;
}

// Measurement indices stay below 2^31 (the batch's measurement count is a
// 32-bit size and far smaller), so the top bit carries the dimension.
__device__ inline stage_cand make_stage_cand(uint32_t m, float chi2, uint32_t dims) {
    stage_cand c;
    c.meas = m | (dims == 2u ? 0x80000000u : 0u);
    c.chi2 = chi2;
    return c;
}

// Filtered-state slot of an input's k-th kept candidate: plane k of in_cap
// slots, so the common case of one kept candidate per input fills
// consecutive slots (coalesced SoA stores here and loads in k_propagate).
// Past flt_cap it returns kInvalid, which every caller treats as overflow.
__device__ inline uint32_t flt_slot(const ckf_params& P, uint32_t i, uint32_t k) {
    const uint64_t s = static_cast<uint64_t>(k) * P.in_cap + i;
    return s < P.flt_cap ? static_cast<uint32_t>(s) : kInvalid;
}

// Slot of listed candidate q of input i: plane-major like the filtered
// states, so a wave's lanes (consecutive inputs) read and write one plane's
// consecutive entries.
__device__ inline size_t list_slot(const ckf_params& P, uint32_t i, uint32_t q) {
    return static_cast<size_t>(q) * P.in_cap + i;
}

// The link a staged slot becomes (a hole link carries the input's own state).
__device__ inline dlink staged_link(const stage_head& h, const stage_cand& c, uint32_t step,
                                    uint32_t slot) {
    const bool hole = c.meas == kInvalid;
    const uint32_t skip = h.hist & 0xffu, consec = h.hist >> 8;
    dlink L;
    L.prev = h.prev;
    L.seed = h.seed;
    if (hole) {
        L.meas = kInvalid;
        L.packed = pack_link(step, skip + 1u, consec + 1u);
        L.chi2 = FLT_MAX;
        L.chi2_sum = h.chi2_sum;
        L.ndf_sum = h.ndf_sum;
        L.state_ref = h.hole_ref;
    } else {
        L.meas = c.meas & 0x7fffffffu;
        L.packed = pack_link(step, skip, 0u);
        L.chi2 = c.chi2;
        L.chi2_sum = h.chi2_sum + c.chi2;
        L.ndf_sum = h.ndf_sum + ((c.meas >> 31) != 0u ? 2u : 1u);
        L.state_ref = (kRefFiltered << kRefKindShift) | slot;
    }
    return L;
}

// Compaction partitions of the emit kernels: a block takes up to kEmitChunks
// consecutive chunks of kBlock items per ticket, counts them, runs one
// decoupled look-back for the whole partition (its first wave), then writes.
// A partition's items are in flight together, one per thread and chunk: with
// one wave walking a partition of 1,024 items chunk by chunk, a step of 90,000
// inputs kept 88 waves of the chip busy and its compaction took 50 us, four
// times what the bytes and one look-back cost.
constexpr uint32_t kEmitWaves = kBlock / kWave;
static_assert(kBlock == kEmitBlock, "a chunk is an item per thread of a block");

struct emit_shared {
    uint32_t ticket;
    uint32_t tot[2][kEmitChunks * kEmitWaves];  // per channel: each wave's items of a chunk
    uint64_t base;
};

// The block's next partition (every thread).  The two barriers also keep the
// shared words of the last partition from being overwritten too early.
__device__ inline uint32_t block_ticket(uint32_t* counter, emit_shared& S) {
    __syncthreads();
    if (threadIdx.x == 0u) {
        S.ticket = atomicAdd(counter, 1u);
    }
    __syncthreads();
    return S.ticket;
}

// Exclusive prefixes of v[chunk] over the partition's items in order (chunk
// by chunk, thread by thread), in place; returns the partition's total.  Ends
// with a barrier behind it.
__device__ inline uint32_t block_prefix(uint32_t (&v)[kEmitChunks], int channel, emit_shared& S) {
    const uint32_t w = threadIdx.x / kWave;
#pragma unroll
    for (uint32_t ch = 0; ch < kEmitChunks; ++ch) {
        const uint32_t incl = wave_inclusive_scan(v[ch]);
        if (lane() == kWave - 1) {
            S.tot[channel][ch * kEmitWaves + w] = incl;
        }
        v[ch] = incl - v[ch];
    }
    __syncthreads();
    uint32_t run = 0u;
#pragma unroll
    for (uint32_t ch = 0; ch < kEmitChunks; ++ch) {
#pragma unroll
        for (uint32_t q = 0; q < kEmitWaves; ++q) {
            if (q == w) {
                v[ch] += run;
            }
            run += S.tot[channel][ch * kEmitWaves + q];
        }
    }
    return run;
}

// The partition's look-back by the block's first wave; every thread gets the
// exclusive prefix of both channels.
__device__ inline uint64_t block_lookback(uint64_t* lo_words, uint64_t* hi_words, uint32_t p, uint32_t epoch,
                                          uint64_t agg, emit_shared& S) {
    if (threadIdx.x < kWave) {
        const uint64_t b = wave_lookback(lo_words, hi_words, p, epoch, agg);
        if (threadIdx.x == 0u) {
            S.base = b;
        }
    }
    __syncthreads();
    return S.base;
}

// A listed candidate's MLP row (16 shorts, 32 B): features 0-8, 10 and 11
// normalised and rounded to BF16 exactly as the scorer takes them, short 9
// zero, and feature 9 (standing) as its raw FP32 running value in shorts
// 12-13 -- it needs every seed's minimum of the step, so k_score_update
// finalises it.  Shorts 14-15 are zero.
constexpr int kRowShorts = 16;

__device__ inline void store_list_row(const mlp_dev& W, short* row, const float (&f)[kFeatures]) {
    uint32_t w[8];
#pragma unroll
    for (int e = 0; e < 6; ++e) {
        const int a = 2 * e, b = 2 * e + 1;
        const uint16_t lo = a == kFeatStanding ? 0u
                                               : static_cast<uint16_t>(f2bf((f[a] - W.mean[a]) * W.inv_std[a]));
        const uint16_t hi = b == kFeatStanding ? 0u
                                               : static_cast<uint16_t>(f2bf((f[b] - W.mean[b]) * W.inv_std[b]));
        w[e] = static_cast<uint32_t>(lo) | (static_cast<uint32_t>(hi) << 16);
    }
    w[6] = __float_as_uint(f[kFeatStanding]);
    w[7] = 0u;
    uint4* dst = reinterpret_cast<uint4*>(row);
    dst[0] = make_uint4(w[0], w[1], w[2], w[3]);
    dst[1] = make_uint4(w[4], w[5], w[6], w[7]);
}

// Scorer-pruned finding, first kernel: per input the list_len best candidates
// in (chi2, index) order and their MLP rows, at the input's fixed slots
// list_slot(input, q); k_score_update scores and updates them.
__global__ __launch_bounds__(kBlock) void k_find_list(ckf_params P) {
    step_ctl* ctl = P.ctl;
    if (ctl->done) {
        return;
    }
    const uint32_t step = ctl->step;
    const uint32_t n_in = ctl->n_in < P.in_cap ? ctl->n_in : P.in_cap;
    const uint32_t prev_base = ctl->prev_link_base;
    const uint32_t team = lane() / kListTeam;
    const uint32_t tl = lane() % kListTeam;
    const uint32_t Lc = P.list_len;
    const uint32_t epoch = ctl->epoch;
    const uint32_t n_parts = (n_in + (kWave / kListTeam) - 1) / (kWave / kListTeam);
    // dynamic partitions (dense surfaces make some inputs far heavier)
    xcd_ticket_run queue(&ctl->xcd_ticket[1][0].v, n_parts);
    for (;;) {
        const uint32_t p = queue.next();
        if (p >= n_parts) {
            break;
        }
        const uint32_t i0 = p * (kWave / kListTeam);
        const uint32_t i = i0 + team;
        const bool active = i < n_in;
        find_input in;
        uint32_t n_pass = 0u, k = 0u;
        // candidate q of the list is held by team lane q % kListTeam in slot q / kListTeam
        uint32_t sm[kListSlots];
        float sc[kListSlots];
        if (active) {
            load_input(P, step, i, prev_base, in);
            cand_stream<6, kListTeam> cs;
            stream_init(P, in, tl, cs);
            n_pass = cs.n_pass;
            for (; k < Lc; ++k) {
                float best_c;
                uint32_t best_m;
                stream_next(P, in, tl, cs, best_c, best_m);
                if (best_m == kInvalid) {
                    break;
                }
#pragma unroll
                for (int j = 0; j < kListSlots; ++j) {
                    if (k == static_cast<uint32_t>(j * kListTeam) + tl) {
                        sm[j] = best_m;
                        sc[j] = best_c;
                    }
                }
            }
        }
        if (active) {
            if (tl == 0u) {
                P.list_n[i] = k;
                P.list_seed[i] = in.seed;
            }
            // the team's lanes write the list and the features of their
            // candidates, at the input's fixed slots list_slot(i, q)
#pragma unroll
            for (int j = 0; j < kListSlots; ++j) {
                const uint32_t q = static_cast<uint32_t>(j * kListTeam) + tl;
                if (q < k) {
                    const size_t r = list_slot(P, i, q);
                    P.list_m[r] = sm[j];
                    P.list_c[r] = sc[j];
                    const meas_data md = load_meas(P.meas_pos, P.meas_var, P.meas_info, sm[j]);
                    float f[kFeatures];
                    candidate_features(P, md, in.x, in.c, in.sf, step, in.skip, in.consec,
                                       in.chi2_prev, in.ndf_prev, sc[j], q, n_pass, f);
                    store_list_row(P.scorer, P.list_row + r * kRowShorts, f);
                    if (q == 0u) {
                        standing_offer(P.seed_run_min, in.seed, epoch, f[kFeatStanding]);
                    }
                }
            }
        }
    }
}

// Diagnostics: one scored candidate's verdict as a key a CPU checker replays.
// The key names the candidate by its branch's history, so it does not depend
// on where the branch sits in the step's input order: splitmix64 chained over
// the seed, the step, the measurement of every earlier link of the branch
// (latest first, holes as all-ones) and the candidate's measurement; low 63
// bits, bit 63 = kept.
__device__ inline uint64_t verdict_mix(uint64_t h, uint64_t v) {
    uint64_t z = (h ^ v) + 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

__device__ inline void log_verdict(const ckf_params& P, uint32_t step, uint32_t input,
                                   uint32_t meas, bool keep) {
    const uint32_t at = atomicAdd(P.verdict_n, 1u);
    if (at >= P.verdict_cap) {
        return;
    }
    uint64_t h = verdict_mix(0u, P.list_seed[input]);
    h = verdict_mix(h, step);
    if (step > 0u) {
        uint32_t g = P.ctl->prev_link_base + P.live[input];
        for (uint32_t k = 0; k < step && g < P.link_cap; ++k) {
            const dlink L = P.links[g];
            h = verdict_mix(h, L.meas);
            if (link_step(L) == 0u) {
                break;
            }
            g = L.prev;
        }
    }
    h = verdict_mix(h, meas);
    P.verdict_log[at] = (h & 0x7fffffffffffffffull) | (keep ? (1ull << 63) : 0ull);
}

// Scorer-pruned finding, second kernel, one input per lane (a wave holds 64
// inputs).  The wave packs its inputs' listed candidates (k_find_list's
// fixed slots) densely into LDS rows -- the features normalised and rounded
// to BF16, feature 9 finalised from its seed's minimum -- kRows at a time,
// scores them 16 rows per matrix-core pass, and keeps one 16-bit verdict mask
// per sub-tile in LDS; then each lane walks its input's kept entries in list
// order, runs the gain update until N succeed and stages the links as the
// plain find does (k_find_emit builds them).
constexpr uint32_t kRows = 128;    // LDS rows of a wave per packing pass
constexpr int kListMax = kListTeam * kListSlots;
constexpr uint32_t kSubTiles = (kWave * kListMax) / 16u;  // sub-tiles of a full partition
static_assert(kListMax <= 32, "kept-entry mask is 32 bits");

// The update of one input after the MLP: its kept entries in list order (a
// mask read from the sub-tiles' verdicts), the gain update until N succeed,
// staging as the plain find.
__device__ __forceinline__ void score_update_input(const ckf_params& P, uint32_t i, uint32_t k,
                                                   uint32_t base, const uint16_t* keep16,
                                                   uint32_t step, uint32_t prev_base) {
    step_ctl* ctl = P.ctl;
    const uint32_t N = P.n_branch_surface;
    uint32_t kept = 0u;
    for (uint32_t q = 0; q < k; ++q) {
        const uint32_t r = base + q;
        if ((keep16[r / 16u] >> (r % 16u)) & 1u) {
            kept |= 1u << q;
        }
    }
    if (P.verdict_log != nullptr) {
        for (uint32_t q = 0; q < k; ++q) {
            log_verdict(P, step, i, P.list_m[list_slot(P, i, q)], ((kept >> q) & 1u) != 0u);
        }
    }
    find_input in;
    load_input<false>(P, step, i, prev_base, in);
    P.stage_in[i] = make_stage_head(in, step, i);
    uint32_t count = 0u;
    while (count < N && kept != 0u) {
        const uint32_t li = static_cast<uint32_t>(__builtin_ctz(kept));
        kept &= kept - 1u;
        const uint32_t best_m = P.list_m[list_slot(P, i, li)];
        const float best_c = P.list_c[list_slot(P, i, li)];
        const meas_data md = load_meas(P.meas_pos, P.meas_var, P.meas_info, best_m);
        float fx[6], fc[21];
#pragma unroll
        for (int e = 0; e < 6; ++e) fx[e] = in.x[e];
#pragma unroll
        for (int e = 0; e < 21; ++e) fc[e] = in.c[e];
        int res = CKF_FIT_SUCCESS;
        if (in.rule0) {
            // step 0 on a surface without material: keep the seed, take the
            // measurement variances
            fc[sym_idx(0, 0)] = md.v0;
            fc[sym_idx(1, 1)] = md.v1;
        } else {
            res = gain_update(md, fx, fc);
        }
        if (res == CKF_FIT_SUCCESS) {
            const uint32_t slot = flt_slot(P, i, count);
            if (slot < P.flt_cap) {
                store_soa(P.flt, P.flt_cap, slot, fx, fc, in.sf);
                P.stage_slot[slot] = make_stage_cand(best_m, best_c, md.dims);
            } else {
                set_overflow(ctl, 4u);
            }
            ++count;
        }
    }
    if (count == 0u) {
        // no candidate kept: the input continues as one hole link
        const uint32_t slot = flt_slot(P, i, 0u);
        if (slot < P.flt_cap) {
            P.stage_slot[slot] = stage_cand{kInvalid, 0.f};
        } else {
            set_overflow(ctl, 4u);
        }
    }
    P.find_count[i] = count;
}

// Three waves per SIMD: the compiler's own allocation lands four registers
// above the three-wave budget, and the hint costs no spill.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3, 8)))
void k_score_update(ckf_params P) {
    __shared__ __attribute__((aligned(16))) short s_rows[kBlock / kWave][kRows * kRowShorts];
    __shared__ uint16_t s_keep[kBlock / kWave][kSubTiles];
    __shared__ mlp_vecs V;
    __shared__ mlp_frags_lds F;
    step_ctl* ctl = P.ctl;
    if (ctl->done) {
        return;  // the whole grid returns: no barrier is left waiting
    }
    mlp_fill_vecs(P.scorer, V, threadIdx.x, blockDim.x);
    mlp_fill_frags(P.scorer, F, threadIdx.x, blockDim.x);
    __syncthreads();
    const uint32_t step = ctl->step;
    const uint32_t n_in = ctl->n_in < P.in_cap ? ctl->n_in : P.in_cap;
    const uint32_t prev_base = ctl->prev_link_base;
    const uint32_t epoch = ctl->epoch;
    const uint32_t l = lane();
    const uint32_t wave = threadIdx.x / kWave;
    short* rows = s_rows[wave];
    uint16_t* keep16 = s_keep[wave];
    const uint32_t n_parts = (n_in + kWave - 1u) / kWave;
    xcd_ticket_run queue(&ctl->xcd_ticket[0][0].v, n_parts);
    for (;;) {
        const uint32_t p = queue.next();
        if (p >= n_parts) {
            break;
        }
        const uint32_t i = p * kWave + l;
        const bool valid = i < n_in;
        const uint32_t k = valid ? P.list_n[i] : 0u;
        const uint32_t seed = valid ? P.list_seed[i] : 0u;
        const uint32_t incl = wave_inclusive_scan(k);
        const uint32_t total = wave_broadcast(incl, kWave - 1);
        const uint32_t base = incl - k;
        // rows [r0, r0 + kRows) per pass: pack, then score 16 at a time
        for (uint32_t r0 = 0u; r0 < total; r0 += kRows) {
            for (uint32_t q = 0; q < k; ++q) {
                const uint32_t r = base + q;
                if (r < r0 || r >= r0 + kRows) {
                    continue;
                }
                const uint4* src =
                    reinterpret_cast<const uint4*>(P.list_row + list_slot(P, i, q) * kRowShorts);
                const uint4 a = src[0];
                uint4 b = src[1];
                // feature 9 (short 9, the high half of b.x) from the raw
                // running value and the seed's minimum; shorts 12-15 zero
                const float st = standing_of(P.seed_run_min, seed, epoch, __uint_as_float(b.z));
                const uint16_t bf9 = static_cast<uint16_t>(mlp_feature_bf(V, st, kFeatStanding));
                b.x = (b.x & 0xffffu) | (static_cast<uint32_t>(bf9) << 16);
                b.z = 0u;
                b.w = 0u;
                uint4* row = reinterpret_cast<uint4*>(rows + (r - r0) * kRowShorts);
                row[0] = a;
                row[1] = b;
            }
            wave_lds_sync();
            const uint32_t n_rows = total - r0 < kRows ? total - r0 : kRows;
            for (uint32_t t = 0; t < (n_rows + 15u) / 16u; ++t) {
                const uint32_t r = t * 16u + (l % 16u);
                bf16x4 xb = {0, 0, 0, 0};
                if (r < n_rows) {
                    xb = load4(rows + r * kRowShorts + 4u * (l / 16u));
                }
                const float s = mlp_logit16_lds(F, V, xb);
                const uint64_t bits = wave_ballot(l < 16u && r < n_rows && s >= P.score_threshold);
                if (l == 0u) {
                    keep16[r0 / 16u + t] = static_cast<uint16_t>(bits & 0xffffull);
                }
            }
            wave_lds_sync();  // the next pass overwrites the rows
        }
        if (l == 0u && total > 0u) {
            atomicAdd(&ctl->n_rows.v, total);
        }
        if (valid) {
            score_update_input(P, i, k, base, keep16, step, prev_base);
        }
    }
}

// A team of kFindTeam lanes handles one input branch.  Plain: the lanes split
// the surface's measurements (the candidate stream) and take candidates in
// (chi2, index) order; logged: the same, with every filtered slot's features
// kept for the branch log.  The gain update runs redundantly on the team (so
// it stays uniform) and the team leader writes.  A wave holds kWave / kT
// inputs.  (The scorer-pruned update is k_score_update.)
enum find_mode : int { kFindPlain = 0, kFindLogged = 1 };

template <int kMode>
__global__ __launch_bounds__(kBlock) void k_find(ckf_params P) {
    constexpr bool logging = (kMode == kFindLogged);
    constexpr int kT = kFindTeam;
    constexpr uint32_t kPerWave = kWave / kT;
    step_ctl* ctl = P.ctl;
    if (ctl->done) {
        return;
    }
    const uint32_t step = ctl->step;
    const uint32_t n_in = ctl->n_in < P.in_cap ? ctl->n_in : P.in_cap;
    const uint32_t prev_base = ctl->prev_link_base;
    const uint32_t n_parts = (n_in + kPerWave - 1) / kPerWave;
    const uint32_t N = P.n_branch_surface;
    const uint32_t team = lane() / kT;
    const uint32_t tl = lane() % kT;
    const bool leader = (tl == 0u);

    xcd_ticket_run queue(&ctl->xcd_ticket[0][0].v, n_parts);
    for (;;) {
        const uint32_t p = queue.next();
        if (p >= n_parts) {
            break;
        }
        const uint32_t i = p * kPerWave + team;
        const bool valid = i < n_in;
        uint32_t count = 0u;
        if (valid) {
            find_input in;
            load_input(P, step, i, prev_base, in);
            if (leader) {
                P.stage_in[i] = make_stage_head(in, step, i);
            }
            uint32_t n_pass = 0u;
            {
                // candidates in stream order; the gain update runs on every
                // lane of the team (uniform), the leader writes
                cand_stream<6, kFindTeam> cs;
                stream_init(P, in, tl, cs);
                n_pass = cs.n_pass;
                bool rank0 = true;
                while (count < N) {
                    float best_c = 0.f;
                    uint32_t best_m = kInvalid;
                    stream_next(P, in, tl, cs, best_c, best_m);
                    if (best_m == kInvalid) {
                        break;
                    }
                    const meas_data md = load_meas(P.meas_pos, P.meas_var, P.meas_info, best_m);
                    if constexpr (logging) {
                        if (rank0 && leader) {
                            standing_offer(P.seed_run_min, in.seed, ctl->epoch,
                                           branch_run(in.chi2_prev, in.ndf_prev, best_c, md.dims));
                        }
                        rank0 = false;
                    }
                    float fx[6], fc[21];
#pragma unroll
                    for (int k = 0; k < 6; ++k) fx[k] = in.x[k];
#pragma unroll
                    for (int k = 0; k < 21; ++k) fc[k] = in.c[k];
                    int res = CKF_FIT_SUCCESS;
                    if (in.rule0) {
                        // step 0 on a surface without material: keep the
                        // seed, take the measurement variances
                        fc[sym_idx(0, 0)] = md.v0;
                        fc[sym_idx(1, 1)] = md.v1;
                    } else {
                        res = gain_update(md, fx, fc);
                    }
                    if (res == CKF_FIT_SUCCESS) {
                        const uint32_t slot = flt_slot(P, i, count);
                        if (leader) {
                            if (slot < P.flt_cap) {
                                store_soa(P.flt, P.flt_cap, slot, fx, fc, in.sf);
                                P.stage_slot[slot] = make_stage_cand(best_m, best_c, md.dims);
                                if constexpr (logging) {
                                    candidate_features(P, md, in.x, in.c, in.sf, step, in.skip, in.consec,
                                                       in.chi2_prev, in.ndf_prev, best_c, count, n_pass,
                                                       P.feat_slot + static_cast<size_t>(slot) * kFeatures);
                                }
                            } else {
                                set_overflow(ctl, 4u);
                            }
                        }
                        ++count;
                    }
                }
            }
            if (count == 0u && leader) {
                // no candidate kept: the input continues as one hole link
                const uint32_t slot = flt_slot(P, i, 0u);
                if (slot < P.flt_cap) {
                    P.stage_slot[slot] = stage_cand{kInvalid, 0.f};
                } else {
                    set_overflow(ctl, 4u);
                }
            }
        }
        if (valid && leader) {
            P.find_count[i] = count;
        }
    }
}

// Duplicate removal drops a link when another one has its measurement
// history.  Both are longer than dup_min_len measurements, so they agree in
// that many of their latest ones: every link carries a summary of its history
// (from its previous link's), links enter a list by the hash of those that must
// agree, and k_dedup_mark walks the histories of two links of a list only where
// their summaries allow it.  (Lists by the last measurement alone, as the rule
// states it, held 50 and more links in dense events, and the branches of a seed
// that parted early agree in all that follows: a chain of dependent loads of
// 50-110 us a step, however few links the step had.)
__device__ inline uint32_t hash16(uint32_t m) { return (m * 0x85ebca77u) >> 16; }
__device__ inline uint32_t hash12(uint32_t m) { return (m * 0x9e3779b1u) >> 20; }

__device__ inline link_history extend_history(const link_history& h, uint32_t meas) {
    link_history r = h;
    if (meas != kInvalid) {
        r.m0 = meas;
        r.m1 = h.m0;
        r.tail = hash16(h.m1) | (h.tail << 16);
        const uint32_t f = (h.all ^ meas) * 0x9e3779b1u;
        r.all = f ^ (f >> 15);
        const uint32_t count = h.ends >> 24;
        r.ends = (h.ends & 0xffffffu) | (count < 255u ? count + 1u : 255u) << 24;
        if (count < 2u) r.ends |= hash12(meas) << (12u * count);
    }
    return r;
}

__device__ inline link_history load_history(const ckf_params& P, uint32_t parity, uint32_t i) {
    const uint4 q = P.history[parity][i];
    return {q.x, q.y, q.z, q.w, history_ends(P, parity)[i]};
}

__device__ inline void store_history(const ckf_params& P, uint32_t parity, uint32_t i, const link_history& h) {
    P.history[parity][i] = make_uint4(h.m0, h.m1, h.tail, h.all);
    history_ends(P, parity)[i] = h.ends;
}

// Hash of the latest measurements that duplicates share: dup_min_len + 1 of them,
// up to four.  Where holes may outnumber what a link counts of them, a link that
// counts as long enough may have fewer: only the latest one is sure.
__device__ inline uint32_t latest_hash(const ckf_params& P, const link_history& r) {
    const uint32_t more = P.max_skip < 255u ? P.dup_min_len : 0u;
    uint32_t h = r.m0 * 0x9e3779b1u;
    h ^= h >> 15;
    if (more >= 1u) h = (h ^ r.m1) * 0x85ebca77u;
    h ^= h >> 13;
    if (more >= 2u) h = (h ^ (r.tail & 0xffffu)) * 0xc2b2ae3du;
    h ^= h >> 16;
    if (more >= 3u) h = (h ^ (r.tail >> 16)) * 0x27d4eb2fu;
    return h ^ (h >> 15);
}

// Enter link i of the step (L, with its history) into its list, with its
// p-value, computed once per link instead of once per pair (the series and the
// continued fraction take ~50 divisions).  A link that is too short neither
// drops another one nor is dropped: kDedupShort stands for it.
constexpr uint32_t kDedupShort = 0xffffffffu;

__device__ inline void dedup_insert(const ckf_params& P, const dlink& L, const link_history& r, uint32_t i,
                                    uint32_t step, uint32_t epoch) {
    if (step + 1u - link_skipped(L) <= P.dup_min_len) {
        dedup_nodes(P, step)[i].head = kDedupShort;
        return;
    }
    dedup_node node;
    node.hash = latest_hash(P, r);
    node.head = static_cast<uint32_t>((static_cast<uint64_t>(node.hash) * (P.n_meas + 1u)) >> 32);
    // list heads carry the step's epoch: a head from an earlier step reads as empty
    const unsigned long long tagged = (static_cast<unsigned long long>(epoch) << 32) | i;
    const unsigned long long old =
        atomicExch(reinterpret_cast<unsigned long long*>(&P.dedup_head[node.head]), tagged);
    node.next = (static_cast<uint32_t>(old >> 32) == epoch) ? static_cast<uint32_t>(old) : kInvalid;
    node.p = prob_chi2(L.chi2_sum, static_cast<float>(L.ndf_sum - 5u));
    node.all = r.all;
    node.ends = r.ends;
    node.pad[0] = node.pad[1] = 0u;
    dedup_nodes(P, step)[i] = node;
}

// Can a's history be contained in b's?  Equal numbers of measurements: the
// whole histories agree.  One more in b: a's first is b's second.
__device__ inline bool may_contain(const dedup_node& a, const dedup_node& b) {
    const uint32_t na = a.ends >> 24, nb = b.ends >> 24;
    if (na == 255u || nb == 255u) return true;
    if (na == nb) return a.all == b.all;
    if (na + 1u == nb) return (a.ends & 0xfffu) == ((b.ends >> 12) & 0xfffu);
    return na < nb;
}

// Links of the step, after k_find: the inputs' link counts (kept branches, or
// one hole link) laid out in input order, then the links written.  Kept apart
// from k_find so a partition with heavy inputs never holds the look-back
// chain of every later partition while it works.
template <bool kLogging>
__global__ __launch_bounds__(kBlock) void k_find_emit(ckf_params P) {
    __shared__ emit_shared S;
    step_ctl* ctl = P.ctl;
    if (ctl->done) {
        return;
    }
    const uint32_t step = ctl->step;
    const uint32_t n_in = ctl->n_in < P.in_cap ? ctl->n_in : P.in_cap;
    const uint32_t link_base = ctl->link_base;
    const uint32_t epoch = ctl->epoch;
    const bool dedup = step >= P.dup_min_len;
    const uint32_t kc = emit_chunks(n_in, kHeavyParts);
    const uint32_t part = kBlock * kc;
    const uint32_t n_parts = (n_in + part - 1u) / part;
    if (blockIdx.x == 0u && threadIdx.x == 0u) {
        // k_prop_emit's queue is cleared here, between its launches: a block
        // of it that starts after the step's advance then still finds it spent
        ctl->ticket[5].v = 0u;
    }
    if (blockIdx.x >= n_parts) {
        return;
    }
    for (;;) {
        const uint32_t p = block_ticket(&ctl->ticket[4].v, S);
        if (p >= n_parts) {
            break;
        }
        const uint32_t i0 = p * part + threadIdx.x;
        uint32_t n_out[kEmitChunks], first[kEmitChunks];
#pragma unroll
        for (uint32_t ch = 0; ch < kEmitChunks; ++ch) {
            const uint32_t i = i0 + ch * kBlock;
            const bool valid = ch < kc && i < n_in;
            const uint32_t count = valid ? P.find_count[i] : 0u;
            n_out[ch] = valid ? (count > 0u ? count : 1u) : 0u;
            first[ch] = n_out[ch];
        }
        const uint32_t total = block_prefix(first, 0, S);
        const uint32_t base = lo32(block_lookback(P.lb_lo[0], nullptr, p, epoch, pack2(total, 0u), S));
        if (p == n_parts - 1u && threadIdx.x == 0u) {
            ctl->n_links = base + total;
            ctl->emit_links = base + total;
        }
#pragma unroll
        for (uint32_t ch = 0; ch < kEmitChunks; ++ch) {
            const uint32_t i = i0 + ch * kBlock;
            const bool valid = ch < kc && i < n_in;
            const stage_head h = valid ? P.stage_in[i] : stage_head{};
            const uint32_t seed = valid ? h.seed : kInvalid;
            // head of the seed's contiguous run of inputs
            uint32_t prev_seed = __shfl(seed, (lane() + kWave - 1u) % kWave, kWave);
            if (lane() == 0u) {
                prev_seed = valid && i > 0u ? P.stage_in[i - 1u].seed : kInvalid;
            }
            if (!valid) {
                continue;
            }
            const uint32_t at = base + first[ch];
            if (i == 0u || prev_seed != seed) {
                P.seed_first[seed] = at;
            }
            // the previous link's history (a hole's state reference names its slot)
            link_history before{};
            if (step > 0u) {
                before = load_history(P, (step + 1u) & 1u, h.hole_ref & kRefMask);
            }
            for (uint32_t k = 0; k < n_out[ch]; ++k) {
                const uint32_t slot = flt_slot(P, i, k);
                if (slot >= P.flt_cap) {
                    break;  // k_find raised the overflow that discards this step
                }
                const dlink L = staged_link(h, P.stage_slot[slot], step, slot);
                const uint32_t g = link_base + at + k;
                if (g < P.link_cap && at + k < P.state_cap) {
                    P.links[g] = L;
                    const link_history r = extend_history(before, L.meas);
                    store_history(P, step & 1u, at + k, r);
                    if (dedup) {
                        dedup_insert(P, L, r, at + k, step, epoch);
                    }
                    if constexpr (kLogging) {
                        if (L.meas != kInvalid) {
                            // a row is 48 B: three 16-byte pieces each way
                            const float4* src = reinterpret_cast<const float4*>(
                                P.feat_slot + static_cast<size_t>(slot) * kFeatures);
                            float4* dst = reinterpret_cast<float4*>(
                                P.log_feat + static_cast<size_t>(g) * kFeatures);
                            const float4 f0 = src[0], f1 = src[1];
                            float4 f2 = src[2];
                            static_assert(kFeatures == 12 && kFeatStanding == 9, "feature 9 is .y of the third piece");
                            f2.y = standing_of(P.seed_run_min, seed, epoch, f2.y);
                            dst[0] = f0;
                            dst[1] = f1;
                            dst[2] = f2;
                        }
                    }
                } else {
                    set_overflow(ctl, 1u);
                }
            }
        }
    }
}

namespace {
// Is track `a` dominated by `b` (identical measurement history down to a's
// first link)?  traccc host :431-471.  Two links with the same previous link
// have the same history from there on, which ends the walk: the branches of a
// seed mostly part a few links back.
__device__ inline bool history_contained(const ckf_params& P, dlink a, dlink b) {
    for (;;) {
        while (a.meas == kInvalid && link_step(a) != 0u) a = load_link(P, a.prev);
        while (b.meas == kInvalid && link_step(b) != 0u) b = load_link(P, b.prev);
        if (a.meas != b.meas) return false;
        if (link_step(a) == 0u) return true;
        if (link_step(b) == 0u) return false;
        if (a.prev == b.prev) return true;
        a = load_link(P, a.prev);
        b = load_link(P, b.prev);
    }
}
}  // namespace

// Which links survive: one bit each, a 64-bit word per partition of 64.  A
// link is dropped when another has its history and a higher p-value (the lower
// index on equal ones).  The list's nodes carry the p-values and what the
// histories must agree in, so a pair costs one 32-byte load, and the histories
// are walked only for the pairs that they decide.  k_propagate counts the bits of a seed's links for the
// branch cap.
__global__ __launch_bounds__(kBlock) void k_dedup_mark(ckf_params P) {
    step_ctl* ctl = P.ctl;
    if (ctl->done || ctl->step < P.dup_min_len || (ctl->overflow & kFindOverflow) != 0u) {
        return;
    }
    const uint32_t n = step_links(*ctl, P.state_cap, P.link_cap);
    const uint32_t base = ctl->link_base;
    const uint32_t epoch = ctl->epoch;
    const uint32_t n_parts = (n + kWave - 1) / kWave;
    const dedup_node* nodes = dedup_nodes(P, ctl->step);
    xcd_ticket_run queue(&ctl->xcd_ticket[3][0].v, n_parts, 1u);
    for (;;) {
        const uint32_t p = queue.next();
        if (p >= n_parts) {
            break;
        }
        const uint32_t i = p * kWave + lane();
        bool alive = i < n;
        dedup_node own{};
        if (alive) {
            own = nodes[i];
        }
        if (alive && own.head != kDedupShort) {
            const uint64_t h = P.dedup_head[own.head];
            uint32_t j = (static_cast<uint32_t>(h >> 32) == epoch) ? static_cast<uint32_t>(h) : kInvalid;
            while (j != kInvalid) {
                const dedup_node node = nodes[j];
                const bool better = own.p != node.p ? node.p >= own.p : j < i;
                if (j != i && node.hash == own.hash && better && may_contain(own, node)) {
                    const dlink Li = load_link(P, base + i);
                    if (Li.ndf_sum > 5u && history_contained(P, Li, load_link(P, base + j))) {
                        alive = false;
                        break;
                    }
                }
                j = node.next;
            }
        }
        const uint64_t bits = wave_ballot(alive);
        if (lane() == 0u) {
            P.alive_bits[p] = bits;
        }
    }
}

// Surviving links among the step's links [from, to).
__device__ inline uint32_t count_alive(const uint64_t* bits, uint32_t from, uint32_t to) {
    uint32_t count = 0u;
    for (uint32_t w = from / 64u; w * 64u < to; ++w) {
        uint64_t b = bits[w];
        if (w == from / 64u) {
            b &= ~0ull << (from % 64u);
        }
        if (to - w * 64u < 64u) {
            b &= (1ull << (to % 64u)) - 1ull;
        }
        count += static_cast<uint32_t>(__popcll(b));
    }
    return count;
}

__device__ void advance_step(const ckf_params& P, step_ctl* ctl);

// ---------------------------------------------------------------------------
// propagate_to_next_surface
// ---------------------------------------------------------------------------
// The end of a link's propagation (status from the navigator): on NAV_FOUND
// the covariance (read now; the navigation does not need it, so it is not
// held in registers meanwhile) with the start surface's material at step 0,
// the transport to the new surface, its material, the sanity checks and the
// new state; the outcome flag (bit 0: next input, bits 1-2: tips).
template <int kT>
__device__ inline uint8_t finish_link(const ckf_params& P, const navigator<float, true, kT>& nav,
                                      int status, uint32_t end_sf, uint32_t i, uint32_t ref,
                                      uint32_t step, bool leader) {
    const uint32_t in_par = (step + 1u) & 1u;
    const uint32_t out_par = step & 1u;
    const bool success = (status == NAV_FOUND);
    bool ok = success;
    bool succ = false;
    uint32_t ntip = 0u;
    if (success) {
        float x[6], c[21];
        uint32_t sf = 0u;
        load_ref(P, ref, in_par, x, c, sf);
        if (step == 0u) {
            add_material(P, sf, x, c);
        }
        const geo_view G{P.sfs, P.n_layers, P.field};
        finish_transport<kT>(G, P.nav, nav, end_sf, x, c);
        sf = end_sf;
        add_material(P, sf, x, c);
        const float th = x[e_theta];
        if (th <= 0.f || th >= 6.28318530717958647692f) ok = false;
        if (!isfinite(x[e_phi])) ok = false;
        if (fabsf(x[e_qop]) == 0.f) ok = false;
        if (ok) {
            if (leader) {
                store_soa(P.state[out_par], P.state_cap, i, x, c, sf);
            }
            succ = true;
        }
    }
    if (!ok && step + 1u >= P.min_cands) ++ntip;
    if (success && step == P.max_cands - 1u) ++ntip;
    return static_cast<uint8_t>((succ ? 1u : 0u) | (ntip << 1));
}

// kT lanes propagate one link together (team navigator); 64 / kT links per
// wave partition.  The team leader writes the results.  With one lane per
// link and defer_links links or more, a propagation that needs a second layer
// search (a few % of them, but nearly every wave has one) is written to the
// defer buffer and continued by k_propagate_resume, so the wave does not run a
// second search, approach and window for one or two of its lanes.
//
// A propagation is a serial chain of ~100 us on one lane (Runge-Kutta steps,
// layer search, module windows): a step whose waves all fit on the chip is
// bound by that chain, which a team shortens, a larger one by the lanes, which
// a team spends on redundant steps.  So a launch runs only when its step has
// [from, below) links: two launches with different teams share the steps of a
// call (propagate_schedule, runtime.hip); the other one's blocks leave at once.
template <int kT>
__global__ __launch_bounds__(kBlock) void k_propagate(ckf_params P, uint32_t from, uint32_t below) {
    step_ctl* ctl = P.ctl;
    if (ctl->done) {
        return;
    }
    const uint32_t n = step_links(*ctl, P.state_cap, P.link_cap);
    // the grid is sized for the largest step: a block without a partition leaves
    if (n < from || n >= below || static_cast<uint64_t>(blockIdx.x) * kBlock >= static_cast<uint64_t>(n) * kT) {
        return;
    }
    // the navigation layers and groups live in LDS for the whole kernel
    __shared__ nav_tables s_nav;
    stage_nav_tables(s_nav, P.layers, P.n_layers, P.groups, P.n_groups, P.nav.mask_tol_max);
    const uint32_t step = ctl->step;
    const uint32_t base = ctl->link_base;
    constexpr uint32_t kLinksPerWave = kWave / kT;
    const uint32_t n_parts = (n + kLinksPerWave - 1) / kLinksPerWave;
    const uint32_t in_par = (step + 1u) & 1u;
    const bool dedup = step >= P.dup_min_len;
    const uint32_t tl = lane() % kT;
    const bool leader = (tl == 0u);
    const bool defer = (kT == 1) && P.defer_cap > 0u && n >= P.defer_links;

    xcd_ticket_run queue(&ctl->xcd_ticket[2][0].v, n_parts, 1u);
    for (;;) {
        const uint32_t p = queue.next();
        if (p >= n_parts) {
            break;
        }
        const uint32_t i = p * kLinksPerWave + lane() / kT;
        const bool valid = i < n;
        bool propagated = false;
        bool deferred = false;
        uint8_t flag = 0u;
        if (valid) {
            const dlink L = load_link(P, base + i);
            // its place among the seed's (surviving) links, for the branch cap
            const uint32_t first = P.seed_first[L.seed];
            bool alive = true;
            uint32_t rank = i - first;
            if (dedup) {
                alive = ((P.alive_bits[i / 64u] >> (i % 64u)) & 1ull) != 0ull;
                if (rank >= P.n_branch_seed) {
                    rank = count_alive(P.alive_bits, first, i);
                }
            }
            if (alive && rank < P.n_branch_seed) {
                if (link_skipped(L) > P.max_skip || link_consec(L) > P.max_consec) {
                    flag = static_cast<uint8_t>(1u << 1);
                } else {
                    float x[6];
                    uint32_t sf = 0u;
                    {
                        float c_later[21];
                        load_ref(P, L.state_ref, in_par, x, c_later, sf);
                    }
                    propagated = true;
                    const geo_view G{P.sfs, P.n_layers, P.field};
                    navigator<float, true, kT> nav =
                        make_navigator<kT>(G, s_nav.layers, P.nav, tl, &s_nav, P.n_groups);
                    bound_to_free<float, true>(P.sfs[sf], x, nav.st, nav.J);
                    uint32_t end_sf = 0u;
                    int status = nav.propagate(static_cast<int>(sf), end_sf, defer);
                    if (status == NAV_DEFER) {
                        const uint32_t k = atomicAdd(&ctl->n_defer.v, 1u);
                        if (k < P.defer_cap) {
                            uint32_t w[kDeferWords];
                            w[0] = i;
                            w[1] = static_cast<uint32_t>(nav.deferred_visited);
                            w[2] = static_cast<uint32_t>(nav.deferred_visited >> 32);
                            w[3] = nav.n_steps;
                            w[4] = __float_as_uint(nav.path);
                            const float fs[11] = {nav.st.pos.x, nav.st.pos.y, nav.st.pos.z,
                                                  nav.st.dir.x, nav.st.dir.y, nav.st.dir.z,
                                                  nav.st.qop,   nav.st.time,  nav.st.lo.x,
                                                  nav.st.lo.y,  nav.st.lo.z};
#pragma unroll
                            for (int e = 0; e < 11; ++e) w[5 + e] = __float_as_uint(fs[e]);
#pragma unroll
                            for (int r = 0; r < 3; ++r) {
#pragma unroll
                                for (int j = 0; j < 5; ++j) {
                                    w[16 + 5 * r + j] = __float_as_uint(nav.J.p[r][j]);
                                    w[31 + 5 * r + j] = __float_as_uint(nav.J.d[r][j]);
                                }
                            }
                            w[46] = __float_as_uint(nav.J.t_qop);
                            w[47] = L.state_ref;
#pragma unroll
                            for (uint32_t e = 0; e < kDeferWords; ++e) {
                                defer_words(P, step)[static_cast<size_t>(e) * P.defer_cap + k] = w[e];
                            }
                            deferred = true;
                        } else {
                            // no room: continue here
                            status = nav.layer_loop(nav.deferred_visited, 1u, end_sf, false);
                        }
                    }
                    if (!deferred) {
                        flag = finish_link<kT>(P, nav, status, end_sf, i, L.state_ref, step, leader);
                    }
                }
            }
        }
        // the link's outcome for k_prop_emit (a deferred one's comes from
        // k_propagate_resume); the propagation count here
        if (valid && leader && !deferred) {
            P.prop_flag[i] = flag;
        }
        const uint64_t mp = wave_ballot(leader && propagated);
        if (lane() == 0u && mp != 0ull) {
            atomicAdd(reinterpret_cast<unsigned long long*>(&ctl->n_props.v),
                      static_cast<unsigned long long>(__popcll(mp)));
        }
    }
}

// The deferred propagations of k_propagate<1>, one lane each: the layer
// loop continues from its second iteration with the saved state, then the
// same end as in k_propagate.
__global__ __launch_bounds__(kBlock) void k_propagate_resume(ckf_params P) {
    step_ctl* ctl = P.ctl;
    if (ctl->done) {
        return;
    }
    __shared__ nav_tables s_nav;
    stage_nav_tables(s_nav, P.layers, P.n_layers, P.groups, P.n_groups, P.nav.mask_tol_max);
    const uint32_t step = ctl->step;
    const uint32_t nd = ctl->n_defer.v;
    const uint32_t n = nd < P.defer_cap ? nd : P.defer_cap;
    const uint32_t n_parts = (n + kWave - 1u) / kWave;
    const bool takes = wave_takes_tickets(n_parts);
    for (;;) {
        const uint32_t p = takes ? wave_ticket(&ctl->ticket[7].v) : n_parts;
        if (p >= n_parts) {
            break;
        }
        const uint32_t k = p * kWave + lane();
        if (k >= n) {
            continue;
        }
        uint32_t w[kDeferWords];
#pragma unroll
        for (uint32_t e = 0; e < kDeferWords; ++e) {
            w[e] = defer_words(P, step)[static_cast<size_t>(e) * P.defer_cap + k];
        }
        const geo_view G{P.sfs, P.n_layers, P.field};
        navigator<float, true, 1> nav = make_navigator<1>(G, s_nav.layers, P.nav, 0u, &s_nav, P.n_groups);
        const uint64_t visited = static_cast<uint64_t>(w[1]) | (static_cast<uint64_t>(w[2]) << 32);
        nav.n_steps = w[3];
        nav.path = __uint_as_float(w[4]);
        nav.st.pos = {__uint_as_float(w[5]), __uint_as_float(w[6]), __uint_as_float(w[7])};
        nav.st.dir = {__uint_as_float(w[8]), __uint_as_float(w[9]), __uint_as_float(w[10])};
        nav.st.qop = __uint_as_float(w[11]);
        nav.st.time = __uint_as_float(w[12]);
        nav.st.lo = {__uint_as_float(w[13]), __uint_as_float(w[14]), __uint_as_float(w[15])};
#pragma unroll
        for (int r = 0; r < 3; ++r) {
#pragma unroll
            for (int j = 0; j < 5; ++j) {
                nav.J.p[r][j] = __uint_as_float(w[16 + 5 * r + j]);
                nav.J.d[r][j] = __uint_as_float(w[31 + 5 * r + j]);
            }
        }
        nav.J.t_qop = __uint_as_float(w[46]);
        uint32_t end_sf = 0u;
        const int status = nav.layer_loop(visited, 1u, end_sf, false);
        const uint32_t i = w[0];
        P.prop_flag[i] = finish_link<1>(P, nav, status, end_sf, i, w[47], step, true);
    }
}

// After k_propagate: the next step's inputs (links that reached a surface)
// and the tips, compacted in link order (partitions of up to 1,024 links); the
// block that finishes the step's last partition runs the step advance
// (fused_advance) so the step loop never waits on the host.
__global__ __launch_bounds__(kBlock) void k_prop_emit(ckf_params P, int fused_advance) {
    __shared__ emit_shared S;
    step_ctl* ctl = P.ctl;
    if (ctl->done) {
        return;
    }
    const emit_extent extent = emit_extent_of(*ctl);
    const uint32_t n = extent.n, kc = extent.chunks, n_parts = extent.parts;
    const uint32_t part = kBlock * kc;
    const uint32_t base = ctl->link_base;
    const uint32_t epoch = ctl->epoch;
    const uint32_t tip_base = ctl->n_tips;
    if (blockIdx.x >= n_parts) {
        // a step abandoned by an overflow has no links and no partition that
        // could end it
        if (blockIdx.x == 0u && threadIdx.x == 0u && fused_advance && (ctl->overflow & kFindOverflow) != 0u) {
            ctl->n_live = 0u;
            ctl->n_tips_step = 0u;
            advance_step(P, ctl);
        }
        return;
    }
    for (;;) {
        const uint32_t p = block_ticket(&ctl->ticket[5].v, S);
        if (p >= n_parts) {
            break;
        }
        const uint32_t i0 = p * part + threadIdx.x;
        uint32_t fl[kEmitChunks], live_at[kEmitChunks], tip_at[kEmitChunks];
#pragma unroll
        for (uint32_t ch = 0; ch < kEmitChunks; ++ch) {
            const uint32_t i = i0 + ch * kBlock;
            fl[ch] = (ch < kc && i < n) ? P.prop_flag[i] : 0u;
            live_at[ch] = fl[ch] & 1u;
            tip_at[ch] = fl[ch] >> 1;
        }
        const uint32_t s_tot = block_prefix(live_at, 0, S);
        const uint32_t t_tot = block_prefix(tip_at, 1, S);
        const uint64_t b = block_lookback(P.lb_lo[2], P.lb_hi[2], p, epoch, pack2(s_tot, t_tot), S);
#pragma unroll
        for (uint32_t ch = 0; ch < kEmitChunks; ++ch) {
            const uint32_t i = i0 + ch * kBlock;
            if ((fl[ch] & 1u) != 0u) {
                const uint32_t pos = lo32(b) + live_at[ch];
                if (pos < P.in_cap) {
                    P.live[pos] = i;
                } else {
                    set_overflow(ctl, 16u);
                }
            }
            uint32_t pos = tip_base + hi32(b) + tip_at[ch];
            for (uint32_t k = 0; k < (fl[ch] >> 1); ++k, ++pos) {
                if (pos < P.tip_cap) {
                    P.tips[pos] = base + i;
                } else {
                    set_overflow(ctl, 8u);
                }
            }
        }
        if (!fused_advance) {
            if (p == n_parts - 1u && threadIdx.x == 0u) {
                ctl->n_live = lo32(b) + s_tot;
                ctl->n_tips_step = hi32(b) + t_tot;
            }
            continue;
        }
        // The block that finishes the last partition advances the step: every
        // partition counts itself once it is written (counting every block of
        // the grid instead cost a 1,024-block grid 15 us of atomics on one
        // word).  A block that starts during or after the advance does nothing
        // (emit_extent).  The step's totals come from the last partition's
        // look-back words, which carry their own visibility; the overflow bits
        // that other blocks raise are read with a device-scope atomic load;
        // everything else the advance reads was written by earlier kernels, and
        // its own stores reach the next kernel at the launch boundary.
        __syncthreads();
        if (threadIdx.x == 0u) {
            const uint32_t before = atomicAdd(&ctl->exit_count.v, 1u);
            if (before + 1u == n_parts) {
                ctl->exit_count.v = 0u;
                ctl->n_live = lookback_inclusive(P.lb_lo[2], n_parts - 1u, epoch);
                ctl->n_tips_step = lookback_inclusive(P.lb_hi[2], n_parts - 1u, epoch);
                advance_step(P, ctl);
            }
        }
    }
}

// The advance by k_advance, or by the block that ends k_prop_emit: the overflow
// bits that other blocks raised with atomicOr live at the device's coherence point.
__device__ void advance_step(const ckf_params& P, step_ctl* ctl) {
    advance_ctl(ctl, P.max_cands, __hip_atomic_load(&ctl->overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

__global__ void k_advance(ckf_params P) {
    step_ctl* ctl = P.ctl;
    if (ctl->done) {
        return;
    }
    advance_step(P, ctl);
}

// ---------------------------------------------------------------------------
// build_tracks
// ---------------------------------------------------------------------------
// Tips in (step, event) segments: each tip's kept rank and constituent
// prefix, and every segment's bounds.  A partition is emit_chunks(n) chunks
// of kBlock tips with one look-back; the (event, step) key of a tip is
// ev * max_cands + step (the host keeps n_events * max_cands below 2^31).
__global__ __launch_bounds__(kBlock) void k_build_scan(ckf_params P) {
    __shared__ emit_shared S;
    step_ctl* ctl = P.ctl;
    const uint32_t n = ctl->n_tips < P.tip_cap ? ctl->n_tips : P.tip_cap;
    const uint32_t epoch = ctl->epoch;
    const uint32_t kc = emit_chunks(n, kLightParts);
    const uint32_t part = kBlock * kc;
    const uint32_t n_parts = (n + part - 1u) / part;
    const uint32_t n_steps = P.max_cands;
    if (blockIdx.x >= n_parts) {
        return;
    }
    for (;;) {
        const uint32_t p = block_ticket(&ctl->ticket[3].v, S);
        if (p >= n_parts) {
            break;
        }
        const uint32_t t0 = p * part + threadIdx.x;
        uint32_t kn[kEmitChunks];    // keep << 31 | n_cands
        uint32_t key[kEmitChunks];   // segment key
        uint32_t prev[kEmitChunks];  // segment key of the tip before
        uint32_t kp[kEmitChunks], cp[kEmitChunks];
#pragma unroll
        for (uint32_t ch = 0; ch < kEmitChunks; ++ch) {
            const uint32_t t = t0 + ch * kBlock;
            kn[ch] = key[ch] = prev[ch] = 0u;
            if (ch < kc && t < n) {
                const dlink L = load_link(P, P.tips[t]);
                const uint32_t st = link_step(L);
                const uint32_t nc = st + 1u - link_skipped(L);
                const bool keep = nc >= P.min_cands && nc <= P.max_cands;
                kn[ch] = (keep ? 0x80000000u : 0u) | nc;
                key[ch] = P.seed_event[L.seed] * n_steps + st;
                if (lane() == 0u && t > 0u) {
                    const dlink B = load_link(P, P.tips[t - 1u]);
                    prev[ch] = P.seed_event[B.seed] * n_steps + link_step(B);
                }
            }
            const uint32_t below = __shfl(key[ch], static_cast<int>((lane() + kWave - 1u) % kWave), kWave);
            prev[ch] = lane() == 0u ? prev[ch] : below;
            kp[ch] = kn[ch] >> 31;
            cp[ch] = (kn[ch] >> 31) != 0u ? kn[ch] & 0x7fffffffu : 0u;
        }
        const uint32_t k_tot = block_prefix(kp, 0, S);
        const uint32_t c_tot = block_prefix(cp, 1, S);
        const uint64_t b = block_lookback(P.lb_lo[3], P.lb_hi[3], p, epoch, pack2(k_tot, c_tot), S);
#pragma unroll
        for (uint32_t ch = 0; ch < kEmitChunks; ++ch) {
            const uint32_t t = t0 + ch * kBlock;
            if (ch >= kc || t >= n) {
                continue;
            }
            const bool keep = (kn[ch] >> 31) != 0u;
            const uint32_t kr = lo32(b) + kp[ch];
            const uint32_t cr = hi32(b) + cp[ch];
            P.tip_keep[t] = kn[ch];
            P.tip_rank[t] = kr;
            P.tip_cprefix[t] = cr;
            const uint32_t seg = key[ch];
            if (t == 0u || prev[ch] != seg) {
                P.seg_base[seg] = kr;
                P.seg_cbase[seg] = cr;
                // the previous segment ends where this one starts
                if (t > 0u) {
                    P.seg_count[prev[ch]] = kr;
                    P.seg_ccount[prev[ch]] = cr;
                }
            }
            if (t + 1u == n) {
                P.seg_count[seg] = kr + (keep ? 1u : 0u);
                P.seg_ccount[seg] = cr + (keep ? kn[ch] & 0x7fffffffu : 0u);
            }
        }
    }
}

// One workgroup: exclusive scan of the (event, step) table, event offsets and
// totals.
__global__ __launch_bounds__(1024) void k_build_table(ckf_params P) {
    __shared__ uint32_t s_a[1024];
    __shared__ uint32_t s_b[1024];
    const uint32_t S = P.max_cands;
    const uint32_t total = P.n_events * S;
    const uint32_t per = (total + blockDim.x - 1) / blockDim.x;
    const uint32_t lo = threadIdx.x * per;
    const uint32_t hi = lo + per < total ? lo + per : total;
    // seg_count / seg_ccount hold the kept / constituent prefix at the end of
    // each present segment (0 for absent ones); turn them into counts
    for (uint32_t k = lo; k < hi; ++k) {
        const uint32_t e = P.seg_count[k];
        const uint32_t ce = P.seg_ccount[k];
        P.seg_count[k] = e - (e ? P.seg_base[k] : 0u);
        P.seg_ccount[k] = ce - (e || ce ? P.seg_cbase[k] : 0u);
    }
    uint32_t a = 0u, b = 0u;
    for (uint32_t k = lo; k < hi; ++k) {
        a += P.seg_count[k];
        b += P.seg_ccount[k];
    }
    s_a[threadIdx.x] = a;
    s_b[threadIdx.x] = b;
    __syncthreads();
    for (uint32_t d = 1; d < blockDim.x; d <<= 1) {
        uint32_t va = 0u, vb = 0u;
        if (threadIdx.x >= d) {
            va = s_a[threadIdx.x - d];
            vb = s_b[threadIdx.x - d];
        }
        __syncthreads();
        s_a[threadIdx.x] += va;
        s_b[threadIdx.x] += vb;
        __syncthreads();
    }
    uint32_t ra = s_a[threadIdx.x] - a;
    uint32_t rb = s_b[threadIdx.x] - b;
    for (uint32_t k = lo; k < hi; ++k) {
        if (k % S == 0u) {
            P.event_track_off[k / S] = ra;
            P.event_const_off[k / S] = rb;
        }
        P.seg_off[k] = ra;
        P.seg_coff[k] = rb;
        ra += P.seg_count[k];
        rb += P.seg_ccount[k];
    }
    if (threadIdx.x == blockDim.x - 1) {
        P.event_track_off[P.n_events] = s_a[threadIdx.x];
        P.event_const_off[P.n_events] = s_b[threadIdx.x];
        P.ctl->n_tracks = s_a[threadIdx.x];
        P.ctl->n_constituents = s_b[threadIdx.x];
    }
}

// Ranking key of a kept tip among its seed's tips: more measurements first,
// then the lower chi2 sum, then the lower tip index.
__device__ inline uint64_t tip_rank_key(uint32_t n_cands, float chi2_sum, uint32_t t) {
    const uint32_t cb = __float_as_uint(chi2_sum >= 0.f ? chi2_sum : 0.f);  // order-preserving
    return (static_cast<uint64_t>(n_cands & 0xffu) << 56) |
           (static_cast<uint64_t>(~cb) << 24) |
           static_cast<uint64_t>((0xffffffu - (t < 0xffffffu ? t : 0xffffffu)) & 0xffffffu);
}

// Branch log: each seed's best kept tip (its survive labels go to that
// track's links only).
__global__ __launch_bounds__(kBlock) void k_label_best(ckf_params P) {
    const step_ctl* ctl = P.ctl;
    const uint32_t n = ctl->n_tips < P.tip_cap ? ctl->n_tips : P.tip_cap;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const uint32_t kv = P.tip_keep[t];
        if ((kv >> 31) == 0u) {
            continue;
        }
        const dlink L = load_link(P, P.tips[t]);
        atomicMax(reinterpret_cast<unsigned long long*>(&P.seed_best[L.seed]),
                  static_cast<unsigned long long>(tip_rank_key(kv & 0x7fffffffu, L.chi2_sum, t)));
    }
}

__global__ __launch_bounds__(kBlock) void k_build_write(ckf_params P) {
    const step_ctl* ctl = P.ctl;
    const uint32_t n = ctl->n_tips < P.tip_cap ? ctl->n_tips : P.tip_cap;
    const uint32_t S = P.max_cands;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const uint32_t kv = P.tip_keep[t];
        if ((kv >> 31) == 0u) {
            continue;
        }
        const uint32_t nc = kv & 0x7fffffffu;
        uint32_t g = P.tips[t];
        dlink L = load_link(P, g);
        const uint32_t ev = P.seed_event[L.seed];
        const size_t seg = static_cast<size_t>(ev) * S + link_step(L);
        const uint32_t pos = P.seg_off[seg] + (P.tip_rank[t] - P.seg_base[seg]);
        const uint32_t cpos = P.seg_coff[seg] + (P.tip_cprefix[t] - P.seg_cbase[seg]);
        if (pos >= P.out_cap || cpos + nc > P.out_const_cap) {
            continue;
        }
        const uint32_t moff = P.event_meas_off[ev];
        // logged runs: only the seed's best track marks its links as survivors
        const bool mark = P.log_label != nullptr &&
                          P.seed_best[L.seed] == tip_rank_key(nc, L.chi2_sum, t);
        if (P.vote_key != nullptr) {
            // p-value of the tip's running sums ranks the track in measurement votes
            const float vp = prob_chi2(L.chi2_sum, static_cast<float>(L.ndf_sum) - 5.f);
            P.vote_key[pos] = (static_cast<uint64_t>(__float_as_uint(vp)) << 32) |
                              static_cast<uint64_t>(0xffffffffu - pos);
        }
        float ndf = 0.f, chi2 = 0.f;
        for (int k = static_cast<int>(nc) - 1; k >= 0; --k) {
            while (L.meas == kInvalid && link_step(L) != 0u) {
                g = L.prev;
                L = load_link(P, g);
            }
            P.out_const[cpos + static_cast<uint32_t>(k)] = L.meas - moff;
            ndf += static_cast<float>(P.meas_info[L.meas] & 0xffu);
            chi2 += L.chi2;
            if (mark) {
                P.log_label[g] = 1u;  // this measurement link is on the seed's best track
            }
            if (k > 0) {
                g = L.prev;
                L = load_link(P, g);
            }
        }
        ndf -= 5.f;
        const uint32_t s = L.seed;
        P.out_outcome[pos] = 0u;
        P.out_surface[pos] = P.seed_surface[s];
        copy_track_params(P.seed_vec + 6u * static_cast<size_t>(s), P.seed_cov + 36u * static_cast<size_t>(s),
                          P.out_vec + 6u * static_cast<size_t>(pos), P.out_cov + 36u * static_cast<size_t>(pos));
        P.out_ndf[pos] = ndf;
        P.out_chi2[pos] = chi2;
        P.out_pval[pos] = prob_chi2(chi2, ndf);
        P.out_nholes[pos] = link_skipped(L);
        P.out_offsets[pos] = cpos;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        P.out_offsets[ctl->n_tracks < P.out_cap ? ctl->n_tracks : P.out_cap] = ctl->n_constituents;
    }
}

// ---------------------------------------------------------------------------
// diagnostics: single pieces of the step pipeline on plain arrays
// ---------------------------------------------------------------------------
__global__ void k_debug_kf(uint32_t n, const float* vec, const float* cov, const float2* meas,
                           const float2* var, const uint32_t* info, float* chi2, int32_t* status,
                           float* out_vec, float* out_cov) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) {
        return;
    }
    float x[6], c[21];
    #pragma unroll
    for (int k = 0; k < 6; ++k) x[k] = vec[6u * i + k];
    #pragma unroll
    for (int r = 0; r < 6; ++r)
        #pragma unroll
        for (int q = r; q < 6; ++q) c[sym_idx(r, q)] = cov[36u * i + 6u * r + q];
    const meas_data md = load_meas(meas, var, info, i);
    chi2[i] = predicted_chi2(md, x, c);
    const int st = gain_update(md, x, c);
    status[i] = st;
    #pragma unroll
    for (int k = 0; k < 6; ++k) out_vec[6u * i + k] = x[k];
    #pragma unroll
    for (int r = 0; r < 6; ++r)
        #pragma unroll
        for (int q = 0; q < 6; ++q) out_cov[36u * i + 6u * r + q] = c[sym_idx(r, q)];
}

__global__ void k_debug_propagate(ckf_params P, uint32_t n, const uint32_t* start, const float* vec,
                                  const float* cov, int apply_start_material, int32_t* status,
                                  uint32_t* end_surface, float* out_vec, float* out_cov, float* path,
                                  uint32_t* n_steps) {
    __shared__ nav_tables s_nav;
    stage_nav_tables(s_nav, P.layers, P.n_layers, P.groups, P.n_groups, P.nav.mask_tol_max);
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) {
        return;
    }
    float x[6], c[21];
    #pragma unroll
    for (int k = 0; k < 6; ++k) x[k] = vec[6u * i + k];
    #pragma unroll
    for (int r = 0; r < 6; ++r)
        #pragma unroll
        for (int q = r; q < 6; ++q) c[sym_idx(r, q)] = cov[36u * i + 6u * r + q];
    const uint32_t sf = start[i];
    if (apply_start_material) {
        add_material(P, sf, x, c);
    }
    navigator<float, true> nav;
    nav.sfs = P.sfs;
    nav.layers = s_nav.layers;
    nav.n_layers = P.n_layers;
    nav.groups = s_nav.groups;
    nav.n_groups = P.n_groups;
    nav.layer_boxes = s_nav.boxes;
    nav.group_boxes = s_nav.boxes + 64;
    nav.field = P.field;
    nav.cfg = P.nav;
    bound_to_free<float, true>(P.sfs[sf], x, nav.st, nav.J);
    uint32_t end_sf = 0u;
    const int st = nav.propagate(static_cast<int>(sf), end_sf);
    status[i] = st;
    path[i] = nav.path;
    n_steps[i] = nav.n_steps;
    end_surface[i] = end_sf;
    if (st != NAV_FOUND) {
        return;
    }
    float nx[6];
    float Jb[6][6];
    free_to_bound<float, true>(P.sfs[end_sf], nav.st, nav.J, P.field, P.nav.mass, P.nav.abs_q, nx,
                               Jb);
    float M[6][6];
    #pragma unroll
    for (int r = 0; r < 6; ++r)
        #pragma unroll
        for (int q = 0; q < 6; ++q) {
            float acc = 0.f;
            #pragma unroll
            for (int k = 0; k < 6; ++k) acc += Jb[r][k] * c[sym_idx(k, q)];
            M[r][q] = acc;
        }
    float nc[21];
    #pragma unroll
    for (int r = 0; r < 6; ++r)
        #pragma unroll
        for (int q = r; q < 6; ++q) {
            float acc = 0.f;
            #pragma unroll
            for (int k = 0; k < 6; ++k) acc += M[r][k] * Jb[q][k];
            nc[sym_idx(r, q)] = acc;
        }
    add_material(P, end_sf, nx, nc);
    #pragma unroll
    for (int k = 0; k < 6; ++k) out_vec[6u * i + k] = nx[k];
    #pragma unroll
    for (int r = 0; r < 6; ++r)
        #pragma unroll
        for (int q = 0; q < 6; ++q) out_cov[36u * i + 6u * r + q] = nc[sym_idx(r, q)];
}

hipError_t launch_debug_kf(uint32_t n, const float* vec, const float* cov, const float2* meas,
                           const float2* var, const uint32_t* info, float* chi2, int32_t* status,
                           float* out_vec, float* out_cov, hipStream_t stream) {
    hipLaunchKernelGGL(k_debug_kf, dim3((n + 255u) / 256u), dim3(256), 0, stream, n, vec, cov, meas,
                       var, info, chi2, status, out_vec, out_cov);
    return hipGetLastError();
}

hipError_t launch_debug_propagate(const ckf_params& P, uint32_t n, const uint32_t* start,
                                  const float* vec, const float* cov, int apply_start_material,
                                  int32_t* status, uint32_t* end_surface, float* out_vec,
                                  float* out_cov, float* path, uint32_t* n_steps,
                                  hipStream_t stream) {
    hipLaunchKernelGGL(k_debug_propagate, dim3((n + 63u) / 64u), dim3(64), 0, stream, P, n, start,
                       vec, cov, apply_start_material, status, end_surface, out_vec, out_cov, path,
                       n_steps);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_find_work(const ckf_params& P, const launch_shape& s, hipStream_t stream) {
    if (P.scored) {
        hipLaunchKernelGGL(k_find_list, dim3(s.list_blocks), dim3(kBlock), 0, stream, P);
        hipLaunchKernelGGL(k_score_update, dim3(s.score_blocks), dim3(kBlock), 0, stream, P);
    } else if (P.feat_slot != nullptr) {
        hipLaunchKernelGGL(k_find<kFindLogged>, dim3(s.find_blocks), dim3(kBlock), 0, stream, P);
    } else {
        hipLaunchKernelGGL(k_find<kFindPlain>, dim3(s.find_blocks), dim3(kBlock), 0, stream, P);
    }
    return hipGetLastError();
}

hipError_t launch_find_emit(const ckf_params& P, const launch_shape& s, hipStream_t stream) {
    if (P.feat_slot != nullptr) {
        hipLaunchKernelGGL(k_find_emit<true>, dim3(s.emit_blocks), dim3(kBlock), 0, stream, P);
    } else {
        hipLaunchKernelGGL(k_find_emit<false>, dim3(s.emit_blocks), dim3(kBlock), 0, stream, P);
    }
    return hipGetLastError();
}

hipError_t launch_find(const ckf_params& P, const launch_shape& s, hipStream_t stream) {
    const hipError_t e = launch_find_work(P, s, stream);
    if (e != hipSuccess) {
        return e;
    }
    return launch_find_emit(P, s, stream);
}

// Branch log compaction: measurement links [0, n) in order, 1024 per block.
__global__ __launch_bounds__(1024) void k_log_count(ckf_params P, uint32_t n, uint32_t* block_n) {
    __shared__ uint32_t s_n;
    if (threadIdx.x == 0) s_n = 0u;
    __syncthreads();
    const uint32_t g = blockIdx.x * 1024u + threadIdx.x;
    if (g < n && P.links[g].meas != kInvalid) atomicAdd(&s_n, 1u);
    __syncthreads();
    if (threadIdx.x == 0) block_n[blockIdx.x] = s_n;
}

__global__ __launch_bounds__(1024) void k_log_write(ckf_params P, uint32_t n, const uint32_t* block_off,
                                                    float* features, uint8_t* labels, uint32_t cap) {
    __shared__ uint32_t s_w[16];
    const uint32_t g = blockIdx.x * 1024u + threadIdx.x;
    const bool is_meas = g < n && P.links[g].meas != kInvalid;
    const uint64_t m = wave_ballot(is_meas);
    const uint32_t wv = threadIdx.x / kWave;
    if (lane() == 0u) s_w[wv] = static_cast<uint32_t>(__popcll(m));
    __syncthreads();
    uint32_t before = 0u;
    for (uint32_t w = 0; w < wv; ++w) before += s_w[w];
    if (is_meas) {
        const uint32_t pos = block_off[blockIdx.x] + before + prefix_count(m);
        if (pos < cap) {
#pragma unroll
            for (int q = 0; q < kFeatures; ++q) {
                features[static_cast<size_t>(pos) * kFeatures + q] = P.log_feat[static_cast<size_t>(g) * kFeatures + q];
            }
            labels[pos] = P.log_label[g];
        }
    }
}

hipError_t launch_label_best(const ckf_params& P, const launch_shape& s, hipStream_t stream) {
    hipLaunchKernelGGL(k_label_best, dim3(s.build_blocks), dim3(kBlock), 0, stream, P);
    return hipGetLastError();
}

hipError_t launch_log_count(const ckf_params& P, uint32_t n, uint32_t* block_n, hipStream_t stream) {
    hipLaunchKernelGGL(k_log_count, dim3((n + 1023u) / 1024u), dim3(1024), 0, stream, P, n, block_n);
    return hipGetLastError();
}

hipError_t launch_log_write(const ckf_params& P, uint32_t n, const uint32_t* block_off,
                            float* features, uint8_t* labels, uint32_t cap, hipStream_t stream) {
    hipLaunchKernelGGL(k_log_write, dim3((n + 1023u) / 1024u), dim3(1024), 0, stream, P, n,
                       block_off, features, labels, cap);
    return hipGetLastError();
}

hipError_t launch_dedup(const ckf_params& P, const launch_shape& s, hipStream_t stream) {
    hipLaunchKernelGGL(k_dedup_mark, dim3(s.dedup_blocks), dim3(kBlock), 0, stream, P);
    return hipGetLastError();
}

hipError_t launch_propagate(const ckf_params& P, const launch_shape& s, hipStream_t stream,
                            bool fused_advance) {
    const hipError_t e = launch_propagate_work(P, s, stream);
    if (e != hipSuccess) {
        return e;
    }
    return launch_prop_emit(P, s, stream, fused_advance);
}

hipError_t launch_prop_emit(const ckf_params& P, const launch_shape& s, hipStream_t stream,
                            bool fused_advance) {
    hipLaunchKernelGGL(k_prop_emit, dim3(s.emit_blocks), dim3(kBlock), 0, stream, P,
                       fused_advance ? 1 : 0);
    return hipGetLastError();
}

template <int kT>
void launch_team(const ckf_params& P, const prop_launch& l, hipStream_t stream) {
    hipLaunchKernelGGL(k_propagate<kT>, dim3(l.blocks), dim3(kBlock), 0, stream, P, l.from, l.below);
}

hipError_t launch_propagate_work(const ckf_params& P, const launch_shape& s, hipStream_t stream) {
    for (const prop_launch& l : s.prop) {
        switch (l.team) {
            case 16u: launch_team<16>(P, l, stream); break;
            case 8u: launch_team<8>(P, l, stream); break;
            case 4u: launch_team<4>(P, l, stream); break;
            case 2u: launch_team<2>(P, l, stream); break;
            case 1u: launch_team<1>(P, l, stream); break;
            default: break;  // an unused entry
        }
    }
    if (s.resume_blocks > 0u) {
        hipLaunchKernelGGL(k_propagate_resume, dim3(s.resume_blocks), dim3(kBlock), 0, stream, P);
    }
    return hipGetLastError();
}

hipError_t launch_advance(const ckf_params& P, hipStream_t stream) {
    hipLaunchKernelGGL(k_advance, dim3(1), dim3(1), 0, stream, P);
    return hipGetLastError();
}

hipError_t launch_ckf_step(const ckf_params& P, const launch_shape& s, hipStream_t stream,
                           bool with_dedup) {
    hipError_t e = launch_find(P, s, stream);
    if (e == hipSuccess && with_dedup) e = launch_dedup(P, s, stream);
    if (e == hipSuccess) e = launch_propagate(P, s, stream, true);
    return e;
}

hipError_t launch_build_count(const ckf_params& P, const launch_shape& s, hipStream_t stream) {
    hipLaunchKernelGGL(k_build_scan, dim3(s.build_blocks), dim3(kBlock), 0, stream, P);
    hipLaunchKernelGGL(k_build_table, dim3(1), dim3(1024), 0, stream, P);
    return hipGetLastError();
}

hipError_t launch_build_write(const ckf_params& P, const launch_shape& s, uint32_t n_tips,
                              hipStream_t stream) {
    // pointer chasing back from every tip: as many lanes in flight as there
    // are tips, so the walks overlap instead of queueing in a strided loop
    (void)s;
    const uint32_t want = (n_tips + kBlock - 1u) / kBlock;
    const uint32_t blocks = want < 1u ? 1u : (want > (1u << 20) ? (1u << 20) : want);
    hipLaunchKernelGGL(k_build_write, dim3(blocks), dim3(kBlock), 0, stream, P);
    return hipGetLastError();
}

}  // namespace tamd
