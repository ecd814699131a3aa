// Triplet seeding, spacepoint formation and track-parameter estimation for
// MI355X (C ABI: include/traccc_amd/seeding.h).
//
// The reference seeds one middle spacepoint at a time, grid bin by grid bin
// (core/src/seeding/seed_finding.cpp:62-118): bottom and top doublets over
// the phi x z neighbourhood (doublet_finding.hpp:55-105), triplets per bottom
// doublet with compatible-seed weights (triplet_finding.hpp:60-183), and the
// per-middle filter (seed_filtering.cpp:28-122).  Here:
//   k_sd_prep       per spacepoint: radius, phi, the selection and the grid
//                   bin; key (bin << 32 | index)
//   radix sort      the keys: spacepoints in the reference's grid order
//                   (bin, then index), the middle order of the seeding
//   k_sd_place      the spacepoints in that order (16 B each) and the bins'
//                   bounds, from where neighbouring keys differ
//   k_sd_doublets   one wave per middle spacepoint: the neighbourhood's
//                   candidates in zone order, 64 at a time; a ballot keeps
//                   the compatible ones in order (count pass, scan, fill pass)
//   k_sd_middle     one wave per middle: its triplets, their weights (the
//                   compatible-seed bonus over the triplets of the same bottom,
//                   in the reference's order) and the filter (weight bonus,
//                   single-seed cut, the best maxSeedsPerSpM by (weight,
//                   y^2 + z^2 sum, finding order), the per-middle cut), in LDS
//   k_sd_triplets, k_sd_weights, k_sd_filter
//                   the same in HBM for the middles whose tops or triplets do
//                   not fit there
//   k_sd_compact    the seeds in middle order
// Every single-precision expression rounds as written (no contraction), as
// in the oracle, so the cut decisions agree exactly.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "../ckf/handles.hpp"
#include "../ckf/wave.hpp"
#include "../common/errors.hpp"
#include "../common/readback.hpp"
#include "../common/scan.hpp"
#include "../core/geometry.hpp"
#include "traccc_amd/seeding.h"

#pragma clang fp contract(off)

namespace tamd {
namespace {

constexpr uint32_t kSdBlock = 256;
constexpr uint32_t kSdWaves = kSdBlock / kWave;
constexpr uint32_t kNoSp = 0xffffffffu;

struct sd_axes {
    uint32_t nphi, nz;
    float phi_min, phi_max, z_min, z_max;
};

struct doublet_rec {
    uint32_t sp;
    float Zo, cot, iDR, Er, U, V;
};

struct triplet_rec {
    uint32_t b, t;
    float curv, w;
    uint32_t seg0, seg1;  // the triplets of the same bottom doublet
};

struct seed_rec {
    uint32_t b, m, t;
    float w;
};

struct sd_ctl {
    uint32_t n_valid;
    uint32_t n_bot, n_top, n_trip, n_seeds;
    uint32_t pad[3];
};

struct sd_params {
    ckf_seedfinder_config c;
    ckf_seedfilter_config f;
    sd_axes A;
    uint32_t n_sp;
    const float* xyz;
    const float* vr;  // may be null
    const float* vz;  // may be null
    float* rad;
    float* phi;
    uint64_t* keys;
    const uint64_t* sorted;
    float4* pts;  // grid order: x, y, z, radius
    uint32_t* bin_off;
    uint32_t nbins;
    uint32_t* cnt_b;  // per middle (grid order)
    uint32_t* off_b;
    uint32_t* cnt_t;
    uint32_t* off_t;
    doublet_rec* bot;
    doublet_rec* top;
    uint32_t* cnt_tr;
    uint32_t* off_tr;
    triplet_rec* trip;
    uint32_t* cnt_s;
    uint32_t* off_s;
    seed_rec* slots;
    seed_rec* seeds;
    sd_ctl* ctl;
};

// Order this wave's LDS accesses before and after (no other wave shares them).
__device__ inline void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ inline float sp_vr(const sd_params& P, uint32_t i) { return P.vr ? P.vr[i] : 0.f; }
__device__ inline float sp_vz(const sd_params& P, uint32_t i) { return P.vz ? P.vz[i] : 0.f; }

// the reference's circular axis (core/include/traccc/seeding/grids/axis.hpp:227-420)
__device__ inline uint32_t phi_bin(const sd_axes& A, float v) {
    const int ib = static_cast<int>((v - A.phi_min) / (A.phi_max - A.phi_min) * static_cast<float>(A.nphi));
    if (ib >= 0 && ib < static_cast<int>(A.nphi)) return static_cast<uint32_t>(ib);
    return ib < 0 ? A.nphi + static_cast<uint32_t>(ib) : static_cast<uint32_t>(ib) - A.nphi;
}
__device__ inline uint32_t phi_remap(const sd_axes& A, uint32_t b, int s) {
    const int o = static_cast<int>(b) + s;
    if (o >= 0 && o < static_cast<int>(A.nphi)) return static_cast<uint32_t>(o);
    if (o < 0) return static_cast<uint32_t>(static_cast<int>(A.nphi) + o);
    return static_cast<uint32_t>(o) - A.nphi;
}
// the zone's bins: element q of count (a wrapping zone lists the bins past
// the last one from 0 again)
struct phi_zone {
    uint32_t lo, count, nphi;
    bool wraps;
    __device__ uint32_t at(uint32_t q) const {
        if (!wraps) return lo + q;
        const uint32_t n = lo + q;
        return n > nphi - 1u ? n - nphi : n;
    }
};
__device__ inline phi_zone make_phi_zone(const sd_axes& A, float v, const uint32_t* nh) {
    const uint32_t g = phi_bin(A, v);
    const uint32_t lo = phi_remap(A, g, -static_cast<int>(nh[0]));
    const uint32_t hi = phi_remap(A, g, static_cast<int>(nh[1]));
    phi_zone z;
    z.lo = lo;
    z.nphi = A.nphi;
    z.wraps = !(lo < hi);
    z.count = z.wraps ? A.nphi - lo + hi + 1u : hi - lo + 1u;
    return z;
}
// the reference's closed axis (axis.hpp:37-225)
__device__ inline uint32_t z_bin(const sd_axes& A, float v) {
    const int ib = static_cast<int>((v - A.z_min) / (A.z_max - A.z_min) * static_cast<float>(A.nz));
    if (ib >= 0 && ib < static_cast<int>(A.nz)) return static_cast<uint32_t>(ib);
    return ib < 0 ? 0u : A.nz - 1u;
}
__device__ inline void z_zone(const sd_axes& A, float v, const uint32_t* nh, uint32_t& a, uint32_t& count) {
    const int ib = static_cast<int>((v - A.z_min) / (A.z_max - A.z_min) * static_cast<float>(A.nz));
    const int lo = ib - static_cast<int>(nh[0]);
    const int hi = ib + static_cast<int>(nh[1]);
    a = lo >= 0 ? static_cast<uint32_t>(lo) : 0u;
    const uint32_t b = hi < static_cast<int>(A.nz) ? static_cast<uint32_t>(hi) : A.nz - 1u;
    count = b - a + 1u;
}

// doublet_finding_helper.hpp:53-224
__device__ inline bool doublet_ok(bool bottom, float mx, float my, float mz, float mr, float ox, float oy,
                                  float oz, float orr, const ckf_seedfinder_config& c) {
    float deltaR, cotTheta, zOrigin;
    if (bottom) {
        deltaR = mr - orr;
        cotTheta = mz - oz;
        zOrigin = mz * deltaR - mr * cotTheta;
    } else {
        deltaR = orr - mr;
        cotTheta = oz - mz;
        zOrigin = mz * deltaR - mr * cotTheta;
    }
    if ((deltaR >= c.deltaRMax) || (deltaR <= c.deltaRMin) || (fabsf(cotTheta) >= c.cotThetaMax * deltaR) ||
        (zOrigin <= c.collisionRegionMin * deltaR) || (zOrigin >= c.collisionRegionMax * deltaR) ||
        fabsf(cotTheta) >= c.deltaZMax) {
        return false;
    }
    const float midX = 0.5f * (mx + ox);
    const float midY = 0.5f * (my + oy);
    const float slope = (oy - my) / (ox - mx);
    const float deltaX = ox - mx;
    const float deltaY = oy - my;
    const float deltaXY2 = deltaX * deltaX + deltaY * deltaY;
    const float sagitta = sqrtf(c.minHelixRadius * c.minHelixRadius - deltaXY2 / 4.f);
    const float denom = sqrtf((slope * slope + 1) / (slope * slope));
    const float cosA = 1.f / denom;
    const float sinA = -1.f / (slope * denom);
    const float mdx = sagitta * cosA;
    const float mdy = sagitta * sinA;
    const float mp1X = midX + mdx, mp2X = midX - mdx, mp1Y = midY + mdy, mp2Y = midY - mdy;
    const float mp1R2 = mp1X * mp1X + mp1Y * mp1Y;
    const float mp2R2 = mp2X * mp2X + mp2Y * mp2Y;
    const float m = (mp2R2 < mp1R2) ? mp2R2 : mp1R2;  // std::min
    return !(m <= ((c.minHelixRadius - c.impactMax) * (c.minHelixRadius - c.impactMax)));
}

// doublet_finding_helper.hpp:226-264
__device__ inline doublet_rec transform(bool bottom, uint32_t osp, float mx, float my, float mz, float mr,
                                        float mvr, float mvz, float ox, float oy, float oz, float ovr,
                                        float ovz) {
    const float cosPhiM = mx / mr;
    const float sinPhiM = my / mr;
    const float deltaX = ox - mx;
    const float deltaY = oy - my;
    const float deltaZ = oz - mz;
    const float x = deltaX * cosPhiM + deltaY * sinPhiM;
    const float y = deltaY * cosPhiM - deltaX * sinPhiM;
    const float iDeltaR2 = 1.f / (deltaX * deltaX + deltaY * deltaY);
    const float iDeltaR = sqrtf(iDeltaR2);
    float cot = deltaZ * iDeltaR;
    if (bottom) cot = -cot;
    doublet_rec d;
    d.sp = osp;
    d.cot = cot;
    d.Zo = mz - mr * cot;
    d.iDR = iDeltaR;
    d.U = x * iDeltaR2;
    d.V = y * iDeltaR2;
    d.Er = ((mvz + ovz) + (cot * cot) * (mvr + ovr)) * iDeltaR2;
    return d;
}

// Whether triplet_ok's first cut, |sqrt(d2) - sqrt(e2)| > sqrt(scat2) with the
// scattering angle's d2 and its error e2, ends the pair for certain, without its
// square root: (sqrt(e2) + sqrt(scat2))^2 <= 2 (e2 + scat2), so d2 above that by
// 1e-4 is above the cut by more than the cut's rounding (4e-7 of d2).  Pairs that
// this leaves go through triplet_ok.
__device__ inline bool triplet_scatters(float mvr, float mvz, const doublet_rec& lb, float t_Er, float t_cot,
                                        float t_iDR, float scat2) {
    const float error2 = t_Er + lb.Er + 2.f * (lb.cot * t_cot * mvr + mvz) * lb.iDR * t_iDR;
    const float d = lb.cot - t_cot;
    return error2 >= 0.f && d * d > 2.0002f * (error2 + scat2);
}

// triplet_finding_helper.hpp:46-141
__device__ inline bool triplet_ok(float mr, float mvr, float mvz, const doublet_rec& lb, const doublet_rec& lt,
                                  const ckf_seedfinder_config& c, float iSinTheta2, float scat2, float& curvature,
                                  float& impact) {
    const float error2 = lt.Er + lb.Er + 2.f * (lb.cot * lt.cot * mvr + mvz) * lb.iDR * lt.iDR;
    float deltaCotTheta = lb.cot - lt.cot;
    const float deltaCotTheta2 = deltaCotTheta * deltaCotTheta;
    float dCotThetaMinusError2 = 0.f;
    if (deltaCotTheta2 - error2 > 0) {
        deltaCotTheta = fabsf(deltaCotTheta);
        const float error = sqrtf(error2);
        dCotThetaMinusError2 = deltaCotTheta2 + error2 - 2.f * deltaCotTheta * error;
        if (dCotThetaMinusError2 > scat2) return false;
    }
    const float dU = lt.U - lb.U;
    if (dU == 0.f) return false;
    const float A = (lt.V - lb.V) / dU;
    const float S2 = 1.f + A * A;
    const float B = lb.V - A * lb.U;
    const float B2 = B * B;
    if (S2 < B2 * c.minHelixDiameter2) return false;
    const float iHelixDiameter2 = B2 / S2;
    float pT2scatter = 4.f * iHelixDiameter2 * c.pT2perRadius;
    const float pT = c.pTPerHelixRadius * sqrtf(S2 / B2) / 2.f;
    if (pT > c.maxPtScattering) {
        const float pTscatter = c.highland / c.maxPtScattering;
        pT2scatter = pTscatter * pTscatter;
    }
    const float p2scatter = pT2scatter * iSinTheta2;
    if ((deltaCotTheta2 - error2 > 0.f) &&
        (dCotThetaMinusError2 > p2scatter * c.sigmaScattering * c.sigmaScattering)) {
        return false;
    }
    curvature = B / sqrtf(S2);
    impact = fabsf((A - B * mr) * mr);
    return !(impact > c.impactMax);
}

// spacepoint_binning_helper.hpp:110-127, spacepoint_binning.cpp:40-50
__global__ __launch_bounds__(kSdBlock) void k_sd_prep(sd_params P) {
    for (uint32_t b0 = blockIdx.x * blockDim.x; b0 < P.n_sp; b0 += gridDim.x * blockDim.x) {
        const uint32_t i = b0 + threadIdx.x;
        bool valid = false;
        if (i < P.n_sp) {
            const float x = P.xyz[3 * i], y = P.xyz[3 * i + 1], z = P.xyz[3 * i + 2];
            const float r = sqrtf(x * x + y * y);
            const float phi = atan2f(y, x);
            P.rad[i] = r;
            P.phi[i] = phi;
            const ckf_seedfinder_config& c = P.c;
            valid = !(z > c.zMax || z < c.zMin) && !(phi > c.phiMax || phi < c.phiMin);
            if (valid) {
                const float bx = c.beamPos[0], by = c.beamPos[1];
                const float dx = x - bx, dy = y - by;
                const size_t nr = static_cast<size_t>(c.rMax + sqrtf(bx * bx + by * by));
                valid = static_cast<size_t>(sqrtf(dx * dx + dy * dy)) < nr;
            }
            uint64_t key = ~0ull;
            if (valid) {
                const uint32_t bin = phi_bin(P.A, phi) + P.A.nphi * z_bin(P.A, z);
                key = (static_cast<uint64_t>(bin) << 32) | i;
            }
            P.keys[i] = key;
        }
    }
}

// The spacepoints in grid order and every bin's first one: where the bin of a
// sorted key differs from the one before, the bins in between start (counting
// them with atomics took 140 us for 57,000 spacepoints in 77 bins).  The
// rejected ones come last, as bin nbins: it starts at the number of valid ones.
__global__ __launch_bounds__(kSdBlock) void k_sd_place(sd_params P) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < P.n_sp; k += gridDim.x * blockDim.x) {
        const uint64_t key = P.sorted[k];
        const uint32_t bin = key == ~0ull ? P.nbins : static_cast<uint32_t>(key >> 32);
        uint32_t from = 0u;
        if (k > 0u) {
            const uint64_t below = P.sorted[k - 1u];
            from = (below == ~0ull ? P.nbins : static_cast<uint32_t>(below >> 32)) + 1u;
        }
        for (uint32_t b = from; b <= bin; ++b) P.bin_off[b] = k;
        if (bin == P.nbins && from <= bin) P.ctl->n_valid = k;
        if (k + 1u == P.n_sp && bin < P.nbins) {
            for (uint32_t b = bin + 1u; b <= P.nbins; ++b) P.bin_off[b] = P.n_sp;
            P.ctl->n_valid = P.n_sp;
        }
        if (bin < P.nbins) {
            const uint32_t i = static_cast<uint32_t>(key);
            P.pts[k] = make_float4(P.xyz[3 * i], P.xyz[3 * i + 1], P.xyz[3 * i + 2], P.rad[i]);
        }
    }
}

// One wave per middle spacepoint (grid order p): its bottom and top doublets.
template <bool kFill>
__global__ __launch_bounds__(kSdBlock) void k_sd_doublets(sd_params P) {
    const uint32_t n_mid = P.ctl->n_valid;
    const uint32_t l = lane();
    for (uint32_t p = blockIdx.x * kSdWaves + threadIdx.x / kWave; p < n_mid; p += gridDim.x * kSdWaves) {
        if (kFill && P.cnt_b[p] == 0u) {
            continue;  // no bottoms: nothing of this middle is kept
        }
        const uint32_t mi = static_cast<uint32_t>(P.sorted[p]);
        const float4 mid = P.pts[p];
        const float mx = mid.x, my = mid.y, mz = mid.z, mr = mid.w;
        const float mvr = sp_vr(P, mi), mvz = sp_vz(P, mi);
        const phi_zone pz = make_phi_zone(P.A, P.phi[mi], P.c.neighbor_scope);
        uint32_t za, zc;
        z_zone(P.A, mz, P.c.neighbor_scope, za, zc);
        uint32_t nb = 0u, nt = 0u;
        const uint32_t ob = kFill ? P.off_b[p] : 0u, ot = kFill ? P.off_t[p] : 0u;
        for (uint32_t qp = 0; qp < pz.count; ++qp) {
            const uint32_t pb = pz.at(qp);
            for (uint32_t qz = 0; qz < zc; ++qz) {
                const uint32_t bin = pb + (za + qz) * P.A.nphi;
                const uint32_t s0 = P.bin_off[bin], s1 = P.bin_off[bin + 1u];
                for (uint32_t c0 = s0; c0 < s1; c0 += kWave) {
                    const uint32_t k = c0 + l;
                    bool isb = false, ist = false;
                    uint32_t oi = 0u;
                    float ox = 0.f, oy = 0.f, oz = 0.f, orr = 0.f;
                    if (k < s1) {
                        const float4 o = P.pts[k];
                        ox = o.x;
                        oy = o.y;
                        oz = o.z;
                        orr = o.w;
                        isb = doublet_ok(true, mx, my, mz, mr, ox, oy, oz, orr, P.c);
                        ist = doublet_ok(false, mx, my, mz, mr, ox, oy, oz, orr, P.c);
                    }
                    const uint64_t mb = wave_ballot(isb), mt = wave_ballot(ist);
                    if constexpr (kFill) {
                        if (isb || ist) oi = static_cast<uint32_t>(P.sorted[k]);
                        if (isb) {
                            P.bot[ob + nb + prefix_count(mb)] =
                                transform(true, oi, mx, my, mz, mr, mvr, mvz, ox, oy, oz, sp_vr(P, oi), sp_vz(P, oi));
                        }
                        if (ist) {
                            P.top[ot + nt + prefix_count(mt)] =
                                transform(false, oi, mx, my, mz, mr, mvr, mvz, ox, oy, oz, sp_vr(P, oi), sp_vz(P, oi));
                        }
                    }
                    nb += __popcll(mb);
                    nt += __popcll(mt);
                }
            }
        }
        if (!kFill && l == 0u) {
            // a middle without bottoms makes no seed: its tops are not kept
            P.cnt_b[p] = nb;
            P.cnt_t[p] = nb > 0u ? nt : 0u;
        }
    }
}

// One wave per middle that k_sd_middle left (cnt_tr): per bottom doublet, its
// triplets with the tops.
__global__ __launch_bounds__(kSdBlock) void k_sd_triplets(sd_params P) {
    const uint32_t n_mid = P.ctl->n_valid;
    const uint32_t l = lane();
    const float ss2 = P.c.sigmaScattering * P.c.sigmaScattering;
    for (uint32_t p = blockIdx.x * kSdWaves + threadIdx.x / kWave; p < n_mid; p += gridDim.x * kSdWaves) {
        if (P.cnt_tr[p] == 0u) {
            continue;
        }
        const uint32_t nb = P.cnt_b[p], nt = P.cnt_t[p];
        const uint32_t mi = static_cast<uint32_t>(P.sorted[p]);
        const float mr = P.rad[mi], mvr = sp_vr(P, mi), mvz = sp_vz(P, mi);
        const doublet_rec* B = P.bot + P.off_b[p];
        const doublet_rec* T = P.top + P.off_t[p];
        uint32_t n = P.off_tr[p];
        for (uint32_t jb = 0; jb < nb; ++jb) {
            const doublet_rec lb = B[jb];
            const float iSinTheta2 = 1.f + lb.cot * lb.cot;
            float scat2 = P.c.maxScatteringAngle2 * iSinTheta2;
            scat2 *= ss2;
            // the segment of this bottom is counted first
            uint32_t seg = 0u;
            for (uint32_t c0 = 0; c0 < nt; c0 += kWave) {
                bool ok = false;
                if (c0 + l < nt) {
                    float cv, ip;
                    ok = triplet_ok(mr, mvr, mvz, lb, T[c0 + l], P.c, iSinTheta2, scat2, cv, ip);
                }
                seg += __popcll(wave_ballot(ok));
            }
            uint32_t w = 0u;
            for (uint32_t c0 = 0; c0 < nt; c0 += kWave) {
                bool ok = false;
                float cv = 0.f, ip = 0.f;
                if (c0 + l < nt) ok = triplet_ok(mr, mvr, mvz, lb, T[c0 + l], P.c, iSinTheta2, scat2, cv, ip);
                const uint64_t m = wave_ballot(ok);
                if (ok) {
                    triplet_rec r;
                    r.b = lb.sp;
                    r.t = T[c0 + l].sp;
                    r.curv = cv;
                    r.w = -ip * P.f.impactWeightFactor;
                    r.seg0 = n;
                    r.seg1 = n + seg;
                    P.trip[n + w + prefix_count(m)] = r;
                }
                w += __popcll(m);
            }
            n += w;
        }
    }
}

// triplet_finding.hpp:131-178: the compatible-seed bonus of each triplet
// over the triplets of its bottom doublet, in their order.
__global__ __launch_bounds__(kSdBlock) void k_sd_weights(sd_params P) {
    const uint32_t n = P.ctl->n_trip;
    const ckf_seedfilter_config& f = P.f;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const triplet_rec ti = P.trip[i];
        const float rt = P.rad[ti.t];
        const float lo = ti.curv - f.deltaInvHelixDiameter;
        const float hi = ti.curv + f.deltaInvHelixDiameter;
        float compat[8];
        uint32_t nc = 0u;
        float w = ti.w;
        const uint32_t limit = f.compatSeedLimit < 8u ? f.compatSeedLimit : 8u;
        for (uint32_t j = ti.seg0; j < ti.seg1; ++j) {
            if (j == i) continue;
            const triplet_rec tj = P.trip[j];
            const float ro = P.rad[tj.t];
            const float dr = rt - ro;
            if (fabsf(dr) < f.deltaRMin) continue;
            if (tj.curv < lo) continue;
            if (tj.curv > hi) continue;
            bool fresh = true;
            for (uint32_t q = 0; q < nc; ++q) {
                if (fabsf(compat[q] - ro) < f.deltaRMin) {
                    fresh = false;
                    break;
                }
            }
            if (fresh) {
                compat[nc < 8u ? nc : 7u] = ro;
                ++nc;
                w += f.compatSeedWeight;
            }
            if (nc >= limit) break;
        }
        P.trip[i].w = w;
    }
}

struct seed_key {
    float w, ysum;
    uint32_t idx;
};
// a before b in the reference's sort (weight, then the y^2 + z^2 sum, both
// descending); the finding order on a full tie
__device__ inline bool before(const seed_key& a, const seed_key& b) {
    if (a.w != b.w) return a.w > b.w;
    if (a.ysum != b.ysum) return a.ysum > b.ysum;
    return a.idx < b.idx;
}

// What k_sd_middle holds in LDS of a middle (16 KB a wave, ten waves a CU):
// tops, the pairs of 64 bottoms that the first cut leaves, triplets.
constexpr uint32_t kMidTops = 256;
constexpr uint32_t kMidPairs = 1024;
constexpr uint32_t kMidTrips = 256;
constexpr uint32_t kTopWords = kMidTops / 64u;
constexpr uint32_t kTripSlots = kMidTrips / kWave;

struct middle_lds {
    float4 t_Er[kMidTops / 4u], t_cot[kMidTops / 4u], t_iDR[kMidTops / 4u];  // read four at a time
    float t_U[kMidTops], t_V[kMidTops];
    uint32_t t_sp[kMidTops];
    float b_Er[kWave], b_cot[kWave], b_iDR[kWave], b_U[kWave], b_V[kWave];
    uint32_t b_sp[kWave], b_n[kWave];
    uint16_t pair[kMidPairs];  // bottom << 8 | top
    uint32_t b[kMidTrips], t[kMidTrips];
    float curv[kMidTrips], w[kMidTrips], rt[kMidTrips];
    uint16_t seg0[kMidTrips], seg1[kMidTrips];  // seg0: the bottom's lane until its segment is known
};

// The number of a middle's triplets, from HBM: a lane takes a bottom, or a top
// where that takes fewer turns (3 bottoms with 300 tops: 15 turns for 300; 3,000
// such middles in 1,918 us for 2,361).
__device__ __noinline__ uint32_t count_triplets(const sd_params& P, const doublet_rec* B, const doublet_rec* T,
                                                uint32_t nb, uint32_t nt, float mr, float mvr, float mvz) {
    const float ss2 = P.c.sigmaScattering * P.c.sigmaScattering;
    uint32_t n = 0u;
    if (uint64_t(nb) * ((nt + kWave - 1u) / kWave) < uint64_t(nt) * ((nb + kWave - 1u) / kWave)) {
        for (uint32_t jb = 0; jb < nb; ++jb) {
            const doublet_rec lb = B[jb];
            const float iSinTheta2 = 1.f + lb.cot * lb.cot;
            float scat2 = P.c.maxScatteringAngle2 * iSinTheta2;
            scat2 *= ss2;
            for (uint32_t j = lane(); j < nt; j += kWave) {
                float cv, ip;
                n += triplet_ok(mr, mvr, mvz, lb, T[j], P.c, iSinTheta2, scat2, cv, ip) ? 1u : 0u;
            }
        }
        return wave_broadcast(wave_inclusive_scan(n), kWave - 1);
    }
    for (uint32_t jb = lane(); jb < nb; jb += kWave) {
        const doublet_rec lb = B[jb];
        const float iSinTheta2 = 1.f + lb.cot * lb.cot;
        float scat2 = P.c.maxScatteringAngle2 * iSinTheta2;
        scat2 *= ss2;
        for (uint32_t j = 0; j < nt; ++j) {
            float cv, ip;
            n += triplet_ok(mr, mvr, mvz, lb, T[j], P.c, iSinTheta2, scat2, cv, ip) ? 1u : 0u;
        }
    }
    return wave_broadcast(wave_inclusive_scan(n), kWave - 1);
}

// One wave per middle: triplets (triplet_finding.hpp:60-183), weights and
// filter (seed_filtering.cpp:36-121) without a pass through HBM in between.
//
// A lane takes a bottom: the tops come from LDS, the same ones for all lanes, and
// a test without square root or division ends 98 % of the pairs (9,600 a middle
// in a 10,000 muon event).  The rest are listed in the reference's order (bottom,
// then top) and evaluated 64 at a time, so the passing ones are placed by a
// ballot.  The first test's vector arithmetic and LDS reads bound it.  50,000
// middles: 624 us; every pair evaluated with lanes on tops, and twice more to
// count a bottom's segment and the middle's triplets, 4,520 us; a resident grid
// striding over the middles 1,265 (they differ by a factor of a hundred: one
// block each, as the hardware places them), tops read one at a time 877.
__global__ __launch_bounds__(kWave) void k_sd_middle(sd_params P) {
    __shared__ middle_lds S;
    float* t_Er = reinterpret_cast<float*>(S.t_Er);
    float* t_cot = reinterpret_cast<float*>(S.t_cot);
    float* t_iDR = reinterpret_cast<float*>(S.t_iDR);
    const uint32_t n_mid = P.ctl->n_valid;
    const uint32_t l = lane();
    const ckf_seedfilter_config& f = P.f;
    const float ss2 = P.c.sigmaScattering * P.c.sigmaScattering;
    const uint32_t max_s = P.c.maxSeedsPerSpM;
    for (uint32_t p = blockIdx.x; p < n_mid; p += gridDim.x) {
        const uint32_t nb = P.cnt_b[p], nt = P.cnt_t[p];
        if (nb == 0u || nt == 0u) {
            if (l == 0u) {
                P.cnt_tr[p] = 0u;
                P.cnt_s[p] = 0u;
            }
            continue;
        }
        const uint32_t mi = static_cast<uint32_t>(P.sorted[p]);
        const float mr = P.pts[p].w, mvr = sp_vr(P, mi), mvz = sp_vz(P, mi);
        const doublet_rec* B = P.bot + P.off_b[p];
        const doublet_rec* T = P.top + P.off_t[p];
        bool fits = nt <= kMidTops;
        for (uint32_t j = l; fits && j < nt; j += kWave) {
            const doublet_rec t = T[j];
            t_Er[j] = t.Er;
            t_cot[j] = t.cot;
            t_iDR[j] = t.iDR;
            S.t_U[j] = t.U;
            S.t_V[j] = t.V;
            S.t_sp[j] = t.sp;
        }
        uint32_t n = 0u;  // triplets so far
        for (uint32_t c0 = 0; fits && c0 < nb; c0 += kWave) {
            const bool has = c0 + l < nb;
            const doublet_rec own = B[has ? c0 + l : 0u];
            float own_scat2 = P.c.maxScatteringAngle2 * (1.f + own.cot * own.cot);
            own_scat2 *= ss2;
            S.b_Er[l] = own.Er;
            S.b_cot[l] = own.cot;
            S.b_iDR[l] = own.iDR;
            S.b_U[l] = own.U;
            S.b_V[l] = own.V;
            S.b_sp[l] = own.sp;
            S.b_n[l] = 0u;
            wave_lds_order();
            uint64_t left[kTopWords];
            uint32_t mine = 0u;
#pragma unroll
            for (uint32_t q = 0; q < kTopWords; ++q) {
                uint64_t m = 0ull;
                const uint32_t nq = nt > 64u * q ? (nt - 64u * q < 64u ? nt - 64u * q : 64u) : 0u;
                for (uint32_t j = 0; j < nq; j += 4u) {
                    const float4 er = S.t_Er[16u * q + j / 4u], cot = S.t_cot[16u * q + j / 4u],
                                 idr = S.t_iDR[16u * q + j / 4u];
                    uint32_t four = 0u;
                    four |= triplet_scatters(mvr, mvz, own, er.x, cot.x, idr.x, own_scat2) ? 0u : 1u;
                    four |= triplet_scatters(mvr, mvz, own, er.y, cot.y, idr.y, own_scat2) ? 0u : 2u;
                    four |= triplet_scatters(mvr, mvz, own, er.z, cot.z, idr.z, own_scat2) ? 0u : 4u;
                    four |= triplet_scatters(mvr, mvz, own, er.w, cot.w, idr.w, own_scat2) ? 0u : 8u;
                    m |= static_cast<uint64_t>(four) << j;
                }
                // the last four may reach past the tops
                m = has && nq > 0u ? m & (~0ull >> (64u - nq)) : 0ull;
                left[q] = m;
                mine += static_cast<uint32_t>(__popcll(m));
            }
            const uint32_t incl = wave_inclusive_scan(mine);
            const uint32_t pairs = wave_broadcast(incl, kWave - 1);
            if (pairs > kMidPairs) {
                fits = false;
                break;
            }
            uint32_t at = incl - mine;
#pragma unroll
            for (uint32_t q = 0; q < kTopWords; ++q) {
                for (uint64_t rest = left[q]; rest != 0ull; rest &= rest - 1ull) {
                    S.pair[at++] = static_cast<uint16_t>(l << 8 | (64u * q + static_cast<uint32_t>(__builtin_ctzll(rest))));
                }
            }
            wave_lds_order();
            const uint32_t n0 = n;
            for (uint32_t k0 = 0; k0 < pairs; k0 += kWave) {
                const bool in = k0 + l < pairs;
                const uint32_t pr = S.pair[in ? k0 + l : 0u];
                const uint32_t jb = pr >> 8, j = pr & 0xffu;
                const doublet_rec lb{0u, 0.f, S.b_cot[jb], S.b_iDR[jb], S.b_Er[jb], S.b_U[jb], S.b_V[jb]};
                const doublet_rec lt{0u, 0.f, t_cot[j], t_iDR[j], t_Er[j], S.t_U[j], S.t_V[j]};
                const float iSinTheta2 = 1.f + lb.cot * lb.cot;
                float scat2 = P.c.maxScatteringAngle2 * iSinTheta2;
                scat2 *= ss2;
                float cv = 0.f, ip = 0.f;
                const bool ok = in && triplet_ok(mr, mvr, mvz, lb, lt, P.c, iSinTheta2, scat2, cv, ip);
                const uint64_t m = wave_ballot(ok);
                const uint32_t pos = n + prefix_count(m);
                if (ok && pos < kMidTrips) {
                    S.b[pos] = S.b_sp[jb];
                    S.t[pos] = S.t_sp[j];
                    S.curv[pos] = cv;
                    S.w[pos] = -ip * f.impactWeightFactor;
                    S.rt[pos] = P.rad[S.t_sp[j]];
                    S.seg0[pos] = static_cast<uint16_t>(jb);
                    atomicAdd(&S.b_n[jb], 1u);
                }
                n += static_cast<uint32_t>(__popcll(m));
            }
            wave_lds_order();
            if (n > kMidTrips) {
                continue;  // the rest is only counted
            }
            // the bottoms' segments, and every triplet's
            const uint32_t bn = S.b_n[l];
            const uint32_t bi = wave_inclusive_scan(bn);
            for (uint32_t i0 = n0; i0 < n; i0 += kWave) {
                const bool in = i0 + l < n;
                const uint32_t jb = in ? S.seg0[i0 + l] : 0u;
                const uint32_t end = n0 + __shfl(bi, static_cast<int>(jb), kWave);
                const uint32_t len = __shfl(bn, static_cast<int>(jb), kWave);
                if (in) {
                    S.seg0[i0 + l] = static_cast<uint16_t>(end - len);
                    S.seg1[i0 + l] = static_cast<uint16_t>(end);
                }
            }
            wave_lds_order();  // the next bottoms write over these
        }
        if (!fits || n > kMidTrips) {
            const uint32_t total = fits ? n : count_triplets(P, B, T, nb, nt, mr, mvr, mvz);
            if (l == 0u) {
                P.cnt_tr[p] = total;
                P.cnt_s[p] = 0u;
            }
            continue;
        }
        // the weights, then each triplet's sort key (idx kNoSp: none, or cut)
        seed_key keys[kTripSlots];
#pragma unroll
        for (uint32_t q = 0; q < kTripSlots; ++q) {
            const uint32_t i = q * kWave + l;
            keys[q] = seed_key{0.f, 0.f, kNoSp};
            if (i >= n) continue;
            const float rt = S.rt[i];
            const float lo = S.curv[i] - f.deltaInvHelixDiameter;
            const float hi = S.curv[i] + f.deltaInvHelixDiameter;
            float compat[8];
            uint32_t nc = 0u;
            float w = S.w[i];
            const uint32_t limit = f.compatSeedLimit < 8u ? f.compatSeedLimit : 8u;
            for (uint32_t j = S.seg0[i]; j < S.seg1[i]; ++j) {
                if (j == i) continue;
                const float ro = S.rt[j];
                const float cj = S.curv[j];
                const float dr = rt - ro;
                if (fabsf(dr) < f.deltaRMin) continue;
                if (cj < lo) continue;
                if (cj > hi) continue;
                bool fresh = true;
#pragma unroll
                for (uint32_t c = 0; c < 8u; ++c) {
                    if (c < nc && fabsf(compat[c] - ro) < f.deltaRMin) fresh = false;
                }
                if (fresh) {
#pragma unroll
                    for (uint32_t c = 0; c < 8u; ++c) {
                        if (c == nc || (c == 7u && nc > 7u)) compat[c] = ro;
                    }
                    ++nc;
                    w += f.compatSeedWeight;
                }
                if (nc >= limit) break;
            }
            const uint32_t sb = S.b[i], st = S.t[i];
            const float rb = P.rad[sb];
            float bonus = 0;
            if (rb > f.good_spB_min_radius) bonus = f.good_spB_weight_increase;
            if (rt < f.good_spT_max_radius) bonus = f.good_spT_weight_increase;
            w += bonus;
            if (rb > f.good_spB_min_radius && w < f.good_spB_min_weight) continue;  // single-seed cut
            const float by = P.xyz[3 * sb + 1], bz = P.xyz[3 * sb + 2];
            const float ty = P.xyz[3 * st + 1], tz = P.xyz[3 * st + 2];
            keys[q] = seed_key{w, by * by + bz * bz + ty * ty + tz * tz, i};
        }
        uint32_t out = 0u;
        seed_key last{0.f, 0.f, 0u};
        for (uint32_t s = 0; s < max_s && s < n; ++s) {
            seed_key best{0.f, 0.f, kNoSp};
#pragma unroll
            for (uint32_t q = 0; q < kTripSlots; ++q) {
                if (keys[q].idx == kNoSp || (s > 0u && !before(last, keys[q]))) continue;  // none, or taken
                if (best.idx == kNoSp || before(keys[q], best)) best = keys[q];
            }
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {
                seed_key o;
                o.w = __shfl_xor(best.w, d, kWave);
                o.ysum = __shfl_xor(best.ysum, d, kWave);
                o.idx = __shfl_xor(best.idx, d, kWave);
                if (o.idx != kNoSp && (best.idx == kNoSp || before(o, best))) best = o;
            }
            if (best.idx == kNoSp) break;
            last = best;
            const uint32_t sb = S.b[best.idx];
            // the first is always kept; the others need a heavy seed or a far bottom
            const bool keep = s == 0u || best.w > f.seed_min_weight || P.rad[sb] > f.spB_min_radius;
            if (keep) {
                if (l == 0u) {
                    P.slots[static_cast<size_t>(p) * max_s + out] = seed_rec{sb, mi, S.t[best.idx], best.w};
                }
                ++out;
            }
        }
        if (l == 0u) {
            P.cnt_tr[p] = 0u;
            P.cnt_s[p] = out;
        }
        wave_lds_order();  // the next middle writes over this one's tables
    }
}

// seed_filtering.cpp:36-121, one middle per wave (those of k_sd_triplets).
__global__ __launch_bounds__(kSdBlock) void k_sd_filter(sd_params P) {
    const uint32_t n_mid = P.ctl->n_valid;
    const uint32_t l = lane();
    const ckf_seedfilter_config& f = P.f;
    const uint32_t max_s = P.c.maxSeedsPerSpM;
    for (uint32_t p = blockIdx.x * kSdWaves + threadIdx.x / kWave; p < n_mid; p += gridDim.x * kSdWaves) {
        const uint32_t t0 = P.off_tr[p], nt = P.cnt_tr[p];
        if (nt == 0u) {
            continue;  // k_sd_middle's
        }
        const uint32_t mi = static_cast<uint32_t>(P.sorted[p]);
        uint32_t out = 0u;
        seed_key last{0.f, 0.f, 0u};
        // the sorted passing triplets, one at a time: the best after `last`
        for (uint32_t s = 0; s < max_s && s < nt; ++s) {
            seed_key best{0.f, 0.f, kNoSp};
            for (uint32_t c0 = 0; c0 < nt; c0 += kWave) {
                const uint32_t k = c0 + l;
                if (k >= nt) continue;
                const triplet_rec r = P.trip[t0 + k];
                const float rb = P.rad[r.b], rt = P.rad[r.t];
                float bonus = 0;
                if (rb > f.good_spB_min_radius) bonus = f.good_spB_weight_increase;
                if (rt < f.good_spT_max_radius) bonus = f.good_spT_weight_increase;
                const float w = r.w + bonus;
                if (rb > f.good_spB_min_radius && w < f.good_spB_min_weight) continue;  // single-seed cut
                const float by = P.xyz[3 * r.b + 1], bz = P.xyz[3 * r.b + 2];
                const float ty = P.xyz[3 * r.t + 1], tz = P.xyz[3 * r.t + 2];
                const seed_key key{w, by * by + bz * bz + ty * ty + tz * tz, k};
                if (s > 0u && !before(last, key)) continue;  // already taken
                if (best.idx == kNoSp || before(key, best)) best = key;
            }
            // wave minimum under `before`
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) {
                seed_key o;
                o.w = __shfl_xor(best.w, d, kWave);
                o.ysum = __shfl_xor(best.ysum, d, kWave);
                o.idx = __shfl_xor(best.idx, d, kWave);
                if (o.idx != kNoSp && (best.idx == kNoSp || before(o, best))) best = o;
            }
            if (best.idx == kNoSp) break;
            last = best;
            const triplet_rec r = P.trip[t0 + best.idx];
            // the first is always kept; the others need a heavy seed or a far bottom
            const bool keep = s == 0u || best.w > f.seed_min_weight || P.rad[r.b] > f.spB_min_radius;
            if (keep) {
                if (l == 0u) P.slots[static_cast<size_t>(p) * max_s + out] = seed_rec{r.b, mi, r.t, best.w};
                ++out;
            }
        }
        if (l == 0u) P.cnt_s[p] = out;
    }
}

__global__ __launch_bounds__(kSdBlock) void k_sd_compact(sd_params P) {
    const uint32_t n_mid = P.ctl->n_valid;
    const uint32_t max_s = P.c.maxSeedsPerSpM;
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n_mid; p += gridDim.x * blockDim.x) {
        const uint32_t o = P.off_s[p];
        for (uint32_t s = 0; s < P.cnt_s[p]; ++s) P.seeds[o + s] = P.slots[static_cast<size_t>(p) * max_s + s];
    }
}

// core/include/traccc/seeding/impl/spacepoint_formation.ipp:20-48: a
// spacepoint per 2D measurement, global = centre + loc0 u + loc1 v.
__global__ __launch_bounds__(kSdBlock) void k_sd_sp_flag(const uint32_t* info, uint32_t m0, uint32_t n,
                                                         uint32_t* flag) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        flag[i] = (info[m0 + i] & 0xffu) == 2u ? 1u : 0u;
    }
}
__global__ __launch_bounds__(kSdBlock) void k_sd_sp_form(const ckf_surface* sfs, const float2* pos,
                                                         const uint32_t* meas_sf, uint32_t m0, uint32_t n,
                                                         const uint32_t* flag, const uint32_t* off,
                                                         float* xyz, uint32_t* midx) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        if (flag[i] == 0u) continue;
        const ckf_surface& S = sfs[meas_sf[m0 + i]];
        const float2 lp = pos[m0 + i];
        const uint32_t o = off[i];
        for (int k = 0; k < 3; ++k) xyz[3 * o + k] = S.center[k] + lp.x * S.axis_u[k] + lp.y * S.axis_v[k];
        midx[o] = i;
    }
}

// track_params_estimation_helper.hpp:47-125 and track_params_estimation.cpp:60-87,
// one seed per thread, in single precision as the reference.
struct tp_params {
    ckf_track_params_estimation_config cfg;
    float b[3];
    uint32_t n;
    const float* xyz;
    const uint32_t* sb;
    const uint32_t* sm;
    const uint32_t* st;
    const float* bottom_local;  // [n][2]
    float* vec;                 // [n][6]
    float* cov;                 // [n][36]
};

__device__ inline void v_sub(const float* a, const float* c, float* o) {
    for (int k = 0; k < 3; ++k) o[k] = a[k] - c[k];
}
__device__ inline void v_cross(const float* a, const float* c, float* o) {
    o[0] = a[1] * c[2] - a[2] * c[1];
    o[1] = a[2] * c[0] - a[0] * c[2];
    o[2] = a[0] * c[1] - a[1] * c[0];
}
__device__ inline float v_norm(const float* a) { return sqrtf(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]); }
__device__ inline void v_unit(float* a) {
    const float n = v_norm(a);
    for (int k = 0; k < 3; ++k) a[k] = a[k] / n;
}

__global__ __launch_bounds__(kSdBlock) void k_track_params(tp_params P) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < P.n; i += gridDim.x * blockDim.x) {
        const float* p0 = P.xyz + 3u * P.sb[i];
        const float* p1 = P.xyz + 3u * P.sm[i];
        const float* p2 = P.xyz + 3u * P.st[i];
        // frame at the bottom spacepoint: z along the field, y normal to
        // the bottom -> middle chord
        float rel[3], z[3] = {P.b[0], P.b[1], P.b[2]}, y[3], x[3];
        v_sub(p1, p0, rel);
        v_unit(z);
        v_cross(z, rel, y);
        v_unit(y);
        v_cross(y, z, x);
        float l1[3], l2[3], d[3];
        v_sub(p1, p0, d);
        l1[0] = d[0] * x[0] + d[1] * x[1] + d[2] * x[2];
        l1[1] = d[0] * y[0] + d[1] * y[1] + d[2] * y[2];
        v_sub(p2, p0, d);
        l2[0] = d[0] * x[0] + d[1] * x[1] + d[2] * x[2];
        l2[1] = d[0] * y[0] + d[1] * y[1] + d[2] * y[2];
        l2[2] = d[0] * z[0] + d[1] * z[1] + d[2] * z[2];
        // conformal map: the circle through the three points is a line v = A u + B
        const float den1 = l1[0] * l1[0] + l1[1] * l1[1];
        const float den2 = l2[0] * l2[0] + l2[1] * l2[1];
        const float u1 = l1[0] / den1, v1 = l1[1] / den1, u2 = l2[0] / den2, v2 = l2[1] / den2;
        const float A = (v2 - v1) / (u2 - u1);
        const float B = v2 - A * u2;
        const float R = -sqrtf(1.f + A * A) / (2.f * B);
        const float perp2 = sqrtf(l2[0] * l2[0] + l2[1] * l2[1]);
        const float invTanTheta = l2[2] / (2.f * R * asinf(perp2 / (2.f * R)));
        float td[3] = {1.f, A, sqrtf(1.f + A * A) * invTanTheta};
        v_unit(td);
        const float dir[3] = {x[0] * td[0] + y[0] * td[1] + z[0] * td[2], x[1] * td[0] + y[1] * td[1] + z[1] * td[2],
                              x[2] * td[0] + y[2] * td[1] + z[2] * td[2]};
        float* v = P.vec + 6 * static_cast<size_t>(i);
        v[0] = P.bottom_local[2 * i];
        v[1] = P.bottom_local[2 * i + 1];
        v[2] = atan2f(dir[1], dir[0]);
        v[3] = atan2f(sqrtf(dir[0] * dir[0] + dir[1] * dir[1]), dir[2]);
        const float qOverPt = 1.f / (R * v_norm(P.b));
        v[4] = qOverPt / sqrtf(1.f + invTanTheta * invTanTheta);
        v[5] = 0.f;
        float* C = P.cov + 36 * static_cast<size_t>(i);
        for (int k = 0; k < 36; ++k) C[k] = 0.f;
        for (int j = 0; j < 6; ++j) {
            float var = P.cfg.initial_sigma[j] * P.cfg.initial_sigma[j];
            if (j == 4) {
                const float vt = C[3 * 6 + 3];
                const float a = P.cfg.initial_sigma_qopt * sinf(v[3]);
                const float b = P.cfg.initial_sigma_pt_rel * v[4];
                const float c = v[4] / tanf(v[3]);
                var += a * a;
                var += b * b;
                var += vt * (c * c);
            }
            var *= P.cfg.initial_inflation[j];
            C[j * 6 + j] = var;
        }
    }
}

uint32_t grid_for(uint64_t items, uint32_t per_block) {
    const uint64_t b = (items + per_block - 1u) / per_block;
    return static_cast<uint32_t>(std::max<uint64_t>(1u, std::min<uint64_t>(b, 65536u)));
}

// spacepoint_binning_helper.hpp:22-108; false where the reference throws
bool make_axes(const ckf_spacepoint_grid_config& g, sd_axes& A, std::string& why) {
    uint32_t phiBins;
    if (g.bFieldInZ == 0.f) {
        phiBins = 100u;
    } else {
        const float minHelixRadius = g.minPt / g.bFieldInZ;
        if (minHelixRadius < g.rMax / 2) {
            why = "the minimum helix radius (minPt / bFieldInZ) is smaller than rMax / 2";
            return false;
        }
        const float maxR2 = g.rMax * g.rMax;
        const float xOuter = maxR2 / (2 * minHelixRadius);
        const float yOuter = std::sqrt(maxR2 - xOuter * xOuter);
        const float outerAngle = std::atan(xOuter / yOuter);
        float innerAngle = 0;
        float rMin = g.rMax;
        if (g.rMax > g.deltaRMax) {
            rMin = g.rMax - g.deltaRMax;
            const float innerCircleR2 = (g.rMax - g.deltaRMax) * (g.rMax - g.deltaRMax);
            const float xInner = innerCircleR2 / (2 * minHelixRadius);
            const float yInner = std::sqrt(innerCircleR2 - xInner * xInner);
            innerAngle = std::atan(xInner / yInner);
        }
        const float deltaAngleWithMaxD0 = std::fabs(std::asin(g.impactMax / (rMin)) - std::asin(g.impactMax / g.rMax));
        const float deltaPhi =
            (outerAngle - innerAngle + deltaAngleWithMaxD0) / static_cast<float>(g.phiBinDeflectionCoverage);
        if (deltaPhi <= 0.) {
            why = "the phi bin width is not positive";
            return false;
        }
        phiBins = static_cast<uint32_t>(std::llround(2 * M_PI / deltaPhi + 0.5));
    }
    const float zBinSize = g.cotThetaMax * g.deltaRMax;
    const uint32_t zBins = std::max(1u, static_cast<uint32_t>(std::floor((g.zMax - g.zMin) / zBinSize)));
    A = sd_axes{phiBins, zBins, g.phiMin, g.phiMax, g.zMin, g.zMax};
    return true;
}

}  // namespace
}  // namespace tamd

using tamd::ckf_error;
using tamd::guarded;
using tamd::hip_check;

struct ckf_seeding {
    ckf_seedfinder_config finder{};
    ckf_spacepoint_grid_config grid{};
    ckf_seedfilter_config filter{};
    tamd::sd_axes axes{};
    hipStream_t stream = nullptr;
    uint32_t n_seeds = 0;
    int device = 0;  // where the seeds of the last run are
    tamd::dbuf in_xyz, in_vr, in_vz, rad, phi, keys, sorted, sort_tmp, pts, bin_off, cnt_b, off_b,
        cnt_t, off_t, bot, top, cnt_tr, off_tr, trip, cnt_s, off_s, slots, seeds, sums, ctl;
    tamd::sd_ctl* h_ctl = nullptr;
    ~ckf_seeding() {
        tamd::dbuf* bs[] = {&in_xyz, &in_vr,  &in_vz,  &rad,   &phi,    &keys,  &sorted, &sort_tmp, &pts,
                            &bin_off, &cnt_b, &off_b,  &cnt_t, &off_t,  &bot,   &top,    &cnt_tr,   &off_tr,
                            &trip,   &cnt_s,  &off_s,  &slots, &seeds,  &sums,  &ctl};
        for (tamd::dbuf* b : bs) b->release();
        if (h_ctl != nullptr) (void)hipHostFree(h_ctl);
    }
};

namespace {

void read_ctl(ckf_seeding& S) {
    hip_check(hipMemcpyAsync(S.h_ctl, S.ctl.p, sizeof(tamd::sd_ctl), hipMemcpyDeviceToHost, S.stream), "readback");
    hip_check(hipStreamSynchronize(S.stream), "seeding");
}

void run_seeding(ckf_seeding& S, uint32_t n_sp, const float* d_xyz, const float* d_vr, const float* d_vz) {
    using namespace tamd;
    const hipStream_t s = S.stream;
    S.device = current_device();
    const uint32_t nbins = S.axes.nphi * S.axes.nz;
    const uint32_t N = std::max(n_sp, 1u);
    S.rad.ensure(4u * size_t(N));
    S.phi.ensure(4u * size_t(N));
    S.keys.ensure(8u * size_t(N));
    S.sorted.ensure(8u * size_t(N));
    S.pts.ensure(16u * size_t(N));
    S.bin_off.ensure(4u * (size_t(nbins) + 1u));
    S.sums.ensure(4u * size_t(scan_sums_size(N + 1u)));
    S.ctl.ensure(sizeof(sd_ctl));
    if (S.h_ctl == nullptr) {
        hip_check(hipHostMalloc(reinterpret_cast<void**>(&S.h_ctl), sizeof(sd_ctl)), "hipHostMalloc");
    }
    hip_check(hipMemsetAsync(S.ctl.p, 0, sizeof(sd_ctl), s), "memset");
    sd_params P{};
    P.c = S.finder;
    P.f = S.filter;
    P.A = S.axes;
    P.n_sp = n_sp;
    P.xyz = d_xyz;
    P.vr = d_vr;
    P.vz = d_vz;
    P.rad = S.rad.as<float>();
    P.phi = S.phi.as<float>();
    P.keys = S.keys.as<uint64_t>();
    P.sorted = S.sorted.as<uint64_t>();
    P.pts = S.pts.as<float4>();
    P.bin_off = S.bin_off.as<uint32_t>();
    P.nbins = nbins;
    P.ctl = S.ctl.as<sd_ctl>();
    if (n_sp > 0u) {
        hipLaunchKernelGGL(k_sd_prep, dim3(grid_for(n_sp, kSdBlock)), dim3(kSdBlock), 0, s, P);
        hip_check(hipGetLastError(), "prep");
        // (bin << 32 | index): the bits above the largest bin are zero
        int end_bit = 32;
        while (end_bit < 64 && (uint64_t(1) << (end_bit - 32)) <= nbins) ++end_bit;
        end_bit = 64;  // invalid spacepoints carry all-ones keys
        size_t tmp = 0;
        hip_check(rocprim::radix_sort_keys(nullptr, tmp, P.keys, const_cast<uint64_t*>(P.sorted), n_sp, 0,
                                           end_bit, s),
                  "sort size");
        S.sort_tmp.ensure(std::max<size_t>(tmp, 256));
        hip_check(rocprim::radix_sort_keys(S.sort_tmp.p, tmp, P.keys, const_cast<uint64_t*>(P.sorted), n_sp, 0,
                                           end_bit, s),
                  "sort");
    }
    if (n_sp > 0u) {
        hipLaunchKernelGGL(k_sd_place, dim3(grid_for(n_sp, kSdBlock)), dim3(kSdBlock), 0, s, P);
        hip_check(hipGetLastError(), "place");
    }
    read_ctl(S);
    const uint32_t nm = S.h_ctl->n_valid;
    const uint32_t M = std::max(nm, 1u);
    S.cnt_b.ensure(4u * size_t(M));
    S.off_b.ensure(4u * (size_t(M) + 1u));
    S.cnt_t.ensure(4u * size_t(M));
    S.off_t.ensure(4u * (size_t(M) + 1u));
    S.cnt_tr.ensure(4u * size_t(M));
    S.off_tr.ensure(4u * (size_t(M) + 1u));
    S.cnt_s.ensure(4u * size_t(M));
    S.off_s.ensure(4u * (size_t(M) + 1u));
    S.slots.ensure(sizeof(seed_rec) * size_t(M) * std::max(S.finder.maxSeedsPerSpM, 1u));
    S.sums.ensure(4u * size_t(scan_sums_size(M + 1u)));
    P.cnt_b = S.cnt_b.as<uint32_t>();
    P.off_b = S.off_b.as<uint32_t>();
    P.cnt_t = S.cnt_t.as<uint32_t>();
    P.off_t = S.off_t.as<uint32_t>();
    P.cnt_tr = S.cnt_tr.as<uint32_t>();
    P.off_tr = S.off_tr.as<uint32_t>();
    P.cnt_s = S.cnt_s.as<uint32_t>();
    P.off_s = S.off_s.as<uint32_t>();
    P.slots = S.slots.as<seed_rec>();
    const dim3 gw(grid_for(nm, kSdWaves));
    if (nm > 0u) {
        hipLaunchKernelGGL(k_sd_doublets<false>, gw, dim3(kSdBlock), 0, s, P);
        hip_check(hipGetLastError(), "doublet count");
    }
    exclusive_scan(P.cnt_b, P.off_b, S.sums.as<uint32_t>(), nm, &P.ctl->n_bot, s);
    exclusive_scan(P.cnt_t, P.off_t, S.sums.as<uint32_t>(), nm, &P.ctl->n_top, s);
    read_ctl(S);
    S.bot.ensure(sizeof(doublet_rec) * std::max<size_t>(S.h_ctl->n_bot, 1u));
    S.top.ensure(sizeof(doublet_rec) * std::max<size_t>(S.h_ctl->n_top, 1u));
    P.bot = S.bot.as<doublet_rec>();
    P.top = S.top.as<doublet_rec>();
    if (nm > 0u) {
        hipLaunchKernelGGL(k_sd_doublets<true>, gw, dim3(kSdBlock), 0, s, P);
        hipLaunchKernelGGL(k_sd_middle, dim3(std::min(nm, 1u << 20)), dim3(kWave), 0, s, P);
        hip_check(hipGetLastError(), "triplets");
    }
    exclusive_scan(P.cnt_tr, P.off_tr, S.sums.as<uint32_t>(), nm, &P.ctl->n_trip, s);
    read_ctl(S);
    if (S.h_ctl->n_trip > 0u) {
        // the middles with more tops or triplets than LDS holds
        S.trip.ensure(sizeof(triplet_rec) * size_t(S.h_ctl->n_trip));
        P.trip = S.trip.as<triplet_rec>();
        hipLaunchKernelGGL(k_sd_triplets, gw, dim3(kSdBlock), 0, s, P);
        hipLaunchKernelGGL(k_sd_weights, dim3(grid_for(S.h_ctl->n_trip, kSdBlock)), dim3(kSdBlock), 0, s, P);
        hipLaunchKernelGGL(k_sd_filter, gw, dim3(kSdBlock), 0, s, P);
        hip_check(hipGetLastError(), "filter");
    }
    exclusive_scan(P.cnt_s, P.off_s, S.sums.as<uint32_t>(), nm, &P.ctl->n_seeds, s);
    read_ctl(S);
    S.n_seeds = S.h_ctl->n_seeds;
    S.seeds.ensure(sizeof(seed_rec) * std::max<size_t>(S.n_seeds, 1u));
    P.seeds = S.seeds.as<seed_rec>();
    if (nm > 0u) {
        hipLaunchKernelGGL(k_sd_compact, dim3(grid_for(nm, kSdBlock)), dim3(kSdBlock), 0, s, P);
        hip_check(hipGetLastError(), "compact");
    }
    hip_check(hipStreamSynchronize(s), "seeding");
}

}  // namespace

extern "C" {

ckf_status ckf_seeding_create(const ckf_seedfinder_config* finder, const ckf_spacepoint_grid_config* grid,
                              const ckf_seedfilter_config* filter, ckf_seeding** out) {
    return guarded([&] {
        if (!finder || !grid || !filter || !out) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "null argument");
        tamd::sd_axes A{};
        std::string why;
        if (!tamd::make_axes(*grid, A, why)) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, why);
        if (finder->maxSeedsPerSpM == 0u) {
            throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "maxSeedsPerSpM must be at least 1");
        }
        if (filter->compatSeedLimit > 8u) {
            throw ckf_error(CKF_ERR_UNSUPPORTED, "compatSeedLimit above 8 is not supported");
        }
        if (uint64_t(A.nphi) * A.nz > 0xfffffff0ull) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "too many grid bins");
        auto* s = new ckf_seeding();
        s->finder = *finder;
        s->grid = *grid;
        s->filter = *filter;
        s->axes = A;
        *out = s;
    });
}

ckf_status ckf_seeding_destroy(ckf_seeding* s) {
    return guarded([&] { delete s; });
}

ckf_status ckf_seeding_set_stream(ckf_seeding* s, void* hip_stream) {
    return guarded([&] {
        if (s == nullptr) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "null seeding");
        s->stream = static_cast<hipStream_t>(hip_stream);
    });
}

ckf_status ckf_seeding_run(ckf_seeding* s, const ckf_spacepoints* sp, uint32_t* n_seeds) {
    return guarded([&] {
        if (s == nullptr || sp == nullptr || (sp->size > 0u && sp->global == nullptr)) {
            throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "null argument");
        }
        const uint32_t n = sp->size;
        const size_t N = std::max<size_t>(n, 1u);
        s->in_xyz.ensure(12u * N);
        if (n > 0u) {
            hip_check(hipMemcpyAsync(s->in_xyz.p, sp->global, 12u * size_t(n), hipMemcpyHostToDevice, s->stream),
                      "upload");
        }
        const float* vr = nullptr;
        const float* vz = nullptr;
        if (sp->radius_variance != nullptr && n > 0u) {
            s->in_vr.ensure(4u * N);
            hip_check(hipMemcpyAsync(s->in_vr.p, sp->radius_variance, 4u * size_t(n), hipMemcpyHostToDevice,
                                     s->stream), "upload");
            vr = s->in_vr.as<float>();
        }
        if (sp->z_variance != nullptr && n > 0u) {
            s->in_vz.ensure(4u * N);
            hip_check(hipMemcpyAsync(s->in_vz.p, sp->z_variance, 4u * size_t(n), hipMemcpyHostToDevice, s->stream),
                      "upload");
            vz = s->in_vz.as<float>();
        }
        run_seeding(*s, n, s->in_xyz.as<float>(), vr, vz);
        if (n_seeds) *n_seeds = s->n_seeds;
    });
}

ckf_status ckf_seeding_run_device(ckf_seeding* s, const ckf_spacepoints* sp, uint32_t* n_seeds) {
    return guarded([&] {
        if (s == nullptr || sp == nullptr || (sp->size > 0u && sp->global == nullptr)) {
            throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "null argument");
        }
        run_seeding(*s, sp->size, sp->global, sp->radius_variance, sp->z_variance);
        if (n_seeds) *n_seeds = s->n_seeds;
    });
}

ckf_status ckf_seeding_result_size(const ckf_seeding* s, uint32_t* n_seeds) {
    return guarded([&] {
        if (s == nullptr || n_seeds == nullptr) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "null argument");
        *n_seeds = s->n_seeds;
    });
}

ckf_status ckf_seeding_result_download(const ckf_seeding* s, ckf_seeds* out) {
    return guarded([&] {
        if (s == nullptr || out == nullptr) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "null argument");
        if (out->size < s->n_seeds) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "output smaller than the seeds");
        static_assert(sizeof(tamd::seed_rec) == 16u, "a seed is four words: bottom, middle, top, weight");
        tamd::readback rb(s->device);
        rb.words(out->bottom, s->seeds.p, s->n_seeds, 4u, 0u, 1u);
        rb.words(out->middle, s->seeds.p, s->n_seeds, 4u, 1u, 1u);
        rb.words(out->top, s->seeds.p, s->n_seeds, 4u, 2u, 1u);
        rb.words(out->weight, s->seeds.p, s->n_seeds, 4u, 3u, 1u);
        rb.run();
    });
}

ckf_status ckf_spacepoint_formation(const ckf_device_detector* det, const ckf_device_event* ev, uint32_t event,
                                    float* global, uint32_t* measurement_index, uint32_t* n) {
    return guarded([&] {
        if (det == nullptr || ev == nullptr || n == nullptr) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "null argument");
        if (event >= ev->n_events) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "event index out of range");
        if (ev->n_surfaces != det->h_sfs.size()) {
            throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "events and detector do not match");
        }
        const uint32_t m0 = ev->meas_off[event], nm = ev->meas_off[event + 1] - m0;
        const hipStream_t s = nullptr;
        const int device = tamd::current_device();
        tamd::rbuf flag, off, sums, d_total, xyz, midx;
        const uint32_t N = std::max(nm, 1u);
        flag.take(4u * size_t(N), device);
        off.take(4u * (size_t(N) + 1u), device);
        sums.take(4u * size_t(tamd::scan_sums_size(N)), device);
        d_total.take(4u, device);
        const tamd::staging_block h_total(4u);
        try {
            if (nm > 0u) {
                hipLaunchKernelGGL(tamd::k_sd_sp_flag, dim3(tamd::grid_for(nm, tamd::kSdBlock)), dim3(tamd::kSdBlock),
                                   0, s, ev->d_info, m0, nm, flag.as<uint32_t>());
                hip_check(hipGetLastError(), "spacepoint flags");
            }
            tamd::exclusive_scan(flag.as<uint32_t>(), off.as<uint32_t>(), sums.as<uint32_t>(), nm,
                                 d_total.as<uint32_t>(), s);
            hip_check(hipMemcpyAsync(h_total.p, d_total.p, 4u, hipMemcpyDeviceToHost, s), "readback");
            hip_check(hipStreamSynchronize(s), "readback");
            const uint32_t total = *static_cast<const uint32_t*>(h_total.p);
            *n = total;
            if ((global != nullptr || measurement_index != nullptr) && total > 0u) {
                xyz.take(12u * size_t(total), device);
                midx.take(4u * size_t(total), device);
                hipLaunchKernelGGL(tamd::k_sd_sp_form, dim3(tamd::grid_for(nm, tamd::kSdBlock)), dim3(tamd::kSdBlock), 0,
                                   s, det->d_sfs, ev->d_pos, ev->d_meas_sf, m0, nm, flag.as<uint32_t>(),
                                   off.as<uint32_t>(), xyz.as<float>(), midx.as<uint32_t>());
                hip_check(hipGetLastError(), "spacepoints");
                tamd::readback rb(device);
                rb.bytes(global, xyz.p, 12u * size_t(total));
                rb.bytes(measurement_index, midx.p, 4u * size_t(total));
                rb.run();
            }
        } catch (...) {
            (void)hipStreamSynchronize(s);  // the blocks may be handed out again
            throw;
        }
    });
}

ckf_status ckf_estimate_track_params(const ckf_track_params_estimation_config* cfg, const ckf_spacepoints* sp,
                                     const ckf_seeds* seeds, const ckf_measurements* meas, const float bfield[3],
                                     uint64_t* surface_link, float* vector, float* covariance) {
    return guarded([&] {
        if (!cfg || !sp || !seeds || !meas || !bfield) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "null argument");
        const uint32_t n = seeds->size;
        if (n == 0u) return;
        if (!seeds->bottom || !seeds->middle || !seeds->top || !sp->global || !sp->measurement_index_1 ||
            !meas->local_position || !meas->surface_link) {
            throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "null seed, spacepoint or measurement arrays");
        }
        // What the kernel needs, in one device block: the seeds' indices, the
        // bottom spacepoint's local position (gathered here, with its surface)
        // and the spacepoints.  One pinned block holds it on the host: a copy from
        // the caller's own arrays would cost 10 to 100 us each, for the same
        // reasons as on the way back.  Past the largest pinned block the copies are
        // the lesser cost (3 million seeds: 52 ms with a block of 128 MiB pinned
        // for the call, 42 with four copies and column by column back).
        const size_t np = sp->size, in_bytes = 20u * size_t(n) + 12u * np;
        const bool staged = in_bytes <= tamd::pinned_cache::kMaxBlock;
        const tamd::staging_block h_in(staged ? in_bytes : 8u * size_t(n));
        uint32_t* const hi = static_cast<uint32_t*>(h_in.p);
        float* const hb = reinterpret_cast<float*>(hi + (staged ? 3u * size_t(n) : 0u));
        for (uint32_t i = 0; i < n; ++i) {
            const uint32_t b = seeds->bottom[i];
            if (b >= np || seeds->middle[i] >= np || seeds->top[i] >= np) {
                throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "seed spacepoint index out of range");
            }
            const uint32_t m = sp->measurement_index_1[b];
            if (m >= meas->size) throw ckf_error(CKF_ERR_INVALID_ARGUMENT, "spacepoint measurement index out of range");
            hb[2u * size_t(i)] = meas->local_position[2u * size_t(m)];
            hb[2u * size_t(i) + 1u] = meas->local_position[2u * size_t(m) + 1u];
            if (surface_link) surface_link[i] = meas->surface_link[m];
        }
        if (staged) {
            std::memcpy(hi, seeds->bottom, 4u * size_t(n));
            std::memcpy(hi + n, seeds->middle, 4u * size_t(n));
            std::memcpy(hi + 2u * size_t(n), seeds->top, 4u * size_t(n));
            std::memcpy(hb + 2u * size_t(n), sp->global, 12u * np);
        }
        const int device = tamd::current_device();
        tamd::rbuf d_in, d_vec, d_cov;
        d_in.take(in_bytes, device);
        d_vec.take(24u * size_t(n), device);
        d_cov.take(144u * size_t(n), device);
        try {
            uint32_t* const di = d_in.as<uint32_t>();
            if (staged) {
                hip_check(hipMemcpyAsync(di, h_in.p, in_bytes, hipMemcpyHostToDevice, nullptr), "upload");
            } else {
                hip_check(hipMemcpy(di, seeds->bottom, 4u * size_t(n), hipMemcpyHostToDevice), "upload");
                hip_check(hipMemcpy(di + n, seeds->middle, 4u * size_t(n), hipMemcpyHostToDevice), "upload");
                hip_check(hipMemcpy(di + 2u * size_t(n), seeds->top, 4u * size_t(n), hipMemcpyHostToDevice), "upload");
                hip_check(hipMemcpy(di + 3u * size_t(n), hb, 8u * size_t(n), hipMemcpyHostToDevice), "upload");
                hip_check(hipMemcpy(di + 5u * size_t(n), sp->global, 12u * np, hipMemcpyHostToDevice), "upload");
            }
            tamd::tp_params P{};
            P.cfg = *cfg;
            for (int k = 0; k < 3; ++k) P.b[k] = bfield[k];
            P.n = n;
            P.sb = di;
            P.sm = di + n;
            P.st = di + 2u * size_t(n);
            P.bottom_local = d_in.as<float>() + 3u * size_t(n);
            P.xyz = P.bottom_local + 2u * size_t(n);
            P.vec = d_vec.as<float>();
            P.cov = d_cov.as<float>();
            hipLaunchKernelGGL(tamd::k_track_params, dim3(tamd::grid_for(n, tamd::kSdBlock)), dim3(tamd::kSdBlock), 0,
                               nullptr, P);
            hip_check(hipGetLastError(), "track parameters");
            tamd::readback rb(device);
            rb.bytes(vector, d_vec.p, 24u * size_t(n));
            rb.bytes(covariance, d_cov.p, 144u * size_t(n));
            rb.run();
            hip_check(hipStreamSynchronize(nullptr), "track parameters");
        } catch (...) {
            (void)hipStreamSynchronize(nullptr);  // the blocks may be handed out again
            throw;
        }
    });
}

}  // extern "C"
