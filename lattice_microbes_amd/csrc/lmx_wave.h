// Reactions of a wave's sites, shared by the boxed step's reaction launch and
// the resident runs: a lane per site sums propensities (packed_propensity), and
// a site that reacts is taken by the whole wave (wave_products), a slot per
// lane to count and evaluate, a reaction per lane to select.  Loops over slots
// are rolled, so that sites of 16 slots cost no more registers than those of
// four.
#pragma once

#include "lmx_device.h"

namespace lmx {

__device__ inline uint32_t lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }

__device__ inline uint32_t lane_of(uint32_t v, uint32_t src)
{
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)src);
}

// total_propensity's sum for a site of `count` particles in its first slots:
// the same terms in the same order, a row of up to 8 pairs loaded at a time.
// slots: the wave's copy of its sites' slots, slot-major, for this lane (a
// slot's index is not known at compile time).
template <uint32_t P, class Slot>
__device__ inline float packed_propensity(const Params &p, uint32_t st, const Slot (*slots)[64], uint32_t lane,
                                          uint32_t count)
{
    constexpr uint32_t kRow = P < 8u ? P : 8u;
    float a = p.qp0[st];
#pragma unroll 1
    for (uint32_t m = 0; m < count; m++) {
        const uint32_t row = st * p.nS + slots[m][lane] - 1u;
        const float one = p.qp1[row];
        const float *pairs = p.qp2 + (size_t)row * p.nS;
        uint32_t n = m + 1u;
        float v[kRow];
        auto load = [&] {
#pragma unroll
            for (uint32_t k = 0; k < kRow; k++) {
                const uint32_t q = n + k < count ? n + k : m;
                v[k] = pairs[slots[q][lane] - 1u];
            }
        };
        load();
        a += one;
#pragma unroll 1
        for (;;) {
#pragma unroll
            for (uint32_t k = 0; k < kRow; k++)
                if (n + k < count) a += v[k];
            n += kRow;
            if (n >= count) break;
            load();
        }
    }
    return a;
}

// Which reaction happens at site si (type sst, total propensity a) and the
// particles it leaves: lane j < P holds slot j before (mine; the site's first
// slots) and after (the result).  Products without a slot are recorded as
// overflow entries; underflow tells that a reactant was not present.  Every
// lane of the wave calls it.
template <uint32_t P>
__device__ inline uint32_t wave_products(const Params &p, uint32_t si, uint32_t sst, uint32_t mine, float a,
                                         unsigned long long h3, bool &underflow)
{
    constexpr uint32_t kNone = 0xFFFFFFFFu;
    const uint32_t lane = lane_id();
    uint32_t earlier = 0;  // of the same species
#pragma unroll 1
    for (uint32_t q = 0; q < P; q++) earlier += q < lane && lane_of(mine, q) == mine ? 1u : 0u;
    // determineReactionIndex (byte_reaction_dev.cu:146-177): the reactions in
    // ascending index, each with a positive propensity moving rp, among those
    // listed under a species of the site (lane j: of slot j, if it is the
    // first of its kind) and the zero-order ones (lane P).
    uint32_t start = 0, len = 0;
    if (lane == P || (mine != 0u && earlier == 0u)) {
        const uint32_t bucket = lane == P ? p.nS : mine - 1u;
        start = p.rx_off[bucket];
        len = p.rx_off[bucket + 1] - start;
    }
    uint32_t total = 0;
#pragma unroll 1
    for (uint32_t j = 0; j <= P; j++) total += lane_of(len, j);
    float rp = uniform01(si, 1, 1, h3) * a;
    uint32_t idx = 0, r = kNone, s0 = p.sto_off[0], s1 = p.sto_off[1], k0 = s0, k1 = s1;
    float pr = 0.0f;
    bool any = false;
    while (rp > 0.0f) {
        uint32_t br = kNone;  // this lane's lowest reaction above idx, and its propensity
        float bp = 0.0f;
        uint32_t bs0 = 0, bs1 = 0;
#pragma unroll 1
        for (uint32_t c = 0; c < total; c += 64u) {
            if (!any || total > 64u) {  // one a lane is evaluated once and kept
                uint32_t left = c + lane, at = kNone;
#pragma unroll 1
                for (uint32_t j = 0; j <= P; j++) {
                    const uint32_t lj = lane_of(len, j), sj = lane_of(start, j);
                    if (left < lj) at = sj + left;
                    left = left < lj ? kNone : left - lj;
                }
                if (c + lane >= total) at = kNone;
                r = kNone;
                if (at != kNone) {
                    r = p.rx_list[at];
                    const bool here = p.RL[r * p.nST + sst] != 0;
                    const uint32_t d1 = p.D1[r], d2 = p.D2[r], order = p.order[r];
                    const float k = p.rate[r];
                    s0 = p.sto_off[r];
                    s1 = p.sto_off[r + 1];
                    float n1 = 0.0f, n2 = 0.0f;
#pragma unroll 1
                    for (uint32_t q = 0; q < P; q++) {
                        const uint32_t s = lane_of(mine, q);
                        n1 += s && s == d1 ? 1.0f : 0.0f;
                        n2 += s && s == d2 ? 1.0f : 0.0f;
                    }
                    // (reaction_propensity's expressions)
                    pr = order == kZeroOrder ? k
                         : order == kFirstOrder ? k * n1
                         : order == kSecondOrder ? k * n1 * n2
                         : order == kSecondOrderSelf ? k * n1 * (n1 - 1.0f) : 0.0f;
                    if (!here || !(pr > 0.0f)) r = kNone;
                }
            }
            if (r != kNone && (!any || r > idx) && r < br) {
                br = r;
                bp = pr;
                bs0 = s0;
                bs1 = s1;
            }
        }
        uint32_t low = kNone;
#pragma unroll 1
        for (unsigned long long m = __ballot(br != kNone); m; m &= m - 1) {
            const uint32_t v = lane_of(br, (uint32_t)__builtin_ctzll(m));
            low = v < low ? v : low;
        }
        if (low == kNone) break;
        const uint32_t who = (uint32_t)__builtin_ctzll(__ballot(br == low));
        rp -= __uint_as_float(lane_of(__float_as_uint(bp), who));
        k0 = lane_of(bs0, who);
        k1 = lane_of(bs1, who);
        idx = low;
        any = true;
    }
    // evaluateReaction (:179-257): the m-th particle of species s is consumed
    // iff fewer than -S[s] earlier ones of s were seen, the others move up,
    // and the products follow in species order.  A reactant that was not
    // present leaves a negative residue, which the reference turns into an
    // unbounded loop.
    // Lane k holds the row's k-th nonzero entry (64 of them at a time).
    uint32_t row_s = 0;
    int row_v = 0;
    auto row = [&](uint32_t c) {
        row_s = 0;
        row_v = 0;
        if (c + lane < k1) {
            row_s = p.sto_sp[c + lane] + 1u;
            row_v = p.sto_val[c + lane];
        }
    };
    row(k0);
    int change = 0;
    underflow = false;
#pragma unroll 1
    for (uint32_t k = k0; k < k1; k++) {
        if (k != k0 && ((k - k0) & 63u) == 0u) row(k);
        const uint32_t s = lane_of(row_s, (k - k0) & 63u);
        const int v = (int)lane_of((uint32_t)row_v, (k - k0) & 63u);
        if (mine == s) change = v;
        if (v < 0 && (int)__popcll(__ballot(mine == s)) < -v) underflow = true;
    }
    if (k1 - k0 > 64u) row(k0);
    const bool stays = mine != 0u && (change >= 0 || (int)earlier >= -change);
    const unsigned long long kept = __ballot(stays);
    uint32_t n = (uint32_t)__popcll(kept);
    const uint32_t to = stays ? __builtin_amdgcn_mbcnt_hi((uint32_t)(kept >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)kept, 0u))
                              : 32u + (lane & 31u);  // (beyond the site)
    uint32_t now = (uint32_t)__builtin_amdgcn_ds_permute((int)(to << 2), (int)mine);
    if (lane >= n) now = 0u;
#pragma unroll 1
    for (uint32_t k = k0; k < k1; k++) {
        if (k != k0 && ((k - k0) & 63u) == 0u) row(k);
        const uint32_t s = lane_of(row_s, (k - k0) & 63u);
#pragma unroll 1
        for (int v = (int)lane_of((uint32_t)row_v, (k - k0) & 63u); v > 0; v--, n++) {
            if (n < P) now = lane == n ? s : now;
            else if (lane == 0u) record_overflow(p.ctl, 3, si, n - P, s);
        }
    }
    return now;
}

}  // namespace lmx
