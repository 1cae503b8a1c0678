// Overflow resolution on the device, shared by the resolver kernels, the boxed
// step's reaction launch, whose last block resolves, and the resident runs,
// which resolve among a block's records.
#pragma once

#include "lmx_device.h"

namespace lmx {

// ---------------------------------------------------------------------------
// Overflow resolution: one workgroup.  Entries are sorted into canonical
// order (phase, site, emission) and placed in that order, each into the first
// site of the reference's candidate list (Lattice::getNearbySites,
// Lattice.cpp:106-128: radius 0..4, shell max(R-1,0)^2 < d^2 <= R^2, x outer,
// z inner) with room and the origin's site type.  The step counter advances
// at the end.
//
// What it costs is the latency of the searches, so every wave searches for an
// entry of its own, a lane per candidate in list order (the first 64
// candidates, radius 2 and a third of radius 3, nearly always suffice).  They
// are committed in order: particles only fill sites, so a search made before
// the earlier entries of its round were placed is still right unless they
// filled the very site it found; from the first such entry on the round is
// searched again.
// ---------------------------------------------------------------------------
__device__ inline uint32_t load_agent(const uint32_t *ptr)
{
    return __hip_atomic_load(ptr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline void store_agent(uint32_t *ptr, uint32_t v)
{
    __hip_atomic_store(ptr, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Particles up to the first empty slot (Lattice::getOccupancy).
__device__ inline uint32_t site_occupancy(const Params &p, const uint32_t *lat, uint32_t s)
{
    uint32_t occ = 0;
    for (uint32_t k = 0; k < p.W; k++) {
        const uint32_t word = load_agent(lat + (size_t)k * p.N + s);
        if (p.word_particles) {
            if (word == 0) return occ;
            occ++;
            continue;
        }
        for (uint32_t b = 0; b < 4; b++) {
            if (((word >> (8 * b)) & 0xFFu) == 0) return occ;
            occ++;
        }
    }
    return occ;
}

__device__ inline void set_error(Control *ctl, uint32_t code, uint32_t step)
{
    if (atomicCAS(&ctl->error, 0u, code) == 0u) ctl->error_step = step;
}

constexpr int kResolveThreads = 256;
constexpr uint32_t kBallSites = 257u;  // candidates of all radii
constexpr int kBallLoads = 5;           // of 64 each

// The candidates' offsets in list order: dx + 4, dy + 4, dz + 4 and the radius,
// four bits each.
struct Ball {
    uint32_t v[kBallLoads * 64];
};
constexpr Ball make_ball()
{
    Ball b{};
    uint32_t n = 0;
    for (int R = 0; R <= (int)kMaxReplacementDist; R++)
        for (int q = 0; q < 729; q++) {
            const int dx = q / 81 - 4, dy = q / 9 % 9 - 4, dz = q % 9 - 4, r2 = dx * dx + dy * dy + dz * dz;
            if (R == 0 ? r2 == 0 : (r2 > (R - 1) * (R - 1) && r2 <= R * R))
                b.v[n++] = (uint32_t)(dx + 4) | (uint32_t)(dy + 4) << 4 | (uint32_t)(dz + 4) << 8 | (uint32_t)R << 12;
        }
    return b;
}
static __constant__ const Ball kBall = make_ball();

// LDS of the resolver's block beside the sorted keys.
template <int kThreads>
struct ResolveLds {
    static constexpr int kRound = kThreads / 64;  // entries searched at once
    uint32_t parts[64], f_site[kRound], f_slot[kRound], f_room[kRound], placed, failure;
};

// What the resolver looks up and changes: the sites of a lattice in device
// memory.
struct LatticeSites {
    const Params &p;
    uint32_t *lat;

    // The first empty slot of site s | the empty slots in a row from there << 8.
    __device__ inline uint32_t look(bool in, uint32_t s) const
    {
        const uint32_t slots = p.word_particles ? 1u : 4u;
        uint32_t slot = 0, room = 0;
#pragma unroll 1
        for (uint32_t k0 = 0; k0 < p.W; k0 += 2u) {
            uint32_t word[2];
#pragma unroll
            for (int k = 0; k < 2; k++)
                word[k] = in && k0 + k < p.W ? load_agent(lat + (size_t)(k0 + k) * p.N + s) : ~0u;
#pragma unroll
            for (int k = 0; k < 2; k++)
                for (uint32_t b = 0; b < slots; b++) {
                    const bool empty = slots == 1u ? word[k] == 0u : (word[k] >> (8u * b) & 0xFFu) == 0u;
                    // (a taken slot after the first empty one ends the row)
                    if (empty && slot + room == (k0 + k) * slots + b) room++;
                    else if (!empty && room == 0u) slot++;
                }
        }
        return slot | room << 8;
    }
    // A particle into an empty slot; several lanes may fill one word.
    __device__ inline void place(uint32_t s, uint32_t slot, uint32_t particle) const
    {
        clear_zero_flag(p, p.word_particles ? slot : slot >> 2, s);
        if (p.word_particles) {
            store_agent(lat + (size_t)slot * p.N + s, particle);
        } else {
            __hip_atomic_store(reinterpret_cast<uint8_t *>(lat + (size_t)(slot >> 2) * p.N + s) + (slot & 3u),
                               (uint8_t)particle, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((slot >> 2) > 0) clear_chunk_flag(p, lat, slot >> 2, s >> 2);
        }
    }
    __device__ inline uint32_t occupancy(uint32_t s) const { return site_occupancy(p, lat, s); }
};

// Places a step's n entries (at most kMaxOverflows, with the carried ones);
// key0 and part0: entry threadIdx.x & 63.  All threads of the block call it.
// On thread 0 it returns how many entries stay listed.
template <int kThreads, class Sites>
__device__ inline uint32_t resolve_entries(const Params &p, const Sites &sites, unsigned long long *keys,
                                           ResolveLds<kThreads> &sh, uint32_t n, uint32_t carried, uint32_t t,
                                           unsigned long long key0, uint32_t part0)
{
    constexpr int kRound = ResolveLds<kThreads>::kRound;
    Control *ctl = p.ctl;
    const int tid = threadIdx.x;
    if (n <= 64u) {
        // Entry k's rank is the number of smaller keys (no two are equal).
        uint32_t rank = 0;
        for (uint32_t q = 0; q < n; q++) {
            const unsigned long long v = (unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)key0, (int)q) |
                                         (unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(key0 >> 32), (int)q) << 32;
            rank += v < key0 ? 1u : 0u;
        }
        if (tid < (int)n) {
            keys[rank] = key0;
            sh.parts[rank] = part0;
        }
        __syncthreads();
    } else {
        uint32_t M = 2;
        while (M < n) M <<= 1;
        for (uint32_t k = tid; k < M; k += kThreads) keys[k] = (k < n) ? __hip_atomic_load(&ctl->ovf_keys[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : ~0ull;
        __syncthreads();
        for (uint32_t k = 2; k <= M; k <<= 1) {
            for (uint32_t j = k >> 1; j > 0; j >>= 1) {
                for (uint32_t a = tid; a < M; a += kThreads) {
                    const uint32_t b = a ^ j;
                    if (b > a) {
                        const unsigned long long ka = keys[a], kb = keys[b];
                        const bool up = (a & k) == 0;
                        if ((ka > kb) == up) {
                            keys[a] = kb;
                            keys[b] = ka;
                        }
                    }
                }
                __syncthreads();
            }
        }
    }

    const uint32_t X = p.X, Y = p.Y, Z = p.Z, lane = tid & 63, wave = tid >> 6;
    if (p.relaxed) {
        // Relaxed handler (correct_overflows, MpdRdmeSolver.cu:1677-1761): the
        // carried entries, then this step's in canonical order, each into its
        // own site's first empty slot; entries of one site go in that order
        // (the kernel's rounds) and different sites do not interact.  So a wave
        // takes 64 of them at a time: an entry's slot is its site's occupancy
        // and the chunk's earlier entries of that site, which all fit if it
        // does.  A full site keeps the entry for the next step.
        uint32_t kept = 0;
        if (wave != 0) return 0;
        for (uint32_t e0 = 0; e0 < carried + n; e0 += 64u) {
            const uint32_t e = e0 + lane;
            const bool have = e < carried + n;
            uint32_t site = ~0u, particle = 0;
            if (e < carried) {
                site = load_agent(&ctl->carry_site[e]);
                particle = load_agent(&ctl->carry_part[e]);
            } else if (have) {
                const unsigned long long key = keys[e - carried];
                site = (uint32_t)((key >> 24) & 0xFFFFFFFFull);
                particle = load_agent(&ctl->ovf_part[key & 0x7FFull]);
            }
            uint32_t slot = have ? sites.occupancy(site) : p.P;
#pragma unroll 1
            for (uint32_t q = 0; q < 63u; q++)
                slot += q < lane && (uint32_t)__builtin_amdgcn_readlane((int)site, (int)q) == site ? 1u : 0u;
            const bool fits = slot < p.P;
            if (fits) sites.place(site, slot, particle);
            const unsigned long long stay = __ballot(have && !fits);
            if (have && !fits) {  // (at its own place or before: those have been read)
                const uint32_t k = kept + __builtin_amdgcn_mbcnt_hi((uint32_t)(stay >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)stay, 0u));
                store_agent(&ctl->carry_site[k], site);
                store_agent(&ctl->carry_part[k], particle);
            }
            kept += (uint32_t)__popcll(stay);
            wait_for_stores();  // the next chunk's loads see them
        }
        if (lane == 0) {
            ctl->carry_count = kept;
            ctl->ovf_total += n;
            if (n > 0) ctl->ovf_steps += 1;
            ctl->ovf_count = 0;
        }
        return kept;
    }

    for (uint32_t e0 = 0; e0 < n;) {
        const uint32_t e = e0 + wave;
        // room: empty slots in a row from sh.f_slot on; 0: no candidate has one,
        // kOut: the search leaves the lattice first.
        constexpr uint32_t kOut = 0xFFu;
        if (lane == 0u) sh.f_room[wave] = 0u;
        if (e < n) {
            const uint32_t site = (uint32_t)((keys[e] >> 24) & 0xFFFFFFFFull);
            const uint32_t st0 = p.sites[site], xc = site % X, yc = (site / X) % Y, zc = site / p.XY;
#pragma unroll 1
            for (uint32_t c = 0; c < kBallSites; c += 64u) {
                const uint32_t off = kBall.v[c + lane], R = off >> 12;
                const int dx = (int)(off & 15u) - 4, dy = (int)(off >> 4 & 15u) - 4, dz = (int)(off >> 8 & 15u) - 4;
                const uint32_t x = xc + (uint32_t)dx, y = yc + (uint32_t)dy, z = zc + (uint32_t)dz;
                // A site beyond the lattice's far side is a candidate only
                // where the reference's clamp, X - 1 - R in unsigned
                // arithmetic, wraps: the search then leaves the lattice, an
                // error.
                const bool before = (dx < 0 && xc < (uint32_t)-dx) || (dy < 0 && yc < (uint32_t)-dy) ||
                                    (dz < 0 && zc < (uint32_t)-dz);
                const bool ox = x >= X, oy = y >= Y, oz = z >= Z;
                const bool listed = c + lane < kBallSites && !before &&
                                    !((ox && X - 1 >= R) || (oy && Y - 1 >= R) || (oz && Z - 1 >= R));
                const bool out = listed && (ox || oy || oz), in = listed && !out;
                const uint32_t s = in ? x + X * y + p.XY * z : site;
                const uint32_t type = p.sites[s];
                const uint32_t seen = sites.look(in, s), slot = seen & 255u, room = seen >> 8;
                const unsigned long long m = __ballot(out || (in && room != 0u && type == st0));
                if (m == 0ull) continue;
                if (lane == (uint32_t)__builtin_ctzll(m)) {
                    sh.f_site[wave] = s;
                    sh.f_slot[wave] = slot;
                    sh.f_room[wave] = out ? kOut : room;
                }
                break;
            }
        }
        __syncthreads();
        if (wave == 0) {
            const uint32_t count = n - e0 < (uint32_t)kRound ? n - e0 : (uint32_t)kRound;
            uint32_t sl = 0, se = 0, particle = 0, room = 1;
            if (lane < count) {
                particle = n <= 64u ? sh.parts[e0 + lane] : load_agent(&ctl->ovf_part[keys[e0 + lane] & 0x7FFull]);
                se = sh.f_site[lane];
                sl = sh.f_slot[lane];
                room = sh.f_room[lane];
                if (room != 0u && room != kOut)
                    for (uint32_t q = 0; q < lane; q++)
                        if (sh.f_site[q] == se) {
                            sl++;
                            room--;
                            if (room == 0u) break;
                        }
            }
            // Entries up to the first whose search did not find a site, or
            // whose site the earlier ones of the round filled.
            const unsigned long long stop = __ballot(lane < count && (room == 0u || room == kOut));
            const uint32_t upto = stop ? (uint32_t)__builtin_ctzll(stop) : count;
            if (lane < upto) sites.place(se, sl, particle);
            if (lane == upto || (upto == 64u && lane == 0u)) {
                sh.placed = upto;
                const uint32_t r = upto < count ? sh.f_room[upto] : 1u;
                sh.failure = r == 0u ? kErrUnplaceable : (r == kOut ? kErrOutOfRange : 0u);
            }
            wait_for_stores();  // the next round's loads see the stores
        }
        __syncthreads();
        if (sh.failure != 0u) {
            if (tid == 0) set_error(ctl, sh.failure, t);
            break;
        }
        e0 += sh.placed;
    }
    if (tid == 0) {
        atomicAdd(&ctl->ovf_total, (unsigned long long)n);
        atomicAdd(&ctl->ovf_steps, 1ull);
        ctl->ovf_count = 0;
    }
    return 0;
}

// The overflow entries of a step on the lattice that it wrote, and the end of
// the step: the reaction list's counters cleared, the step counter advanced.
template <int kThreads>
__device__ inline void resolve_body(const Params &p, uint32_t *lat)
{
    __shared__ unsigned long long keys[kMaxOverflows];
    __shared__ ResolveLds<kThreads> sh;
    __shared__ uint32_t s_t;
    Control *ctl = p.ctl;
    const int tid = threadIdx.x;
    if (tid == 0) s_t = ctl->timestep;
    // A few entries are read along with their number.
    const uint32_t n = load_agent(&ctl->ovf_count);
    const unsigned long long key0 =
        __hip_atomic_load(&ctl->ovf_keys[tid & 63], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t part0 = load_agent(&ctl->ovf_part[tid & 63]);
    __syncthreads();
    // The step's reaction phase has consumed the reaction list.
    for (int k = tid; k < kListShards; k += kThreads) ctl->list_count[k] = 0u;
    if (tid == 0) ctl->list_overflow = 0u;
    const uint32_t t = s_t;
    const uint32_t carried = p.relaxed ? ctl->carry_count : 0u;
    if (n > kMaxOverflows || carried + n > kMaxOverflows) {
        if (tid == 0) {
            set_error(ctl, kErrOverflowCap, t);
            ctl->ovf_count = 0;
        }
    } else if (n != 0 || carried != 0) {
        resolve_entries<kThreads>(p, LatticeSites{p, lat}, keys, sh, n, carried, t, key0, part0);
    }
    if (tid == 0) ctl->timestep = t + 1;
}

}  // namespace lmx
