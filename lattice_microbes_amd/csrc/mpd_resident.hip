// The resident MPD-RDME run for gfx950: a solver of few particles steps inside
// one block, whose LDS holds a record per particle, for as many timesteps as
// the caller asked for in a single launch.
//
//  resident_gather_kernel  lists the particles of the lattice and clears their
//                          words (the whole device)
//  resident_run_kernel     one block per solver: x, y and z sweeps, reactions
//                          and overflow resolution of every step on the
//                          records, then the particles back into the lattice
//
// The sweeps are those of the boxed step (mpd_box.hip): a particle joins the
// hash chain of its target site and its new slot is its rank among the
// particles of that site on the chain.  Here the region is the whole lattice,
// so there is no shell, and the lattice is read and written once per run.
//
// Why: a step of a small lattice is launches, not work.  The bimolecular 64^3
// model (2000 particles) takes 16.5 us a step in boxes, two launches of which
// none fills the device, and an ensemble pays every member's lattice in every
// step although its members hold 2000 particles each.  One block steps them in
// 10.9 us (10.2 to 11.8 on 32^3, where 60 sites hold several particles), and an
// ensemble runs a member per CU: 128 replicates on 32^3 to 128^3 sites take
// 14.6 us a step against 970 us for the batched sweeps.
//
// What bounds it: a step is 28,000 cycles, 5,000 to 7,000 for each of the four
// rounds (vector issue: two records per thread, about 200 instructions each
// with the hash's quarter-rate multiplies, sixteen waves on four SIMDs) and
// 5,000 for the sites to evaluate (latency of one wave's evaluation).
#include "lmx_device.h"
#include "lmx_kernels.h"
#include "lmx_resident.h"
#include "lmx_wave.h"

namespace lmx {

namespace {

constexpr uint32_t kNT = kResidentThreads, kCap = kResidentCap;
constexpr uint32_t kChains = 8192u;      // two per record at least: most chains hold one particle
constexpr uint32_t kEnd = 0xFFFFu, kDead = 0xFFFFFFFFu;
constexpr uint32_t kIdBits = 13u;        // of a chain head: the particle; the sweep's tag above
constexpr uint32_t kTab = 2048u;         // floats of the model's tables kept in LDS
constexpr uint32_t kBall = 729u;         // sites within distance 4 along each axis

// key: x | y << 10 | z << 20.  ord: slot (4), class (2: stayed, from the minus,
// from the plus neighbour), site type (8), species (16).
__device__ inline uint32_t ord_rank(uint32_t o) { return o & 63u; }
__device__ inline uint32_t ord_type(uint32_t o) { return (o >> 6) & 0xFFu; }
__device__ inline uint32_t ord_species(uint32_t o) { return o >> 14; }
__device__ inline uint32_t make_ord(uint32_t slot, uint32_t cls, uint32_t type, uint32_t species)
{
    return slot | (cls << 4) | (type << 6) | (species << 14);
}
__device__ inline uint32_t chain_of(uint32_t key) { return (key ^ (key >> 7) ^ (key >> 15)) & (kChains - 1u); }

struct ResidentLds {
    uint32_t key[2][kCap], ord[2][kCap];
    uint16_t next[2][kCap];
    uint32_t head[2][kChains];
    float tab[kTab];
    uint32_t occ[kBall];            // particles of the sites around an overflow entry
    unsigned long long best;
    uint32_t n[2], nc, ovf, spill, pick;  // records; sites to evaluate; ...
};

__device__ inline uint32_t site_of(const Params &p, uint32_t key)
{
    return (key & 1023u) + __umul24((key >> 10) & 1023u, p.X) + (key >> 20) * p.XY;
}

// A particle into the lattice in global memory.
template <class L>
__device__ inline void put_particle(const Params &p, uint32_t *lat, uint32_t i, uint32_t slot, uint32_t species)
{
    if constexpr (L::kPerWord == 4)
        reinterpret_cast<uint8_t *>(lat + (size_t)(slot >> 2) * p.N + i)[slot & 3u] = (uint8_t)species;
    else
        lat[(size_t)slot * p.N + i] = species;
}

// How many particles of key come before order o on its chain (generation g),
// and how many there are.
__device__ inline void chain_rank(const ResidentLds &s, int g, uint32_t e, uint32_t key, uint32_t o, uint32_t &before,
                                  uint32_t &total)
{
    before = 0;
    total = 1;
    uint32_t q = s.head[g][chain_of(key)] & ((1u << kIdBits) - 1u);
    if (q == e && s.next[g][e] == kEnd) return;
    total = 0;
    while (q != kEnd) {
        if (s.key[g][q] == key) {
            total++;
            before += ord_rank(s.ord[g][q]) < ord_rank(o) ? 1u : 0u;
        }
        q = s.next[g][q];
    }
}

// One more particle at the end of generation 0; past the block's capacity it
// goes into the (otherwise empty) lattice and the run ends after this step.
template <class L>
__device__ inline void append(const Params &p, uint32_t *lat, ResidentLds &s, uint32_t key, uint32_t ord)
{
    const uint32_t k = atomicAdd(&s.n[0], 1u);
    if (k < kCap) {
        s.key[0][k] = key;
        s.ord[0][k] = ord;
    } else {
        s.spill = 1u;
        put_particle<L>(p, lat, site_of(p, key), ord & 15u, ord_species(ord));
    }
}

// Whether a site of several particles with total propensity a reacts
// (checkForReaction, byte_reaction_dev.cu:139-144).  1 - exp(-a) <= a, with room
// for the rounding of both, and u is 0 or at least 2^-32: most sites need no
// exponential.
__device__ inline bool reacts(float a, float u)
{
    if (a == 0.0f || !(u <= a * 1.0001f)) return false;
    const float prob = reaction_probability(a);
    return prob > 0.0f && u <= prob;
}

// The site of record e, by a wave: its total propensity a, or, if known is
// set, its reaction.  The site's particles (the members of its chain in
// generation 1 that fit) lie a slot per lane; a reaction's result goes back as
// records of generation 0 -- in the members' places, further ones appended.
template <class L>
__device__ inline void react_site_wave(const Params &p, uint32_t *lat, ResidentLds &s, uint32_t e, bool known, float a,
                                       uint32_t t, unsigned long long h3)
{
    constexpr uint32_t P = L::P;
    const uint32_t lane = lane_id(), key = s.key[1][e], type = ord_type(s.ord[1][e]);
    uint32_t mine = 0, rec = kDead;  // this lane's slot: its species and its record
    for (uint32_t q = s.head[1][chain_of(key)] & ((1u << kIdBits) - 1u); q != kEnd; q = s.next[1][q]) {
        if (s.key[1][q] != key || s.key[0][q] == kDead) continue;
        const uint32_t o = s.ord[0][q];  // (its slot after the sweeps)
        if (lane == (o & 15u)) {
            mine = ord_species(o);
            rec = q;
        }
    }
    const uint32_t i = site_of(p, key);
    if (!known) {
        // total_propensity's sum: the same terms in the same order, a
        // particle's row of them a lane each.
        const uint32_t count = (uint32_t)__popcll(__ballot(mine != 0u));
        a = p.qp0[type];
#pragma unroll 1
        for (uint32_t m = 0; m < count; m++) {
            const uint32_t row = type * p.nS + lane_of(mine, m) - 1u;
            float v = 0.0f;
            if (lane == m) v = p.qp1[row];
            else if (lane > m && lane < count) v = p.qp2[(size_t)row * p.nS + (mine - 1u)];
#pragma unroll 1
            for (uint32_t n = m; n < count; n++) a += __uint_as_float(lane_of(__float_as_uint(v), n));
        }
        if (!reacts(a, uniform01(i, 1, 0, h3))) return;
    }
    bool underflow;
    const uint32_t now = wave_products<P>(p, i, type, mine, a, h3, underflow);
    if (underflow && lane == 0u && atomicCAS(&p.ctl->error, 0u, kErrReactionUnderflow) == 0u) p.ctl->error_step = t;
    if (lane >= P) return;
    // products without a slot are overflow entries: only a full site has any
    if (lane == P - 1u && now) s.ovf = 1u;
    if (rec != kDead) {
        if (now) s.ord[0][rec] = make_ord(lane, 0u, type, now);
        else s.key[0][rec] = kDead;
    } else if (now) {
        append<L>(p, lat, s, key, make_ord(lane, 0u, type, now));
    }
}

// total_propensity's sum for a site of 2 to K particles, in slot order: the
// terms loaded together, added in its order.
template <uint32_t K>
__device__ inline float few_propensity(const Params &p, uint32_t type, const uint32_t *sp, uint32_t count)
{
    float a = p.qp0[type], one[K], two[K][K];
    uint32_t row[K];
#pragma unroll
    for (uint32_t m = 0; m < K; m++) row[m] = (m < count ? sp[m] : sp[0]) - 1u;
#pragma unroll
    for (uint32_t m = 0; m < K; m++) {
        const uint32_t r = type * p.nS + row[m];
        one[m] = p.qp1[r];
#pragma unroll
        for (uint32_t n = m + 1u; n < K; n++) two[m][n] = p.qp2[(size_t)r * p.nS + row[n]];
    }
#pragma unroll
    for (uint32_t m = 0; m < K; m++) {
        if (m >= count) break;
        a += one[m];
#pragma unroll
        for (uint32_t n = m + 1u; n < K; n++)
            if (n < count) a += two[m][n];
    }
    return a;
}

// The nc sites listed in s.next[0], whose particles are several or whose one
// passed its test.  A lane per site sums the propensities of up to kFew
// particles; the sites that react, and those of more particles, are taken by
// the whole wave.  Latency bounds it where the sites are few, so that one wave
// takes up to 32 of them (32^3, 2000 particles, 60 sites: 10.2 us a step, dealt
// to sixteen waves 10.7), and issue where they are many (16^3, 2000 particles:
// 12.0, in one wave 15.6).  kFew: 12^3, 2500 particles 14.7 us a step, with 4
// of them 16.3.
//
// A thread per site for everything, with the site's slots in registers,
// unrolls the evaluation over every slot: with 16 of them 40 VGPRs and 138
// SGPRs spilled at this block's 128, and 64^3 took 14.6 us a step against
// 10.9 (8 slots, where nothing spilled: 11.4 against 10.9).
template <class L>
__device__ inline void react_sites(const Params &p, uint32_t *lat, ResidentLds &s, uint32_t nc, uint32_t t,
                                   unsigned long long h3, const float2 *tab)
{
    constexpr uint32_t kFew = L::P < 6 ? L::P : 6;
    const uint32_t waves = nc <= 32u ? 1u : (nc >= 512u ? 16u : (nc + 31u) / 32u);
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    if (wave >= waves) return;
#pragma unroll 1
    for (uint32_t k0 = 0; k0 < nc; k0 += 64u * waves) {
        const uint32_t k = k0 + lane_id() * waves + wave;
        uint32_t e = 0, count = 0, type = 0, sp[kFew] = {};
        float a = 0.0f, u = 1.0f;
        bool hit = false;
        if (k < nc) {
            e = s.next[0][k];
            const uint32_t key = s.key[1][e];
            type = ord_type(s.ord[1][e]);
            for (uint32_t q = s.head[1][chain_of(key)] & ((1u << kIdBits) - 1u); q != kEnd; q = s.next[1][q]) {
                if (s.key[1][q] != key || s.key[0][q] == kDead) continue;
                const uint32_t o = s.ord[0][q], j = o & 15u;
                count++;
#pragma unroll
                for (uint32_t m = 0; m < kFew; m++)
                    if (j == m) sp[m] = ord_species(o);
            }
            u = uniform01(site_of(p, key), 1, 0, h3);
        }
        const bool pairs = __ballot(count > 2u && count <= kFew) == 0ull;  // no site of three and more
        if (count == 1u) {
            const float2 ap = tab[type * p.nS + sp[0] - 1u];
            a = ap.x;
            hit = a != 0.0f && ap.y > 0.0f && u <= ap.y;
        } else if (count >= 2u && count <= kFew) {
            a = pairs ? few_propensity<2>(p, type, sp, count) : few_propensity<kFew>(p, type, sp, count);
            hit = reacts(a, u);
        }
#pragma unroll 1
        for (unsigned long long m = __ballot(hit || count > kFew); m; m &= m - 1) {
            const uint32_t src = (uint32_t)__builtin_ctzll(m);
            react_site_wave<L>(p, lat, s, lane_of(e, src), lane_of(count, src) <= kFew,
                               __uint_as_float(lane_of(__float_as_uint(a), src)), t, h3);
        }
    }
}

__device__ inline uint32_t agent_load(const uint32_t *q)
{
    return __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The step's overflow entries into sites with room (resolve_kernel's rules,
// on the records of generation 0): in canonical order, each entry scans the
// candidate sites of growing radius.  All threads call it; rare.
template <class L>
__device__ void resolve_records(const Params &p, uint32_t *lat, ResidentLds &s, uint32_t t)
{
    constexpr uint32_t P = L::P;
    Control *ctl = p.ctl;
    const uint32_t tid = threadIdx.x;
    __threadfence();
    __syncthreads();
    const uint32_t n = agent_load(&ctl->ovf_count);
    const uint32_t carried = p.relaxed ? agent_load(&ctl->carry_count) : 0u;
    __syncthreads();
    if (n > kMaxOverflows || carried + n > kMaxOverflows) {
        if (tid == 0) {
            if (atomicCAS(&ctl->error, 0u, kErrOverflowCap) == 0u) ctl->error_step = t;
            ctl->ovf_count = 0u;
        }
        __threadfence();
        __syncthreads();
        return;
    }
    unsigned long long last = 0ull;
    bool any = false, failed = false;
    uint32_t kept = 0;
    for (uint32_t e = 0; e < carried + n && !failed; e++) {
        uint32_t site, particle;
        if (e < carried) {
            site = agent_load(&ctl->carry_site[e]);
            particle = agent_load(&ctl->carry_part[e]);
        } else {
            // the smallest key above the last one
            if (tid == 0) s.best = ~0ull;
            __syncthreads();
            for (uint32_t k = tid; k < n; k += kNT) {
                const unsigned long long v = __hip_atomic_load(&ctl->ovf_keys[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (!any || v > last) atomicMin(&s.best, v);
            }
            __syncthreads();
            last = s.best;
            any = true;
            __syncthreads();
            site = (uint32_t)((last >> 24) & 0xFFFFFFFFull);
            particle = agent_load(&ctl->ovf_part[last & 0x7FFull]);
        }
        const uint32_t xc = site % p.X, yc = (site / p.X) % p.Y, zc = site / p.XY;
        // particles of every site within distance 4 of it
        for (uint32_t k = tid; k < kBall; k += kNT) s.occ[k] = 0u;
        __syncthreads();
        const uint32_t m = s.n[0] < kCap ? s.n[0] : kCap;
        for (uint32_t k = tid; k < m; k += kNT) {
            const uint32_t key = s.key[0][k];
            if (key == kDead) continue;
            const uint32_t dx = (key & 1023u) + 4u - xc, dy = ((key >> 10) & 1023u) + 4u - yc, dz = (key >> 20) + 4u - zc;
            if (dx <= 8u && dy <= 8u && dz <= 8u) atomicAdd(&s.occ[dx + 9u * (dy + 9u * dz)], 1u);
        }
        __syncthreads();
        if (s.spill) {  // and those past the block's capacity
            for (uint32_t k = tid; k < kBall; k += kNT) {
                const uint32_t x = xc + k % 9u - 4u, y = yc + (k / 9u) % 9u - 4u, z = zc + k / 81u - 4u;
                if (x >= p.X || y >= p.Y || z >= p.Z) continue;
                for (uint32_t q = 0; q < p.W; q++) {
                    const uint32_t v = agent_load(lat + (size_t)q * p.N + x + p.X * y + p.XY * z);
                    for (uint32_t b = 0; b < 4u; b++)
                        s.occ[k] += p.word_particles ? (b == 0u && v ? 1u : 0u) : (((v >> (8u * b)) & 0xFFu) ? 1u : 0u);
                }
            }
            __syncthreads();
        }
        auto occupancy = [&](uint32_t x, uint32_t y, uint32_t z) {
            return s.occ[(x + 4u - xc) + 9u * ((y + 4u - yc) + 9u * (z + 4u - zc))];
        };
        const uint32_t st0 = p.sites[site];
        if (p.relaxed) {
            // its own site, or it stays listed
            const uint32_t occ = occupancy(xc, yc, zc);
            __syncthreads();
            if (tid == 0) {
                if (occ < P) {
                    append<L>(p, lat, s, xc | (yc << 10) | (zc << 20), make_ord(occ, 0u, st0, particle));
                } else {
                    __hip_atomic_store(&ctl->carry_site[kept], site, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(&ctl->carry_part[kept], particle, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            if (occ >= P) kept++;
            __threadfence();
            __syncthreads();
            continue;
        }
        int found = 0x7fffffff;
        for (uint32_t R = 0; R <= kMaxReplacementDist && found == 0x7fffffff; R++) {
            const uint32_t minD = R > 0 ? R - 1 : 0, X = p.X, Y = p.Y, Z = p.Z;
            const uint32_t x0 = xc >= R ? xc - R : 0, x1 = (xc <= X - 1 - R) ? xc + R : X - 1;
            const uint32_t y0 = yc >= R ? yc - R : 0, y1 = (yc <= Y - 1 - R) ? yc + R : Y - 1;
            const uint32_t z0 = zc >= R ? zc - R : 0, z1 = (zc <= Z - 1 - R) ? zc + R : Z - 1;
            const uint32_t ny = y1 - y0 + 1, nz = z1 - z0 + 1, all = (x1 - x0 + 1) * ny * nz;  // at most 729
            if (tid == 0) s.pick = 0x7fffffffu;
            __syncthreads();
            uint32_t x = 0, y = 0, z = 0;
            if (tid < all) {
                x = x0 + tid / (ny * nz);
                const uint32_t rem = tid % (ny * nz);
                y = y0 + rem / nz;
                z = z0 + rem % nz;
                const long long dx = (long long)x - xc, dy = (long long)y - yc, dz = (long long)z - zc;
                const long long r2 = dx * dx + dy * dy + dz * dz;
                if (r2 <= (long long)(R * R) && (r2 > (long long)(minD * minD) || R == 0)) {
                    if (x >= X || y >= Y || z >= Z) atomicMin(&s.pick, 2u * tid + 1u);
                    else if (p.sites[x + X * y + p.XY * z] == st0 && occupancy(x, y, z) < P) atomicMin(&s.pick, 2u * tid);
                }
            }
            __syncthreads();
            found = (int)s.pick;
            if (found != 0x7fffffff && !(found & 1) && tid == (uint32_t)found >> 1)
                append<L>(p, lat, s, x | (y << 10) | (z << 20), make_ord(occupancy(x, y, z), 0u, st0, particle));
            __syncthreads();
        }
        if (found == 0x7fffffff || (found & 1)) {
            if (tid == 0 && atomicCAS(&ctl->error, 0u, found & 1 && found != 0x7fffffff ? kErrOutOfRange : kErrUnplaceable) == 0u)
                ctl->error_step = t;
            failed = true;
        }
    }
    if (tid == 0) {
        if (p.relaxed) ctl->carry_count = kept;
        ctl->ovf_total += n;
        if (n > 0) ctl->ovf_steps += 1;
        ctl->ovf_count = 0u;
        s.ovf = p.relaxed && kept ? 1u : 0u;
    }
    __threadfence();
    __syncthreads();
}

}  // namespace

// The particles of the lattice into the job's list, their words cleared.  Past
// the list's capacity nothing is cleared any more (the run puts the listed
// ones back).
template <class L>
__device__ inline void gather_body(const ResidentJob &job, uint32_t block, uint32_t nblocks)
{
    constexpr int W = L::W;
    const Params &p = job.p;
    if (agent_load(&p.ctl->timestep) != job.start) return;
    uint32_t *lat = job.lat;
    const bool by4 = (p.N & 3u) == 0u;
    const uint32_t items = by4 ? p.N >> 2 : p.N;
    for (uint32_t g0 = block * 256u; g0 < items; g0 += nblocks * 256u) {
        const uint32_t g = g0 + threadIdx.x;
        uint32_t v[4] = {0u, 0u, 0u, 0u};
        if (g < items) {
            for (uint32_t k = 0; k < (p.packed ? 1u : (uint32_t)W); k++) {
                if (by4) {
                    const uint4 q = reinterpret_cast<const uint4 *>(lat + (size_t)k * p.N)[g];
                    v[0] |= q.x;
                    v[1] |= q.y;
                    v[2] |= q.z;
                    v[3] |= q.w;
                } else {
                    v[0] |= lat[(size_t)k * p.N + g];
                }
            }
        }
        if (__ballot((v[0] | v[1] | v[2] | v[3]) != 0u) == 0ull) continue;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (__ballot(v[q] != 0u) == 0ull) continue;
            const uint32_t i = by4 ? 4u * g + q : g;
            uint32_t w[W], c = 0;
#pragma unroll
            for (int k = 0; k < W; k++) w[k] = 0u;
            if (v[q]) {
#pragma unroll
                for (int k = 0; k < W; k++) {
                    if (k == 0 || L::need_next(p, w[k > 0 ? k - 1 : 0])) w[k] = lat[(size_t)k * p.N + i];
                    if constexpr (L::kPerWord == 4) {
                        for (int b = 0; b < 4; b++) c += ((w[k] >> (8 * b)) & 0xFFu) ? 1u : 0u;
                    } else {
                        c += w[k] ? 1u : 0u;
                    }
                }
            }
            // places: a prefix over the wave and one reservation
            uint32_t pre = c;
            const uint32_t lane = threadIdx.x & 63u;
            for (uint32_t d = 1; d < 64u; d <<= 1) {
                const uint32_t o = __shfl_up(pre, d, 64);
                if (lane >= d) pre += o;
            }
            uint32_t base = 0;
            if (lane == 63u) base = atomicAdd(job.count, pre);
            base = __shfl(base, 63, 64) + pre - c;
            if (c == 0u) continue;
            const bool fits = base + c <= kCap;
            uint32_t at = base;
            for (uint32_t j = 0; j < (uint32_t)L::P; j++) {
                uint32_t sp = 0;
#pragma unroll
                for (int k = 0; k < W; k++) {
                    if constexpr (L::kPerWord == 4) sp = (j >> 2) == (uint32_t)k ? (w[k] >> (8u * (j & 3u))) & 0xFFu : sp;
                    else sp = j == (uint32_t)k ? w[k] : sp;
                }
                if (!sp) continue;
                if (at < kCap) job.list[at] = fits ? make_uint2(i, j | (sp << 8)) : make_uint2(kDead, 0u);
                at++;
            }
            if (fits) {
#pragma unroll
                for (int k = 0; k < W; k++)
                    if (w[k]) lat[(size_t)k * p.N + i] = 0u;
            }
        }
    }
}

// Blocks per job: job r runs on blocks r * per .. (r + 1) * per - 1.
// (Two kernels each, so that the job is read through the scalar cache either
// way: a choice at run time made its fields vector registers.)
template <class L>
__global__ __launch_bounds__(256) void resident_gather_kernel(ResidentJob job)
{
    gather_body<L>(job, blockIdx.x, gridDim.x);
}

template <class L>
__global__ __launch_bounds__(256) void resident_gather_jobs_kernel(const ResidentJob *__restrict__ jobs, uint32_t per)
{
    const uint32_t r = blockIdx.x / per;
    gather_body<L>(jobs[r], blockIdx.x - r * per, per);
}

template <class L>
__device__ __attribute__((always_inline)) inline void run_body(const ResidentJob &job, ResidentLds &s)
{
    Params p = job.p;
    constexpr uint32_t P = L::P;
    Control *ctl = p.ctl;
    uint32_t *lat = job.lat;
    const uint32_t tid = threadIdx.x;
    if (agent_load(&ctl->timestep) != job.start) return;
    const uint32_t found = agent_load(job.count);
    const bool periodic = p.boundary == 0;

    for (uint32_t k = tid; k < 2u * kChains; k += kNT) (&s.head[0][0])[k] = 0u;
    // The model's tables in LDS where they are small.
    const uint32_t nT = p.nST * p.nST * p.nS, n1 = p.nST * p.nS;
    const unsigned long long n2 = (unsigned long long)n1 * p.nS;
    if (nT + 3ull * n1 + p.nST + n2 <= kTab) {
        float *q = s.tab;
        auto keep = [&](const float *&v, uint32_t n) {
            for (uint32_t k = tid; k < n; k += kNT) q[k] = v[k];
            v = q;
            q += n;
        };
        keep(p.prob1, 2u * n1);
        keep(p.T, nT);
        keep(p.qp0, p.nST);
        keep(p.qp1, n1);
        keep(p.qp2, (uint32_t)n2);
    }
    if (tid == 0) {
        s.n[0] = found < kCap ? found : kCap;
        s.n[1] = 0u;
        s.ovf = p.relaxed && agent_load(&ctl->carry_count) ? 1u : 0u;
        s.spill = s.nc = 0u;
    }
    for (uint32_t k = tid; k < found && k < kCap; k += kNT) {
        const uint2 v = job.list[k];
        s.key[0][k] = kDead;
        if (v.x == kDead) continue;
        const uint32_t r = v.x / p.X, x = v.x - r * p.X, z = r / p.Y, y = r - z * p.Y;
        s.key[0][k] = x | (y << 10) | (z << 20);
        s.ord[0][k] = make_ord(v.y & 255u, 0u, p.nST > 1u ? p.sites[v.x] : 0u, v.y >> 8);
    }
    const float2 *tab = reinterpret_cast<const float2 *>(p.prob1);
    __syncthreads();

    // Sweep of one particle along an axis: its target's key and record.
    auto move = [&](uint32_t axis, unsigned long long h, uint32_t &key, uint32_t &ord, uint32_t slot) {
        const uint32_t sh = 10u * axis, len = axis == 0 ? p.X : (axis == 1 ? p.Y : p.Z);
        const uint32_t stride = axis == 0 ? 1u : (axis == 1 ? p.X : p.XY);
        const uint32_t co = (key >> sh) & 1023u, i = site_of(p, key);
        const uint32_t st = ord_type(ord), sp = ord_species(ord);
        const bool hm = periodic || co > 0u, hp = periodic || co + 1u < len;
        const uint32_t cm = co > 0u ? co - 1u : len - 1u, cp = co + 1u < len ? co + 1u : 0u;
        uint32_t stm = st, stp = st;
        if (p.nST > 1u) {
            stm = p.sites[hm ? i - co * stride + cm * stride : i];
            stp = p.sites[hp ? i - co * stride + cp * stride : i];
        }
        const float u = uniform01(i, p.pcb, slot, h);
        const float qm = lookup_T_if(p, p.T, hm, sp, st, stm);
        const float qp = lookup_T_if(p, p.T, hp, sp, st, stp);
        const bool minus = u < qm, plus = !minus && u >= 0.5f && u < (qp + 0.5f);
        const uint32_t cn = minus ? cm : (plus ? cp : co);
        key += (cn - co) << sh;
        ord = make_ord(slot, plus ? 1u : (minus ? 2u : 0u), minus ? stm : (plus ? stp : st), sp);
    };
    auto join = [&](int g, uint32_t e, uint32_t key, uint32_t ord, uint32_t tag) {
        s.key[g][e] = key;
        s.ord[g][e] = ord;
        const uint32_t old = atomicExch(&s.head[g][chain_of(key)], e | (tag << kIdBits));
        s.next[g][e] = (uint16_t)((old >> kIdBits) == tag ? old & ((1u << kIdBits) - 1u) : kEnd);
    };

    uint32_t done = 0;
    if (found <= kCap) {
        for (; done < job.nsteps && !s.spill; done++) {
            const uint32_t t = job.start + done, tag = 3u * done;
            if (tid == 0) __hip_atomic_store(&ctl->timestep, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // x: generation 0 to 1, the records packed again
            {
                const unsigned long long h = timestep_hash(p.seed32, t, 0);
                const uint32_t n = s.n[0];
                for (uint32_t e0 = 0; e0 < n; e0 += kNT) {
                    const uint32_t e = e0 + tid;
                    uint32_t key = e < n ? s.key[0][e] : kDead, ord = 0;
                    const bool alive = key != kDead;
                    const unsigned long long m = __ballot(alive);
                    uint32_t base = 0;
                    const uint32_t lane = tid & 63u;
                    if (lane == 0u && m) base = atomicAdd(&s.n[1], (uint32_t)__popcll(m));
                    base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
                    if (!alive) continue;
                    const uint32_t to = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                    ord = s.ord[0][e];
                    move(0, h, key, ord, ord & 15u);
                    join(1, to, key, ord, tag + 1u);
                }
            }
            __syncthreads();
            const uint32_t n = s.n[1];
            // y: 1 to 0, z: 0 to 1
#pragma unroll 1
            for (uint32_t axis = 1; axis < 3; axis++) {
                const int from = (int)(axis & 1u), to = 1 - from;
                const unsigned long long h = timestep_hash(p.seed32, t, axis);
                for (uint32_t e = tid; e < n; e += kNT) {
                    uint32_t key = s.key[from][e], ord = s.ord[from][e], before, total;
                    if (key == kDead) {
                        s.key[to][e] = kDead;
                        continue;
                    }
                    chain_rank(s, from, e, key, ord, before, total);
                    if (before >= P) {
                        record_overflow(ctl, axis - 1u, site_of(p, key), before - P, ord_species(ord));
                        s.ovf = 1u;
                        s.key[to][e] = kDead;
                        continue;
                    }
                    move(axis, h, key, ord, before);
                    join(to, e, key, ord, tag + 1u + axis);
                }
                if (axis == 2 && tid == 0) s.n[0] = n;
                __syncthreads();
            }
            // the step's lattice: generation 1 to 0
            const unsigned long long h3 = timestep_hash(p.seed32, t, 3);
            for (uint32_t e = tid; e < n; e += kNT) {
                const uint32_t key = s.key[1][e], ord = s.ord[1][e];
                uint32_t before, total;
                if (key == kDead) {
                    s.key[0][e] = kDead;
                    continue;
                }
                chain_rank(s, 1, e, key, ord, before, total);
                const uint32_t st = ord_type(ord), sp = ord_species(ord);
                if (before >= P) {
                    record_overflow(ctl, 2u, site_of(p, key), before - P, sp);
                    s.ovf = 1u;
                    s.key[0][e] = kDead;
                    continue;
                }
                s.key[0][e] = key;
                s.ord[0][e] = make_ord(before, 0u, st, sp);
                // A particle alone takes its reaction test from the table; a
                // site that reacts or holds several is evaluated after the
                // barrier, by a wave of its own (beside this loop, every wave
                // with such a site ran the whole evaluation: 19,000 of a
                // step's 40,000 cycles).
                if (p.R > 0 && before == 0u) {
                    bool whole = total > 1u;
                    if (!whole) {
                        const float2 ap = tab[st * p.nS + (sp - 1u)];
                        whole = ap.x != 0.0f && ap.y > 0.0f && uniform01(site_of(p, key), 1, 0, h3) <= ap.y;
                    }
                    if (whole) s.next[0][atomicAdd(&s.nc, 1u)] = (uint16_t)e;  // (the links of generation 0 are free)
                }
            }
            if (tid == 0) s.n[1] = 0u;
            __syncthreads();
            const uint32_t nc = s.nc;
            if (nc) {
                react_sites<L>(p, lat, s, nc, t, h3, tab);
                __syncthreads();
                if (tid == 0) s.nc = 0u;
            }
            if (s.ovf) resolve_records<L>(p, lat, s, t);
        }
    }

    // The particles back into the lattice.
    const uint32_t n = s.n[0] < kCap ? s.n[0] : kCap;
    for (uint32_t e = tid; e < n; e += kNT) {
        const uint32_t key = s.key[0][e];
        if (key == kDead) continue;
        const uint32_t ord = s.ord[0][e];
        put_particle<L>(p, lat, site_of(p, key), ord & 15u, ord_species(ord));
    }
    if (tid == 0) {
        ctl->timestep = job.start + done;
        *job.count = 0u;
    }
}

template <class L>
__global__ __launch_bounds__(kResidentThreads) void resident_run_kernel(ResidentJob job)
{
    __shared__ ResidentLds s;
    run_body<L>(job, s);
}

template <class L>
__global__ __launch_bounds__(kResidentThreads) void resident_run_jobs_kernel(const ResidentJob *__restrict__ jobs)
{
    __shared__ ResidentLds s;
    run_body<L>(jobs[blockIdx.x], s);
}

uint32_t resident_gather_blocks(uint32_t N)
{
    // a few rounds of 256 threads x 4 sites for the largest lattices
    const uint32_t b = (N / 4u + 255u) / 256u;
    return b < 1u ? 1u : (b > 512u ? 512u : b);
}

hipError_t launch_resident(const ResidentJob &one, const ResidentJob *jobs, uint32_t n, uint32_t per, uint32_t P,
                           bool words, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    const dim3 gg(n * per), gr(n);
#define LMX_RESIDENT(LL)                                                                             \
    if (jobs) {                                                                                      \
        hipLaunchKernelGGL((resident_gather_jobs_kernel<LL>), gg, dim3(256), 0, st, jobs, per);      \
        hipLaunchKernelGGL((resident_run_jobs_kernel<LL>), gr, dim3(kResidentThreads), 0, st, jobs); \
    } else {                                                                                         \
        hipLaunchKernelGGL((resident_gather_kernel<LL>), gg, dim3(256), 0, st, one);                 \
        hipLaunchKernelGGL((resident_run_kernel<LL>), gr, dim3(kResidentThreads), 0, st, one);       \
    }                                                                                                \
    break
    switch ((words ? 100 : 0) + (int)P) {
    case 4: LMX_RESIDENT(ByteSites<1>);
    case 8: LMX_RESIDENT(ByteSites<2>);
    case 16: LMX_RESIDENT(ByteSites<4>);
    case 104: LMX_RESIDENT(WordSites<4>);
    case 108: LMX_RESIDENT(WordSites<8>);
    case 116: LMX_RESIDENT(WordSites<16>);
    default: return hipErrorInvalidValue;
    }
#undef LMX_RESIDENT
    return hipGetLastError();
}

}  // namespace lmx
