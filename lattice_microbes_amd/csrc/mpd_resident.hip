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
// What bounds it (64^3, rocprofv3): a step is 26,250 cycles, at least 13,490 of them
// vector issue (13,490 instructions on four SIMDs, four cycles and more each: two
// records a thread in each of four rounds, with the hash's quarter-rate
// multiplies), the rest latency of dependent LDS accesses between five
// barriers.
#include "lmx_device.h"
#include "lmx_kernels.h"
#include "lmx_resident.h"
#include "lmx_resolve.h"
#include "lmx_wave.h"

namespace lmx {

namespace {

constexpr uint32_t kNT = kResidentThreads, kCap = kResidentCap;
constexpr uint32_t kChains = 8192u;      // two per record at least: most chains hold one particle
constexpr uint32_t kEnd = 0xFFFFu, kDead = 0xFFFFFFFFu;
constexpr uint32_t kIdBits = 13u;        // of a chain head: the particle; the sweep's tag above
constexpr uint32_t kTab = 2048u;         // floats of the model's tables kept in LDS

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
    ResolveLds<(int)kNT> resolve;
    uint32_t n[2], nc, ovf, spill;  // records; sites to evaluate; ...
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
__device__ inline uint32_t append(const Params &p, uint32_t *lat, ResidentLds &s, uint32_t key, uint32_t ord)
{
    const uint32_t k = atomicAdd(&s.n[0], 1u);
    if (k < kCap) {
        s.key[0][k] = key;
        s.ord[0][k] = ord;
    } else {
        s.spill = 1u;
        put_particle<L>(p, lat, site_of(p, key), ord & 15u, ord_species(ord));
    }
    return k;
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

// The reaction of record e's site (total propensity a), by a wave.  The site's
// particles (the members of its chain in generation 1 that fit) lie a slot per
// lane; the result goes back as records of generation 0 -- in the members'
// places, further ones appended.
template <class L>
__device__ inline void react_site_wave(const Params &p, uint32_t *lat, ResidentLds &s, uint32_t e, float a, uint32_t t,
                                       unsigned long long h3)
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
    bool underflow;
    const uint32_t now = wave_products<P>(p, site_of(p, key), type, mine, a, h3, underflow);
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
// passed its test.  A lane per site sums its propensities, and a site that
// reacts is taken by the whole wave.  Latency bounds it where the sites are few,
// so that one wave takes up to 32 of them (32^3, 2000 particles, 60 sites: 10.2
// us a step, dealt to sixteen waves 10.7), and issue where they are many (16^3,
// 2000 particles: 12.0, in one wave 15.6).  Sites of up to kFew particles keep
// these in registers and their terms in flight together (8 slots: 64 crowded
// sites in 32^3 19.7 us a step, with six in registers 25.5), fuller ones in LDS,
// a row of terms at a time (16 slots, 100 sites of 14 particles: 73 us, by a
// wave each 148).
//
// A thread per site for everything, with the site's slots in registers,
// unrolls the evaluation over every slot: with 16 of them 40 VGPRs and 138
// SGPRs spilled at this block's 128, and 64^3 took 14.6 us a step against
// 10.9 (8 slots, where nothing spilled: 11.4 against 10.9).
template <class L>
__device__ inline void react_sites(const Params &p, uint32_t *lat, ResidentLds &s, uint32_t nc, uint32_t t,
                                   unsigned long long h3, const float2 *tab)
{
    constexpr uint32_t P = L::P, kFew = P <= 8 ? P : 6;
    const uint32_t waves = nc <= 32u ? 1u : (nc >= 512u ? 16u : (nc + 31u) / 32u);
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = lane_id();
    if (wave >= waves) return;
    // Slots of the fuller sites: this wave's part of the chain heads of
    // generation 0, free until the next y sweep, which finds them zero.
    static_assert(sizeof(s.head[0]) >= kNT / 64u * P * 64u * sizeof(uint16_t), "room for the slots");
    uint16_t (*slots)[64] = reinterpret_cast<uint16_t (*)[64]>(&s.head[0][0]) + wave * P;
#pragma unroll 1
    for (uint32_t k0 = 0; k0 < nc; k0 += 64u * waves) {
        const uint32_t k = k0 + lane * waves + wave;
        uint32_t e = 0, count = 0, type = 0, sp[kFew] = {};
        float a = 0.0f, u = 1.0f;
        bool hit = false;
        auto members = [&](auto &&with) {  // slot and species of each of the site's particles
            const uint32_t key = s.key[1][e];
            for (uint32_t q = s.head[1][chain_of(key)] & ((1u << kIdBits) - 1u); q != kEnd; q = s.next[1][q])
                if (s.key[1][q] == key && s.key[0][q] != kDead) with(s.ord[0][q] & 15u, ord_species(s.ord[0][q]));
        };
        if (k < nc) {
            e = s.next[0][k];
            type = ord_type(s.ord[1][e]);
            members([&](uint32_t j, uint32_t species) {
                count++;
#pragma unroll
                for (uint32_t m = 0; m < kFew; m++)
                    if (j == m) sp[m] = species;
            });
            u = uniform01(site_of(p, s.key[1][e]), 1, 0, h3);
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
        if (kFew < P && __ballot(count > kFew) != 0ull) {
            if (count > kFew) {
                members([&](uint32_t j, uint32_t species) { slots[j][lane] = (uint16_t)species; });
                a = packed_propensity<P>(p, type, slots, lane, count);
                hit = reacts(a, u);
            }
            for (uint32_t m = lane; m < P * 32u; m += 64u) reinterpret_cast<uint32_t *>(slots)[m] = 0u;
        }
#pragma unroll 1
        for (unsigned long long m = __ballot(hit); m; m &= m - 1) {
            const uint32_t src = (uint32_t)__builtin_ctzll(m);
            react_site_wave<L>(p, lat, s, lane_of(e, src), __uint_as_float(lane_of(__float_as_uint(a), src)), t, h3);
        }
    }
}

// What the resolver looks up and changes here: the particles on the chains of
// generation 1 (sweep tag `tag`), those past the block's capacity in the
// lattice.
template <class L>
struct ResidentSites {
    const Params &p;
    uint32_t *lat;
    ResidentLds &s;
    uint32_t tag;

    __device__ inline uint32_t key_of(uint32_t i) const
    {
        const uint32_t r = i / p.X, z = r / p.Y;
        return (i - r * p.X) | ((r - z * p.Y) << 10) | (z << 20);
    }
    // Record k of generation 0 joins its site's chain.
    __device__ inline void link(uint32_t k) const
    {
        const uint32_t key = s.key[0][k], old = atomicExch(&s.head[1][chain_of(key)], k | (tag << kIdBits));
        s.key[1][k] = key;
        s.next[1][k] = (uint16_t)((old >> kIdBits) == tag ? old & ((1u << kIdBits) - 1u) : kEnd);
    }
    __device__ inline uint32_t occupancy(uint32_t i) const
    {
        const uint32_t key = key_of(i), hd = s.head[1][chain_of(key)];
        uint32_t count = 0;
        for (uint32_t q = (hd >> kIdBits) == tag ? hd & ((1u << kIdBits) - 1u) : kEnd; q != kEnd; q = s.next[1][q])
            count += s.key[1][q] == key && s.key[0][q] != kDead ? 1u : 0u;
        if (s.spill)
            for (uint32_t k = 0; k < (uint32_t)L::W; k++) {
                const uint32_t v = load_agent(lat + (size_t)k * p.N + i);
                for (int b = 0; b < L::kPerWord; b++) count += L::part(v, b) != 0u ? 1u : 0u;
            }
        return count;
    }
    __device__ inline uint32_t look(bool in, uint32_t i) const
    {
        const uint32_t count = in ? occupancy(i) : (uint32_t)L::P;
        return count | ((uint32_t)L::P - count) << 8;
    }
    __device__ inline void place(uint32_t i, uint32_t slot, uint32_t particle) const
    {
        const uint32_t k = append<L>(p, lat, s, key_of(i), make_ord(slot, 0u, p.nST > 1u ? p.sites[i] : 0u, particle));
        if (k < kCap) link(k);
        else __threadfence();
    }
};

// The overflow entries of step t into sites with room; n: records before the
// reactions.  All threads call it.
template <class L>
__device__ inline void resolve_records(const Params &p, uint32_t *lat, ResidentLds &s, uint32_t t, uint32_t n, uint32_t tag)
{
    Control *ctl = p.ctl;
    const uint32_t tid = threadIdx.x;
    const ResidentSites<L> sites{p, lat, s, tag};
    __threadfence();  // entries, and particles past the block's capacity
    __syncthreads();
    const uint32_t found = load_agent(&ctl->ovf_count), carried = p.relaxed ? load_agent(&ctl->carry_count) : 0u;
    const unsigned long long key0 =
        __hip_atomic_load(&ctl->ovf_keys[tid & 63], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t part0 = load_agent(&ctl->ovf_part[tid & 63]);
    for (uint32_t k = n + tid; k < s.n[0] && k < kCap; k += kNT) sites.link(k);  // (appended by the reactions)
    __syncthreads();
    uint32_t kept = carried;
    if (found > kMaxOverflows || carried + found > kMaxOverflows) {
        if (tid == 0) {
            set_error(ctl, kErrOverflowCap, t);
            ctl->ovf_count = 0u;
        }
    } else if (found != 0u || carried != 0u) {
        // The keys take the chain heads of generation 0, free until the next
        // y sweep, which finds them zero.
        static_assert(sizeof(s.head[0]) >= kMaxOverflows * sizeof(unsigned long long), "room for the keys");
        kept = resolve_entries<(int)kNT>(p, sites, reinterpret_cast<unsigned long long *>(&s.head[0][0]), s.resolve, found,
                                         carried, t, key0, part0);
        __syncthreads();
        for (uint32_t k = tid; k < 2u * kMaxOverflows; k += kNT) s.head[0][k] = 0u;
    }
    if (tid == 0) s.ovf = p.relaxed && kept ? 1u : 0u;
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
    if (load_agent(&p.ctl->timestep) != job.start) return;
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
    if (load_agent(&ctl->timestep) != job.start) return;
    const uint32_t found = load_agent(job.count);
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
        s.ovf = p.relaxed && load_agent(&ctl->carry_count) ? 1u : 0u;
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
            if (s.ovf) resolve_records<L>(p, lat, s, t, n, tag + 3u);
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
