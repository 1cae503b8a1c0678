// The boxed MPD-RDME step for gfx950 (wave64): the x, y and z sweeps of one
// timestep in one launch, and the reaction tests, with work proportional to the
// particles instead of the sites.
//
// A block owns a box of 16 x TY x TZ sites and steps it together with a shell
// of one site on every side.  It reads word 0 and the site types of that
// region once, keeps a 32-bit record per particle in LDS (site, slot, where it
// came from, species) and sweeps the records:
//
//   x  every particle of the region moves; those with x inside the box stay
//   y  ... those with x and y inside the box stay
//   z  ... those of the box stay
//
// A particle's new slot is its rank among the particles that end the sweep on
// its site: stayers, then the minus neighbour's, then the plus neighbour's,
// each in old slot order.  Every particle joins its target's hash chain (one
// LDS exchange) and, after the block's barrier, counts who comes before it on
// the chain; nearly all are alone.  No neighbour site is ever looked up, one
// barrier per sweep suffices, and a site of many particles costs no branch of
// its own.  The shell is computed by every block that needs it and records
// nothing, so each overflow entry (phase, site, emission) is recorded once, by
// the box that owns the site, and every lattice is bit-identical to the
// separate sweeps'.
//
// Why: the separate sweeps spend their time on sites that hold nothing.  At
// the whole-cell occupancy (3% of the sites) they issue about 1150 vector
// instructions per 256 sites and step and move the lattice through memory
// three times.  Here a site costs a load, a test and a store, and a particle
// about 1000 instructions per 64.
//
// What bounds it (whole-cell 256x256x512, P = 8, 1e6 particles, rocprofv3): one
// launch 113 us against 303 us for the sweeps (x 77, y 105, z 119), 34.8e6
// vector instructions against 151e6, 0.32 GB of HBM traffic against 0.99 GB.  A
// block lives about 32000 cycles, a third of them the region's load; seven
// blocks of 20 KB LDS and 72 VGPRs share a CU, and vector issue takes 65 of the
// 113 us: latency of the dependent phases, then issue.  (Six blocks, with 1024 chains
// and the region's load in one go at 80 VGPRs: whole cell 117 us, 256x256x128
// uint32 lattice 52 -> 44; eight blocks: whole cell 112, but 96x96x96 with
// births 17.9 -> 19.0.)  Versions that kept a list of sites and
// looked each neighbour up in a site map took 244 us (a general path for
// sites of several particles ran in one wave while the others waited).
#include "lmx_batch.h"
#include "lmx_box.h"
#include "lmx_device.h"
#include "lmx_kernels.h"
#include "lmx_resolve.h"
#include "lmx_site.h"
#include "lmx_wave.h"

namespace lmx {

namespace {

constexpr uint32_t kNone = 0xFFFFFFFFu;
constexpr uint32_t kEnd = 0xFFFFu;       // end of a chain
// Hash chains of a sweep's targets (1024 of them keep P = 16's fuller boxes at
// 30.1 us on 128x64x80, 512 at 32.4).
constexpr uint32_t box_chains(int cap) { return cap > 768 ? 1024u : 512u; }

// A particle's record: its site's key (13 bits), slot (4), class (2: stayed,
// came from the minus neighbour, came from the plus neighbour) and, on the
// byte lattice, species (8).  A key is lx | ly << 5 | lz << 9: coordinates in
// the region, 0 and n+1 the shell, 1..n the box; key >> 5 is the row.  Slot
// and class together order the particles that end a sweep on one site: the
// stayers, then the minus neighbour's, then the plus neighbour's, each in slot
// order.
constexpr uint32_t kKeyMask = 0x1FFFu, kDead = 0x1FFFu;
__device__ inline uint32_t make_key(uint32_t lx, uint32_t ly, uint32_t lz) { return lx | (ly << 5) | (lz << 9); }
__device__ inline uint32_t rec_order(uint32_t rec) { return (rec >> 13) & 63u; }
__device__ inline uint32_t rec_slot(uint32_t rec) { return (rec >> 13) & 15u; }
template <uint32_t kChains>
__device__ inline uint32_t chain_of(uint32_t key)
{
    return (key ^ (key >> 4)) & (kChains - 1u);
}

template <class L, int CAP>
struct BoxLds {
    static constexpr uint32_t kChains = box_chains(CAP);
    // Sweeps alternate between two sets of records, chain links and chain
    // heads, so that a wave may begin the next sweep while others still rank
    // the particles of this one.
    uint32_t rec[2][CAP];
    uint32_t head[2][kChains];      // sweep tag << 16 | particle, the last one to join the chain
    uint16_t next[2][CAP];
    uint32_t sp[L::kPerWord == 1 ? CAP : 1];  // species (uint32 lattice)
    uint8_t typ[kMapN];             // region site types
    uint32_t xoff[32], row[256];    // x of lx, and site index of the row's x = 0 (wrapped)
    uint32_t ns, n, nc, base, nz[L::W];  // occupied sites; particles; candidates and their place; plane k holds a particle
};

// Region and box of one pass.
struct Box {
    uint32_t x0, y0, z0, nx, ny, nz;
};

__device__ inline uint32_t least(uint32_t a, uint32_t b) { return a < b ? a : b; }

// Occupied slots of a word: bit j = slot j.
template <class L>
__device__ inline uint32_t word_slots(uint32_t w)
{
    if constexpr (L::kPerWord == 4) {
        const uint32_t hi = (((w & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | w) & 0x80808080u;
        return ((hi >> 7) & 1u) | ((hi >> 14) & 2u) | ((hi >> 21) & 4u) | ((hi >> 28) & 8u);
    } else {
        return w != 0u ? 1u : 0u;
    }
}

// This lane's first slot for c < 32 entries: a ballot prefix inside the wave
// and one LDS reservation per wave.  Every lane of the wave calls it.
__device__ inline uint32_t wave_slots(uint32_t *counter, uint32_t c)
{
    uint32_t pre = 0, tot = 0;
    if (__ballot(c != 0u) == 0ull) return 0u;
#pragma unroll
    for (int b = 0; b < 5; b++) {
        const unsigned long long m = __ballot((c >> b) & 1u);
        pre += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u)) << b;
        tot += (uint32_t)__popcll(m) << b;
    }
    const uint32_t lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(counter, tot);
    return (uint32_t)__builtin_amdgcn_readfirstlane((int)base) + pre;
}

template <class L, int CAP>
struct BoxCtx {
    static constexpr uint32_t kChains = box_chains(CAP);
    const Params &p;
    BoxLds<L, CAP> &s;
    Box b;

    __device__ inline uint32_t at(uint32_t key) const { return (key & 31u) + 1u + kMapX * (key >> 5); }
    __device__ inline uint32_t site(uint32_t key) const { return s.xoff[key & 31u] + s.row[key >> 5]; }
    __device__ inline bool inner(uint32_t key) const
    {
        return (key & 31u) - 1u < b.nx && ((key >> 5) & 15u) - 1u < b.ny && (key >> 9) - 1u < b.nz;
    }
    __device__ inline uint32_t species(uint32_t rec, uint32_t e) const
    {
        if constexpr (L::kPerWord == 4) return rec >> 19;
        else return s.sp[e];
    }
    // The particles that end a sweep on the site of rec: how many come before
    // it, and how many there are.
    __device__ inline void rank(uint32_t par, uint32_t e, uint32_t rec, uint32_t &before, uint32_t &total) const
    {
        before = 0;
        total = 1;
        uint32_t q = s.head[par][chain_of<kChains>(rec & kKeyMask)] & 0xFFFFu;
        const uint32_t nx = s.next[par][e];
        if (q == e && nx == kEnd) return;
        total = 0;
        while (q != kEnd) {
            const uint32_t r = s.rec[par][q];
            q = s.next[par][q];
            if (((r ^ rec) & kKeyMask) == 0u) {
                total++;
                before += rec_order(r) < rec_order(rec) ? 1u : 0u;
            }
        }
    }
};

// One sweep axis: the key's shift and coordinate mask, the map stride, the
// extent of the box, its first coordinate, the lattice's extent and the
// step's hash.
struct Axis {
    uint32_t sh, cm, sm, n, g0, len;
    unsigned long long h;
};

// One pass over a box: a timestep of its particles up to the reactions.
// false: the region's particles did not fit CAP and nothing was written; the
// caller takes smaller boxes.  Plane k of the box is cleared if
// bit k of zero is set (it may hold an older state), nz_planes collects the
// planes that then hold something.
template <class L, int CAP, bool VEC>
__device__ __attribute__((always_inline)) inline bool box_pass(const BoxCtx<L, CAP> &c,
                                                               const uint32_t *__restrict__ src,
                                                               uint32_t *__restrict__ dst, const CandList &rl,
                                                               uint32_t shard, uint32_t t0, uint32_t zero,
                                                               uint32_t &nz_planes)
{
    constexpr int W = L::W;
    constexpr uint32_t P = L::P, kChains = box_chains(CAP);
    const Params &p = c.p;
    auto &s = c.s;
    const uint32_t tid = threadIdx.x;
    const Box b = c.b;
    const bool periodic = p.boundary == 0;

    __syncthreads();  // an earlier pass has left the LDS
    if (tid == 0) s.ns = s.n = s.nc = 0u;
    if (tid < (uint32_t)W) s.nz[tid] = 0u;
#pragma unroll
    for (uint32_t k = 0; k < 2u * kChains / (4u * kBoxThreads); k++)
        reinterpret_cast<uint4 *>(&s.head[0][0])[k * kBoxThreads + tid] = make_uint4(0u, 0u, 0u, 0u);

    // ---- 1. types of the region, keys of its occupied sites -------------------------
    // Rows of the region, 16 x 16: thread tid works out row tid; those past
    // the box's extent or a reflecting edge do not exist.
    {
        // wrapped coordinate of region coordinate l of an axis
        auto wrap = [](uint32_t g0, uint32_t l, uint32_t len) {
            uint32_t v = g0 + l;  // 1 + coordinate
            v = v == 0u ? len : v;
            v -= 1u;
            return v >= len ? v - len : v;
        };
        const uint32_t ly = tid & 15u, lz = tid >> 4;
        const bool ok = ly < b.ny + 2u && lz < b.nz + 2u &&
                        (periodic || (b.y0 + ly - 1u < p.Y && b.z0 + lz - 1u < p.Z));
        s.row[tid] = ok ? wrap(b.y0, ly, p.Y) * p.X + wrap(b.z0, lz, p.Z) * p.XY : kNone;
        if (tid < 32u) s.xoff[tid] = tid < b.nx + 2u && (periodic || b.x0 + tid - 1u < p.X) ? wrap(b.x0, tid, p.X) : kNone;
    }
    __syncthreads();
    // Columns 4 gx + 1 .. 4 gx + 4 of a row as one 16-byte load (VEC): U
    // groups a lane and round, z planes 4 apart, in flight together with the V
    // single sites (the two shell columns; without VEC every column, 32 lanes
    // a row, eight rows at a time).  A lane without a site loads the box's
    // first one, so that no load waits for a branch.
    constexpr uint32_t U = VEC ? 2 : 0, V = VEC ? 1 : 8, ROUNDS = VEC ? 2 : 4;
    const uint32_t gx = tid & 3u, gly = (tid >> 2) & 15u, glz = tid >> 6;
    const uint32_t lx = VEC ? ((tid & 1u) ? b.nx + 1u : 0u) : (tid & 31u);
    auto site_row = [&](uint32_t v) { return VEC ? (tid >> 1) + 128u * v : (tid >> 5) + 8u * v; };
    const uint32_t safe = b.x0 + b.y0 * p.X + b.z0 * p.XY;
#pragma unroll 1
    for (uint32_t r = 0; r < ROUNDS; r++) {
        uint4 v4[U ? U : 1];
        uint32_t t4[U ? U : 1], v1[V], t1[V];
        uint32_t ok = 0;  // bit u: group u exists; bit U + u: single site u
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            const uint32_t row = s.row[gly + 16u * (glz + 4u * (r * U + u))];
            const bool o = row != kNone && 4u * gx < b.nx;
            const uint32_t i = o ? b.x0 + 4u * gx + row : safe;
            v4[u] = *reinterpret_cast<const uint4 *>(src + i);
            t4[u] = *reinterpret_cast<const uint32_t *>(p.sites + i);
            ok |= (o ? 1u : 0u) << u;
        }
        const uint32_t xc = s.xoff[lx];
#pragma unroll
        for (uint32_t u = 0; u < V; u++) {
            const uint32_t row = s.row[site_row(r * V + u)];
            const bool o = row != kNone && xc != kNone;
            const uint32_t i = o ? xc + row : safe;
            v1[u] = src[i];
            t1[u] = p.sites[i];
            ok |= (o ? 1u : 0u) << (U + u);
        }
        uint32_t nz = 0;  // bit 4 u + q: site q of group u; bit 4 U + u: single site u
#pragma unroll
        for (uint32_t u = 0; u < U; u++) {
            if (!((ok >> u) & 1u)) continue;
            uint16_t *tp = reinterpret_cast<uint16_t *>(s.typ + c.at(make_key(1u + 4u * gx, gly, glz + 4u * (r * U + u))));
            tp[0] = (uint16_t)t4[u];
            tp[1] = (uint16_t)(t4[u] >> 16);
            uint4 q4 = v4[u];
            if (!p.packed) {  // a site may be occupied although its word 0 is empty
                const uint32_t i = b.x0 + 4u * gx + s.row[gly + 16u * (glz + 4u * (r * U + u))];
                for (uint32_t k = 1; k < (uint32_t)W; k++) {
                    const uint4 q = *reinterpret_cast<const uint4 *>(src + (size_t)k * p.N + i);
                    q4.x |= q.x;
                    q4.y |= q.y;
                    q4.z |= q.z;
                    q4.w |= q.w;
                }
            }
            nz |= ((q4.x != 0u ? 1u : 0u) | (q4.y != 0u ? 2u : 0u) | (q4.z != 0u ? 4u : 0u) | (q4.w != 0u ? 8u : 0u)) << (4 * u);
        }
#pragma unroll
        for (uint32_t u = 0; u < V; u++) {
            if (!((ok >> (U + u)) & 1u)) continue;
            const uint32_t row = site_row(r * V + u);
            s.typ[c.at(lx | (row << 5))] = (uint8_t)t1[u];
            uint32_t q = v1[u];
            if (!p.packed)
                for (uint32_t k = 1; k < (uint32_t)W; k++) q |= src[(size_t)k * p.N + xc + s.row[row]];
            nz |= (q != 0u ? 1u : 0u) << (4 * U + u);
        }
        uint32_t slot = wave_slots(&s.ns, (uint32_t)__builtin_popcount(nz));
        while (nz) {
            const uint32_t q = (uint32_t)__builtin_ctz(nz);
            nz &= nz - 1;
            const uint32_t key = q < 4u * U ? make_key(1u + 4u * gx + (q & 3u), gly, glz + 4u * U * r + (q & ~3u))
                                            : lx | (site_row(r * V + q - 4u * U) << 5);
            if (slot < (uint32_t)CAP) s.next[0][slot] = (uint16_t)key;
            slot++;
        }
    }
    __syncthreads();
    const uint32_t ns = s.ns;
    if (ns > (uint32_t)CAP) return false;

    // ---- 2. the particles of those sites (word 0 read again: it is in cache) ---------
    for (uint32_t e0 = 0; e0 < ns; e0 += kBoxThreads) {
        const uint32_t e = e0 + tid;
        uint32_t w[W], occ = 0, key = 0;
#pragma unroll
        for (int k = 0; k < W; k++) w[k] = 0u;
        if (e < ns) {
            key = s.next[0][e];
            const uint32_t i = c.site(key);
#pragma unroll
            for (int k = 0; k < W; k++) {
                if (k == 0 || L::need_next(p, w[k > 0 ? k - 1 : 0])) w[k] = src[(size_t)k * p.N + i];
                occ |= word_slots<L>(w[k]) << (L::kPerWord * k);
            }
        }
        uint32_t slot = wave_slots(&s.n, (uint32_t)__builtin_popcount(occ));
        while (occ) {
            const uint32_t j = (uint32_t)__builtin_ctz(occ);
            occ &= occ - 1;
            uint32_t part = w[0];
            if constexpr (L::kPerWord == 4) {
#pragma unroll
                for (int k = 1; k < W; k++) part = (j >> 2) == (uint32_t)k ? w[k] : part;
                part = (part >> (8 * (j & 3u))) & 0xFFu;
            } else {
#pragma unroll
                for (int k = 1; k < W; k++) part = j == (uint32_t)k ? w[k] : part;
            }
            if (slot < (uint32_t)CAP) {
                s.rec[1][slot] = key | (j << 13) | (L::kPerWord == 4 ? part << 19 : 0u);
                if constexpr (L::kPerWord == 1) s.sp[slot] = part;
            }
            slot++;
        }
    }
    __syncthreads();
    const uint32_t n = s.n;
    if (n > (uint32_t)CAP) return false;

    // ---- 3. sweeps --------------------------------------------------------------------
    // Round a ranks the particles that sweep a - 1 brought together on a site
    // (their new slots) and moves each along axis a: it joins its target's
    // chain.  Round 3 only ranks: the step's lattice before the reactions.
    const unsigned long long h3 = timestep_hash(p.seed32, t0, 3);
    const float2 *tab = reinterpret_cast<const float2 *>(p.prob1);
#pragma unroll 1
    for (uint32_t axis = 0; axis < 4; axis++) {
        Axis a;
        a.sh = axis == 0 ? 0u : (axis == 1 ? 5u : 9u);
        a.cm = axis == 0 ? 31u : 15u;
        a.sm = axis == 0 ? 1u : (axis == 1 ? kMapX : kMapX * 16u);
        a.n = axis == 0 ? b.nx : (axis == 1 ? b.ny : b.nz);
        a.g0 = axis == 0 ? b.x0 : (axis == 1 ? b.y0 : b.z0);
        a.len = axis == 0 ? p.X : (axis == 1 ? p.Y : p.Z);
        a.h = timestep_hash(p.seed32, t0, axis);
        const uint32_t to = axis & 1u, from = to ^ 1u;
        // Zeros over the box in the destination, late enough that their lines
        // are still in the L2 when the last round writes the particles.
        if (axis == 2 && zero) {
            if constexpr (VEC) {
                if (4u * gx < b.nx && gly - 1u < b.ny) {
#pragma unroll
                    for (uint32_t u = 0; u < 4u; u++) {
                        if (glz + 4u * u - 1u >= b.nz) continue;
                        const uint32_t i = b.x0 + 4u * gx + s.row[gly + 16u * (glz + 4u * u)];
#pragma unroll
                        for (int k = 0; k < W; k++)
                            if ((zero >> k) & 1u)
                                *reinterpret_cast<uint4 *>(dst + (size_t)k * p.N + i) = make_uint4(0u, 0u, 0u, 0u);
                    }
                }
            } else {
                const uint32_t zx = (tid & 15u) + 1u;
                for (uint32_t row = tid >> 4; row < 256u; row += 16u) {
                    if (zx > b.nx || (row & 15u) - 1u >= b.ny || (row >> 4) - 1u >= b.nz) continue;
                    const uint32_t i = b.x0 + zx - 1u + s.row[row];
#pragma unroll
                    for (int k = 0; k < W; k++)
                        if ((zero >> k) & 1u) dst[(size_t)k * p.N + i] = 0u;
                }
            }
        }
        for (uint32_t e = tid; e < n; e += kBoxThreads) {
            const uint32_t rec = s.rec[from][e], key = rec & kKeyMask;
            if (key == kDead) {
                if (axis < 3) s.rec[to][e] = kDead;
                continue;
            }
            uint32_t j = rec_slot(rec), total = 0;
            if (axis > 0) c.rank(from, e, rec, j, total);
            const uint32_t part = c.species(rec, e), i = c.site(key);
            if (j >= P) {  // no slot left: an overflow entry of the box that owns the site
                if (c.inner(key)) record_overflow(p.ctl, axis - 1u, i, j - P, part);
                if (axis < 3) s.rec[to][e] = kDead;
                continue;
            }
            const uint32_t idx = c.at(key), st = s.typ[idx];
            if (axis < 3) {
                // A site of the shell along the axis only sends particles
                // into the box; a reflecting edge has no neighbour.
                const uint32_t co = (key >> a.sh) & a.cm;
                const bool hm = co > 0u && (periodic || a.g0 + co > 1u);
                const bool hp = co <= a.n && (periodic || a.g0 + co < a.len);
                const uint32_t stm = s.typ[hm ? idx - a.sm : idx], stp = s.typ[hp ? idx + a.sm : idx];
                const float u = uniform01(i, p.pcb, j, a.h);
                const float qm = lookup_T_if(p, p.T, hm, part, st, stm);
                const float qp = lookup_T_if(p, p.T, hp, part, st, stp);
                const bool minus = u < qm, plus = !minus && u >= 0.5f && u < (qp + 0.5f);
                const uint32_t cn = co + (plus ? 1u : 0u) - (minus ? 1u : 0u);
                if (cn - 1u >= a.n) {  // outside the box along this axis
                    s.rec[to][e] = kDead;
                    continue;
                }
                const uint32_t target = key + ((cn - co) << a.sh);
                s.rec[to][e] = target | (j << 13) | ((plus ? 1u : (minus ? 2u : 0u)) << 17) |
                               (L::kPerWord == 4 ? part << 19 : 0u);
                const uint32_t tag = axis + 1u;
                const uint32_t old = atomicExch(&s.head[to][chain_of<kChains>(target)], e | (tag << 16));
                s.next[to][e] = (uint16_t)((old >> 16) == tag ? old & 0xFFFFu : kEnd);
            } else {
                if constexpr (L::kPerWord == 4)
                    reinterpret_cast<uint8_t *>(dst + (size_t)(j >> 2) * p.N + i)[j & 3u] = (uint8_t)part;
                else
                    dst[(size_t)j * p.N + i] = part;
                s.nz[L::kPerWord == 4 ? j >> 2 : j] = 1u;
                // A particle alone takes its reaction test from the table;
                // the sites that react and those of several particles are
                // evaluated by a launch of their own (its code needs twice
                // the registers of this kernel's).
                if (p.R > 0 && j == 0u) {
                    bool cand = total > 1u;
                    if (!cand) {
                        const float2 ap = tab[st * p.nS + (part - 1u)];
                        cand = ap.x != 0.0f && ap.y > 0.0f && uniform01(i, 1, 0, h3) <= ap.y;
                    }
                    if (cand) s.rec[1][atomicAdd(&s.nc, 1u)] = i;  // (that set of records is free in this round)
                }
            }
        }
        // The zeros are in place before any wave of the block writes over them.
        if (axis == 2) wait_for_stores();
        __syncthreads();
    }

    // Zero-order reactions can happen at an empty site: the ones that pass
    // the reaction test join the candidates.
    uint32_t nc = s.nc;
    if (p.any_qp0 && p.R > 0) {
        // kB sites a thread at once: one by one their table loads took 12K of
        // an active box's 33K cycles (expression 96x96x96: the launch 22.8 ->
        // 20.4 us).
        constexpr uint32_t kB = 4u;
        const uint32_t lx = (tid & 15u) + 1u, ly = tid >> 4;
        const bool column = lx <= b.nx && ly - 1u < b.ny;
#pragma unroll 1
        for (uint32_t lz0 = 1u; lz0 <= b.nz; lz0 += kB) {
            float prob[kB], q0[kB];
#pragma unroll
            for (uint32_t k = 0; k < kB; k++) {
                const bool in = column && lz0 + k <= b.nz;
                const uint32_t st = in ? s.typ[c.at(make_key(lx, ly, lz0 + k))] : 0u;
                prob[k] = p.prob0[st];
                q0[k] = p.qp0[st];
                if (!in) prob[k] = 0.0f;
            }
#pragma unroll
            for (uint32_t k = 0; k < kB; k++) {
                if (!(prob[k] > 0.0f && q0[k] != 0.0f)) continue;
                const uint32_t key = make_key(lx, ly, lz0 + k), i = c.site(key);
                if (!(uniform01(i, 1, 0, h3) <= prob[k])) continue;
                const uint32_t hd = s.head[0][chain_of<kChains>(key)];
                bool empty = true;
                for (uint32_t q = (hd >> 16) == 3u ? hd & 0xFFFFu : kEnd; q != kEnd; q = s.next[0][q])
                    if ((s.rec[0][q] & kKeyMask) == key) empty = false;
                if (!empty) continue;
                const uint32_t at = atomicAdd(&p.ctl->list_count[shard], 1u);
                if (at < rl.cap) rl.site[(size_t)shard * rl.cap + at] = i;
                else p.ctl->list_overflow = 1u;
            }
        }
    }
    if (nc) {
        if (tid == 0) s.base = atomicAdd(&p.ctl->list_count[shard], nc);
        __syncthreads();
        const uint32_t base = s.base;
        if (base + nc > rl.cap) {
            if (tid == 0) p.ctl->list_overflow = 1u;
        } else {
            for (uint32_t k = tid; k < nc; k += kBoxThreads) rl.site[(size_t)shard * rl.cap + base + k] = s.rec[1][k];
        }
    }
#pragma unroll
    for (int k = 0; k < W; k++)
        if (s.nz[k]) nz_planes |= 1u << k;
    return true;
}

// One box of a step: box number `logical` of the lattice.  zs and zd hold a
// flag per plane and box of the source and destination buffers: 1 while that
// plane of that box is known to be all zero.
template <class L, int CAP, bool VEC>
__device__ __attribute__((always_inline)) inline void box_body(const Params &p, const BoxGeom &g, const uint32_t *__restrict__ src,
                                uint32_t *__restrict__ dst, const uint32_t *__restrict__ zs, uint32_t *__restrict__ zd,
                                const CandList &rl, uint32_t t0, uint32_t logical, BoxLds<L, CAP> &lds)
{
    constexpr int W = L::W;
    const uint32_t r1 = fast_div(logical, g.div_nbx), bx = logical - r1 * g.nbx;
    const uint32_t bz = fast_div(r1, g.div_nby), by = r1 - bz * g.nby;
    const uint32_t lane = threadIdx.x & 63u;

    // Nothing in this box or its 26 neighbours (all known empty): no reads, and
    // no writes where the destination is known zero.  Lattices are packed
    // except right after an outside write, which clears the flags.
    bool empty = true;
    if (lane < 27u) {
        const uint32_t dz = lane / 9u, dy = (lane / 3u) % 3u, dx = lane % 3u;
        // 0, 1, 2: previous, own, next box, wrapped (beyond a reflecting edge the flag read is another box's: harmless)
        const uint32_t nx = dx == 1u ? bx : (dx == 0u ? (bx == 0u ? g.nbx - 1u : bx - 1u) : (bx + 1u == g.nbx ? 0u : bx + 1u));
        const uint32_t ny = dy == 1u ? by : (dy == 0u ? (by == 0u ? g.nby - 1u : by - 1u) : (by + 1u == g.nby ? 0u : by + 1u));
        const uint32_t nz = dz == 1u ? bz : (dz == 0u ? (bz == 0u ? g.nbz - 1u : bz - 1u) : (bz + 1u == g.nbz ? 0u : bz + 1u));
        empty = zs[nx + g.nbx * (ny + g.nby * nz)] != 0u;
    }
    uint32_t known = 0;
#pragma unroll
    for (int k = 0; k < W; k++) known |= (zd[(size_t)k * g.nboxes + logical] != 0u ? 1u : 0u) << k;
    const bool idle = __ballot(!empty) == 0ull && !(p.any_qp0 && p.R > 0);

    const uint32_t x0 = bx * kBoxX, y0 = by * g.TY, z0 = bz * g.TZ;
    const uint32_t nx = least(kBoxX, p.X - x0), ny = least(g.TY, p.Y - y0), nz = least(g.TZ, p.Z - z0);
    uint32_t planes = 0;
    BoxCtx<L, CAP> c{p, lds, Box{x0, y0, z0, nx, ny, nz}};
    if (idle) {
        if (known == (1u << W) - 1u) return;
        for (uint32_t it = threadIdx.x; it < nx * ny * nz; it += kBoxThreads) {
            const uint32_t row = it / nx, x = x0 + (it - row * nx);
            const uint32_t z = z0 + row / ny, y = y0 + row % ny;
            for (int k = 0; k < W; k++) dst[(size_t)k * p.N + x + p.X * y + p.XY * z] = 0u;
        }
    } else {
        // One pass over the whole box; a box too crowded for that is halved
        // along y and z, and a half that still is, cut into boxes whose
        // regions always fit (box_sub).
        constexpr BoxSub sub = box_sub(CAP, L::P);
        const Box whole = c.b;
        Box half = c.b;
        uint32_t level = 0, zero = ~known;
        // The box after o inside w, in steps of (dx, dy, dz); false after the last.
        auto advance = [](Box &o, const Box &w, uint32_t dx, uint32_t dy, uint32_t dz) -> bool {
            uint32_t x = o.x0 - w.x0 + dx, y = o.y0 - w.y0, z = o.z0 - w.z0;
            if (x >= w.nx) {
                x = 0;
                y += dy;
            }
            if (y >= w.ny) {
                y = 0;
                z += dz;
            }
            if (z >= w.nz) return false;
            o = Box{w.x0 + x, w.y0 + y, w.z0 + z, least(dx, w.nx - x), least(dy, w.ny - y), least(dz, w.nz - z)};
            return true;
        };
        auto first = [](const Box &w, uint32_t dx, uint32_t dy, uint32_t dz) {
            return Box{w.x0, w.y0, w.z0, least(dx, w.nx), least(dy, w.ny), least(dz, w.nz)};
        };
        const uint32_t hy = (ny + 1u) / 2u, hz = (nz + 1u) / 2u;
        for (;;) {
            const bool done = box_pass<L, CAP, VEC>(c, src, dst, rl, logical % (uint32_t)kListShards, t0, zero, planes);
            if (!done && level < 2u) {
                if (level == 0u && threadIdx.x == 0) atomicAdd(&p.ctl->box_splits, 1u);
                level++;
                zero = ~0u;  // nothing is left out in parts of a box
                if (level == 1u) c.b = half = first(whole, nx, hy, hz);
                else c.b = first(half, sub.x, sub.y, sub.z);
                continue;
            }
            if (level == 0u) break;
            if (level == 2u) {
                if (advance(c.b, half, sub.x, sub.y, sub.z)) continue;
                level = 1u;
            }
            if (!advance(half, whole, nx, hy, hz)) break;
            c.b = half;
        }
    }
    __syncthreads();  // every wave has read the flags
    if (threadIdx.x < (uint32_t)W) {
        const uint32_t k = threadIdx.x, f = (planes >> k) & 1u ? 0u : 1u;
        if (f != ((known >> k) & 1u)) zd[(size_t)k * g.nboxes + logical] = f;
    }
}

}  // namespace

template <class L, int CAP, bool VEC, int OCC>
__global__ __launch_bounds__(kBoxThreads, OCC) void box_step_kernel(Params p, BoxGeom g, const uint32_t *__restrict__ src,
                                                                    uint32_t *__restrict__ dst,
                                                                    const uint32_t *__restrict__ zs,
                                                                    uint32_t *__restrict__ zd, CandList rl)
{
    __shared__ BoxLds<L, CAP> lds;
    // Block b runs on XCD b % 8: chunks of neighbouring boxes go to the XCDs
    // in turn, so that an XCD's boxes share shells in its L2 while every XCD
    // gets its part of the crowded regions.
    const uint32_t q = blockIdx.x >> 3, ch = fast_div(q, g.div_chunk);
    const uint32_t logical = (ch * 8u + (blockIdx.x & 7u)) * g.chunk + (q - ch * g.chunk);
    if (logical >= g.nboxes) return;
    box_body<L, CAP, VEC>(p, g, src, dst, zs, zd, rl, p.ctl->timestep, logical, lds);
}

// The boxes of a batch's members in one launch: map gives a block's member.
template <class L, int CAP, int OCC>
__global__ __launch_bounds__(kBoxThreads, OCC) void box_jobs_kernel(const BoxJob *__restrict__ jobs,
                                                                    const uint32_t *__restrict__ map)
{
    __shared__ BoxLds<L, CAP> lds;
    const BoxJob &job = jobs[map[blockIdx.x]];
    const Params &p = job.p;
    const BoxGeom &g = job.g;
    const uint32_t b = blockIdx.x - job.first_box;  // (a multiple of 8 before it: the XCD order holds)
    const uint32_t q = b >> 3, ch = fast_div(q, g.div_chunk);
    const uint32_t logical = (ch * 8u + (b & 7u)) * g.chunk + (q - ch * g.chunk);
    if (logical >= g.nboxes) return;
    box_body<L, CAP, true>(p, g, job.src, job.dst, job.zs, job.zd, job.cand, p.ctl->timestep, logical, lds);
}

// ---------------------------------------------------------------------------
// Reaction phase of the candidate sites that the boxes listed, one wave per
// shard, and the step's overflow resolution by the block that ends last.  A
// shard that ran out makes it the full pass.
//
// The launch is latency: a candidate's chain of dependent loads.  So the table
// entries of a site's particles are loaded together, and a reacting site
// (checkForReaction decides it lane by lane) is taken by the whole wave: a
// slot per lane to count and evaluate, a reaction per lane to select.  The
// loops over slots are rolled, which keeps the kernel at 13 kB of code (71 kB
// unrolled), and a shard's entries are dealt to four waves, so that its
// reacting sites rarely queue behind one another.  Measured, with the
// resolver (a launch of its own before): whole cell 256x256x512 27.0 -> 15.3
// us, 256x256x128 uint32 lattice 21 -> 13.4, crowded P = 16 26 -> 15.4.
// ---------------------------------------------------------------------------

// A reaction at lane src's site i (propensity a, words w), by the whole wave.
// Every lane of the wave calls it, with its own site's values.
template <class L>
__device__ inline void wave_react(const Params &p, uint32_t *__restrict__ lat, uint32_t src, uint32_t i, uint32_t st,
                                  const uint32_t *w, float a, unsigned long long h3)
{
    constexpr uint32_t P = L::P;
    const uint32_t lane = lane_id();
    const uint32_t si = lane_of(i, src), sst = lane_of(st, src);
    // Lane j < P holds slot j.
    uint32_t word = 0;
#pragma unroll
    for (uint32_t k = 0; k < (uint32_t)L::W; k++) {
        const uint32_t v = lane_of(w[k], src);
        if (lane / L::kPerWord == k) word = v;
    }
    const uint32_t mine = lane >= P ? 0u : L::part(word, L::kPerWord == 1 ? 0 : (int)(lane & 3u));
    bool underflow = false;
    const uint32_t now = wave_products<P>(p, si, sst, mine, __uint_as_float(lane_of(__float_as_uint(a), src)), h3, underflow);
    if (underflow && lane == 0u && atomicCAS(&p.ctl->error, 0u, kErrReactionUnderflow) == 0u)
        p.ctl->error_step = p.ctl->timestep;
    // Device-scope stores: the last block may resolve overflow entries beside them.
    if (lane < P && now != mine) {
        if constexpr (L::kPerWord == 1)
            __hip_atomic_store(lat + (size_t)lane * p.N + si, now, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else
            __hip_atomic_store(reinterpret_cast<uint8_t *>(lat + (size_t)(lane >> 2) * p.N + si) + (lane & 3u), (uint8_t)now,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (now != 0u) clear_zero_flag(p, lane / L::kPerWord, si);
    }
}

// Block `block` of a solver's nblocks.
template <class L>
__device__ __attribute__((always_inline)) inline void cand_react_body(const Params &p, uint32_t *__restrict__ lat,
                                                                      const CandList &rl, uint32_t block, uint32_t nblocks)
{
    constexpr int W = L::W;
    constexpr uint32_t P = L::P;
    __shared__ uint32_t slots[kReactThreads / 64][P][64];
    Control *ctl = p.ctl;
    const unsigned long long h3 = timestep_hash(p.seed32, ctl->timestep, 3);
    const bool full = ctl->list_overflow != 0u;
    const uint32_t shard = block * kReactShards + threadIdx.x / kShardThreads, rank = threadIdx.x % kShardThreads;
    const uint32_t n = full ? p.N : ctl->list_count[shard];
    const uint32_t first = full ? shard * kShardThreads : 0u, step = full ? nblocks * kReactThreads : kShardThreads;
#pragma unroll 1
    for (uint32_t k0 = first; k0 < n; k0 += step) {
        // (a wave of the shard takes every kShardWaves-th entry, so that the
        // sites that react are spread over them)
        const uint32_t k = k0 + (rank & 63u) * kShardWaves + (rank >> 6);
        uint32_t i = 0, st = 0, w[W];
        float a = 0.0f;
        bool hit = false;
#pragma unroll
        for (int q = 0; q < W; q++) w[q] = 0u;
        if (k < n) {
            i = full ? k : rl.site[(size_t)shard * rl.cap + k];
            st = p.sites[i];
#pragma unroll
            for (int q = 0; q < W; q++)
                if (q == 0 || L::need_next(p, w[q > 0 ? q - 1 : 0])) w[q] = lat[(size_t)q * p.N + i];
            uint32_t count = 0;
#pragma unroll
            for (int j = 0; j < (int)P; j++) count += L::slot(w, j) != 0u ? 1u : 0u;
            float prob = 0.0f;
            const float u = uniform01(i, 1, 0, h3);
            if (count == 0u) {
                a = p.qp0[st];
                prob = p.prob0[st];
            } else if (count == 1u) {
                const float2 ap = reinterpret_cast<const float2 *>(p.prob1)[st * p.nS + (L::slot(w, 0) - 1u)];
                a = ap.x;
                prob = ap.y;
            } else {
                if (count == 2u) {
                    const uint32_t r1 = st * p.nS + (L::slot(w, 0) - 1u), s2 = L::slot(w, 1) - 1u;
                    const float q0 = p.qp0[st], q1 = p.qp1[r1], q12 = p.qp2[r1 * p.nS + s2], q2 = p.qp1[st * p.nS + s2];
                    a = q0;
                    a += q1;
                    a += q12;
                    a += q2;
                } else {
#pragma unroll
                    for (int j = 0; j < (int)P; j++) slots[threadIdx.x >> 6][j][rank & 63u] = L::slot(w, j);
                    a = packed_propensity<P>(p, st, slots[threadIdx.x >> 6], rank & 63u, count);
                }
                // 1 - exp(-a) <= a, with room for the rounding of both (u is
                // 0 or at least 2^-32): most sites need no exponential
                if (a != 0.0f && u <= a * 1.0001f) prob = reaction_probability(a);
            }
            hit = a != 0.0f && prob > 0.0f && u <= prob;
        }
#pragma unroll 1
        for (unsigned long long m = __ballot(hit); m; m &= m - 1)
            wave_react<L>(p, lat, (uint32_t)__builtin_ctzll(m), i, st, w, a, h3);
    }
    // The block that ends last resolves the step's overflow entries.
    __shared__ uint32_t last;
    // (What it reads of this launch, lattice words and entries, is stored and
    // loaded at device scope, so waiting for the stores is enough: no fence,
    // which would write back and invalidate the L2.)
    wait_for_stores();  // every wave's have arrived
    __syncthreads();
    if (threadIdx.x == 0) last = atomicAdd(&ctl->blocks_done, 1u) == nblocks - 1u ? 1u : 0u;
    __syncthreads();
    if (!last) return;
    if (threadIdx.x == 0) ctl->blocks_done = 0u;
    resolve_body<kReactThreads>(p, lat);
}

template <class L>
__global__ __launch_bounds__(kReactThreads) void cand_react_kernel(Params p, uint32_t *__restrict__ lat, CandList rl)
{
    cand_react_body<L>(p, lat, rl, blockIdx.x, gridDim.x);
}

// A batch's members after box_jobs_kernel's same step.
template <class L>
__global__ __launch_bounds__(kReactThreads) void cand_react_jobs_kernel(const BoxJob *__restrict__ jobs,
                                                                        const uint32_t *__restrict__ map)
{
    const BoxJob &job = jobs[map[blockIdx.x]];
    cand_react_body<L>(job.p, job.dst, job.cand, blockIdx.x - job.first_react, job.react_blocks);
}

template <class L, int CAP, int OCC>
static hipError_t launch_box(const Params &p, const BoxGeom &g, const uint32_t *src, uint32_t *dst, const uint32_t *zs,
                             uint32_t *zd, const CandList &rl, hipStream_t st)
{
    const dim3 grid(box_blocks(g)), block(kBoxThreads);
    if ((p.X & 3u) == 0)
        hipLaunchKernelGGL((box_step_kernel<L, CAP, true, OCC>), grid, block, 0, st, p, g, src, dst, zs, zd, rl);
    else
        hipLaunchKernelGGL((box_step_kernel<L, CAP, false, OCC>), grid, block, 0, st, p, g, src, dst, zs, zd, rl);
    return hipGetLastError();
}

hipError_t launch_box_reactions(const Params &p, const BoxGeom &g, uint32_t *lat, const CandList &rl, hipStream_t st)
{
    Params q = p;
    q.packed = 1u;  // the step has packed every site
    const dim3 grid(box_react_blocks(g)), block(kReactThreads);
    switch (p.word_particles ? 100 + (int)p.P : (int)p.W) {
    case 1: hipLaunchKernelGGL((cand_react_kernel<ByteSites<1>>), grid, block, 0, st, q, lat, rl); break;
    case 2: hipLaunchKernelGGL((cand_react_kernel<ByteSites<2>>), grid, block, 0, st, q, lat, rl); break;
    case 4: hipLaunchKernelGGL((cand_react_kernel<ByteSites<4>>), grid, block, 0, st, q, lat, rl); break;
    case 104: hipLaunchKernelGGL((cand_react_kernel<WordSites<4>>), grid, block, 0, st, q, lat, rl); break;
    case 108: hipLaunchKernelGGL((cand_react_kernel<WordSites<8>>), grid, block, 0, st, q, lat, rl); break;
    case 116: hipLaunchKernelGGL((cand_react_kernel<WordSites<16>>), grid, block, 0, st, q, lat, rl); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_box_step(const Params &p, const BoxGeom &g, const uint32_t *src, uint32_t *dst, const uint32_t *zs,
                           uint32_t *zd, const CandList &rl, hipStream_t st)
{
    // Waves per SIMD: the most without a spill, but for the uint32 lattice's 8
    // and 16 slots, which spill 3 and 6 VGPRs.  (With one wave fewer each they
    // spill none and take 128x128x256 with a crowded spot from 125 to 139 and
    // from 189 to 232 us a step.)
    const int key = p.word_particles ? 100 + (int)p.P : (int)p.W;
    switch (key) {
    case 1: return launch_box<ByteSites<1>, box_cap(4), 7>(p, g, src, dst, zs, zd, rl, st);
    case 2: return launch_box<ByteSites<2>, box_cap(8), 7>(p, g, src, dst, zs, zd, rl, st);
    case 4: return launch_box<ByteSites<4>, box_cap(16), 6>(p, g, src, dst, zs, zd, rl, st);
    case 104: return launch_box<WordSites<4>, box_cap(4), 6>(p, g, src, dst, zs, zd, rl, st);
    case 108: return launch_box<WordSites<8>, box_cap(8), 6>(p, g, src, dst, zs, zd, rl, st);
    case 116: return launch_box<WordSites<16>, box_cap(16), 4>(p, g, src, dst, zs, zd, rl, st);
    }
    return hipErrorInvalidValue;
}

template <int W, int OCC>
static void launch_jobs(const BoxJob *jobs, const uint32_t *map, uint32_t boxes, uint32_t reacts, hipStream_t st)
{
    hipLaunchKernelGGL((box_jobs_kernel<ByteSites<W>, box_cap(4 * W), OCC>), dim3(boxes), dim3(kBoxThreads), 0, st, jobs, map);
    hipLaunchKernelGGL((cand_react_jobs_kernel<ByteSites<W>>), dim3(reacts), dim3(kReactThreads), 0, st, jobs, map + boxes);
}

hipError_t launch_box_jobs(const BoxJob *jobs, const uint32_t *map, uint32_t boxes, uint32_t reacts, uint32_t W, hipStream_t st)
{
    switch (W) {
    case 1: launch_jobs<1, 7>(jobs, map, boxes, reacts, st); break;
    case 2: launch_jobs<2, 7>(jobs, map, boxes, reacts, st); break;
    case 4: launch_jobs<4, 6>(jobs, map, boxes, reacts, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace lmx
