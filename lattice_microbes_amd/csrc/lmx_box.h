// Geometry of the boxed step (mpd_box.hip): the lattice cut into boxes of
// TX x TY x TZ sites, one block each.
#pragma once

#include <stdint.h>

#include <algorithm>

#include "lmx_batch.h"
#include "lmx_device.h"

namespace lmx {

constexpr uint32_t kBoxThreads = 256u;

// A box and its shell are 16 x 16 rows of 18 sites, so that a thread's rows
// and the site -> entry map need shifts and constants only: boxes of 16 sites
// along x and at most 14 along y and z.
constexpr uint32_t kBoxX = 16u, kBoxMaxYZ = 14u;
constexpr uint32_t kMapX = kBoxX + 4u;      // map entries per row: the box's first column lies at index 2
                                            // (its types are stored as 16-bit pairs)
constexpr uint32_t kMapN = kMapX * 256u;

// Sites whose reactions are evaluated after the boxed step: shard s holds
// site indices [s*cap, s*cap + list_count[s]); box b appends to shard
// b % kListShards.
struct CandList {
    uint32_t *site;
    uint32_t cap;
};

struct BoxGeom {
    uint32_t TY, TZ;                  // box extents (smaller at the lattice's far edges)
    uint32_t nbx, nby, nbz, nboxes;
    uint32_t chunk;                   // neighbouring boxes that one XCD takes in turn
    FastDiv div_chunk, div_nbx, div_nby;
};

// Boxes of at most most sites along y and z, of equal extents.
inline BoxGeom box_geom(uint32_t X, uint32_t Y, uint32_t Z, uint32_t most)
{
    auto even = [most](uint32_t len) {
        const uint32_t nb = (len + most - 1) / most;
        return (len + nb - 1) / nb;
    };
    BoxGeom g{};
    const uint32_t TY = g.TY = even(Y), TZ = g.TZ = even(Z);
    g.nbx = (X + kBoxX - 1) / kBoxX;
    g.nby = (Y + TY - 1) / TY;
    g.nbz = (Z + TZ - 1) / TZ;
    g.nboxes = g.nbx * g.nby * g.nbz;
    g.chunk = std::min(std::max(g.nboxes / 64u, 1u), g.nbx * g.nby);
    g.div_chunk = make_fastdiv(g.chunk);
    g.div_nbx = make_fastdiv(g.nbx);
    g.div_nby = make_fastdiv(g.nby);
    return g;
}

// Blocks of the boxed step's two launches.
constexpr uint32_t kReactThreads = 1024u, kShardWaves = 4u, kShardThreads = 64u * kShardWaves,
                   kReactShards = kReactThreads / kShardThreads;
inline uint32_t box_blocks(const BoxGeom &g)
{
    return (g.nboxes + 8u * g.chunk - 1u) / (8u * g.chunk) * 8u * g.chunk;
}
inline uint32_t box_react_blocks(const BoxGeom &g)
{
    return (std::min(g.nboxes, (uint32_t)kListShards) + kReactShards - 1u) / kReactShards;
}

// A step of a batch's member in boxes.  A run has three sets of jobs: its first
// step (which may read an unpacked lattice), the odd ones and the later even
// ones.
constexpr uint32_t kBoxJobSets = 3u;
__host__ __device__ inline uint32_t box_job_set(uint32_t step) { return step == 0u ? 0u : 2u - (step & 1u); }
struct BoxJob {
    Params p;
    BoxGeom g;
    const uint32_t *src, *zs;
    uint32_t *dst, *zd;
    CandList cand;
    uint32_t first_box, first_react, react_blocks;  // its blocks of the two launches
};

// Particles a box's region may hold (its records are kept in LDS).
constexpr int box_cap(uint32_t P) { return P == 16 ? 1024 : 768; }

// Box extents along y and z, from the largest; the largest whose regions fit
// the lattice's particles is taken (plan_boxes).
constexpr uint32_t kBoxLevels = 5u;
constexpr uint32_t kBoxLevel[kBoxLevels] = {kBoxMaxYZ, 10u, 8u, 6u, 4u};

// Boxes whose region always fits cap particles, if every slot of its
// (x+2)(y+2)(z+2) sites were occupied.
struct BoxSub {
    uint32_t x, y, z;
};
constexpr bool box_sub_fits(BoxSub s, uint32_t cap, uint32_t P)
{
    return (s.x + 2u) * (s.y + 2u) * (s.z + 2u) * P <= cap;
}
constexpr BoxSub box_sub(uint32_t cap, uint32_t P)
{
    return box_sub_fits({4, 2, 2}, cap, P) ? BoxSub{4, 2, 2} : BoxSub{4, 1, 1};
}
static_assert(box_sub_fits(box_sub(box_cap(4), 4), box_cap(4), 4) &&
                  box_sub_fits(box_sub(box_cap(8), 8), box_cap(8), 8) &&
                  box_sub_fits(box_sub(box_cap(16), 16), box_cap(16), 16),
              "the fallback boxes must fit");

}  // namespace lmx
