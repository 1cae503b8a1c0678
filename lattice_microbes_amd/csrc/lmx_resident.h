// The resident step (mpd_resident.hip): a small solver's particles kept in one
// block's LDS over many timesteps.
#pragma once

#include <stdint.h>

#include "lmx_device.h"

namespace lmx {

// Particles a block holds, and the most a solver may be expected to hold to be
// run this way (the rest is room for reactions and fluctuations).
constexpr uint32_t kResidentCap = 4096u, kResidentMost = 3000u;
constexpr uint32_t kResidentThreads = 1024u;
constexpr uint32_t kResidentMaxEdge = 1024u;   // a coordinate fits ten bits
constexpr uint32_t kResidentMaxSteps = 65536u; // of one launch (sweep tags of the chains)

// One solver's run: nsteps from step start, if its step counter stands there
// (an earlier run that stopped short leaves it behind, and nothing is done).
struct ResidentJob {
    Params p;
    uint32_t *lat;         // the lattice, emptied into the list and written back in place
    uint2 *list;           // particles: {site, slot | species << 8}, kResidentCap of them
    uint32_t *count;       // particles found (0 between runs)
    uint32_t start, nsteps;
};

}  // namespace lmx
