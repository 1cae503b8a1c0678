// Host-side launchers of the MPD-RDME kernels (implemented in mpd_kernels.hip).
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

#include "lmx_device.h"

namespace lmx {

struct Params;
struct Member;
struct BoxGeom;

hipError_t launch_sweep(const Params &p, const uint32_t *src, uint32_t *dst, int axis, hipStream_t st);
hipError_t launch_reaction(const Params &p, uint32_t *lat, hipStream_t st);
hipError_t launch_resolve(const Params &p, uint32_t *lat, hipStream_t st);
bool fast_path_ok(const Params &p);
hipError_t launch_sweep_fast(const Params &p, const uint32_t *src, uint32_t *dst, int axis, uint32_t seg,
                             hipStream_t st);
bool col_ok(const Params &p, int axis, uint32_t seg);
hipError_t launch_sweep_col(const Params &p, const uint32_t *src, uint32_t *dst, int axis, uint32_t seg,
                            hipStream_t st);
hipError_t launch_sweep_tile(const Params &p, const uint32_t *src, uint32_t *dst, int axis, bool react,
                             const ReactionList &rl, hipStream_t st);
hipError_t launch_sweep_sparse(const Params &p, const uint32_t *src, uint32_t *dst, int axis, bool react,
                               const ReactionList &rl, hipStream_t st);
hipError_t launch_reaction_list(const Params &p, uint32_t *lat, const ReactionList &rl, int num_cu, hipStream_t st);
// The static reaction list (lmx_run_steps_static): kListShards shards of
// kStaticListCap entries in a device array of the library; `device` must be
// current.  Lattices of up to kStaticListMaxSites sites use it.
constexpr uint32_t kStaticListCap = 256;
constexpr size_t kStaticListMaxSites = (size_t)kListShards * kStaticListCap * 8;
constexpr int kMaxDevices = 64;
hipError_t static_reaction_list(int device, uint32_t W, ReactionList *out);
bool fused_ok(const Params &p);
uint32_t fused_tile_rows(uint32_t X, uint32_t W);
hipError_t launch_fused(const Params &p, const uint32_t *src, uint32_t *dst, uint32_t zseg, hipStream_t st);
hipError_t launch_reaction_fast(const Params &p, uint32_t *lat, hipStream_t st);
hipError_t launch_prob_tables(const Params &p, float *prob1, float *prob0, hipStream_t st);
// The boxed step (mpd_box.hip): one timestep from src to dst without the
// reactions and the overflow resolution, which are launch_box_reactions's (a
// model without reactions takes launch_resolve instead).  zs and zd are the
// zero flags of the two buffers, rl the reaction candidates (any capacity is
// correct).
struct CandList;
hipError_t launch_box_step(const Params &p, const BoxGeom &g, const uint32_t *src, uint32_t *dst, const uint32_t *zs,
                           uint32_t *zd, const CandList &rl, hipStream_t st);
hipError_t launch_box_reactions(const Params &p, const BoxGeom &g, uint32_t *lat, const CandList &rl, hipStream_t st);
// A step of a batch's boxed members (byte lattice of W words, X % 4 == 0): all
// their boxes in one launch, then all their reactions and overflow entries.
// jobs: the step's set; map: the member of each of the boxes, then of each of
// the reacts blocks.
struct BoxJob;
hipError_t launch_box_jobs(const BoxJob *jobs, const uint32_t *map, uint32_t boxes, uint32_t reacts, uint32_t W, hipStream_t st);
// Resident runs (mpd_resident.hip) of n solvers of one layout: a single job by
// value (jobs null) or n jobs in device memory, each gathered by `per` blocks.
struct ResidentJob;
uint32_t resident_gather_blocks(uint32_t N);
hipError_t launch_resident(const ResidentJob &one, const ResidentJob *jobs, uint32_t n, uint32_t per, uint32_t P,
                           bool words, hipStream_t st);
uint32_t x4_blocks(const Params &p);
uint32_t reaction_blocks(const Params &p);
struct TileGeom;
uint32_t batch_list_shards(const TileGeom &zgeo, uint32_t threads);
constexpr uint32_t kBatchListBlockSites = 1u << 22;
bool batch_list_by_block(uint32_t sites);
uint32_t batch_list_blocks(uint32_t nshards, uint32_t sites);
// One batched step without the resolver: x, y, z sweeps and (if total[3] > 0)
// the reaction phase.  For launch k (x, y, z, reaction), start[k] is a device
// prefix array of n+1 block offsets and map[k] a device array of total[k]
// member indices (block b belongs to member map[k][b]); total[] holds the
// four grid sizes.
// Tiled sweeps in blocks of tile_threads (a multiple of 64, at most
// tile_threads_for(W)), the size the members' tile geometry was made for.
hipError_t launch_batch_sweeps(const Member *m, const uint32_t *const start[4], const uint32_t *const map[4],
                               uint32_t n, const uint32_t *total, uint32_t W, uint32_t tile_threads, hipStream_t st);
hipError_t launch_batch_resolve(Member *m, uint32_t n, hipStream_t st);
hipError_t launch_copy(const void *src, void *dst, size_t bytes, int num_cu, hipStream_t st);
hipError_t launch_fill(uint32_t *ptr, size_t n, uint32_t value, hipStream_t st);
hipError_t launch_validate(const Params &p, const uint32_t *lat, hipStream_t st);
// Species counts of nwords lattice words to host memory (out, nS entries);
// counts: nS + 1 zeroed device words, left zeroed.
hipError_t launch_counts(const uint32_t *lat, size_t nwords, uint32_t nS, bool words, uint32_t *counts, uint32_t *out,
                         hipStream_t st);
// The first kReportWords words of up to kReportMost control blocks to host
// memory, kReportWords apart.
constexpr uint32_t kReportWords = 16u, kReportMost = 256u;
static_assert(offsetof(Control, box_splits) / sizeof(uint32_t) < kReportWords, "the report ends with box_splits");
struct ReportList {
    const Control *ctl[kReportMost];
    uint32_t n;
};
hipError_t launch_report(const ReportList &c, uint32_t *out, hipStream_t st);
hipError_t launch_exp(const double *x, double *y, size_t n, hipStream_t st);
hipError_t launch_prob(const float *a, float *y, size_t n, hipStream_t st);

}  // namespace lmx
