// Test infrastructure: a stand-in for the HIP runtime and for the library's
// kernels, so that the host side of the library (mpd_capi.cpp) runs without a
// GPU.  Device memory is host memory, streams do nothing, and a launch only
// advances the step counter of its solver and leaves a line in a log:
//
//   box | sweep | fused t=<step> packed=<0,1> N=<sites> R=<reactions>
//   resident t=<step> steps=<asked> packed=<0,1>
//   sync | copy | device      waits, blocking copies, hipSetDevice
//   report | tables           the control blocks' report, new probability tables
//
// A resident run stops after `limit` steps, as one whose block is full.
#include <hip/hip_runtime.h>

#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>

#include "lmx_batch.h"
#include "lmx_box.h"
#include "lmx_device.h"
#include "lmx_kernels.h"
#include "lmx_resident.h"

namespace {

std::string g_log;
uint32_t g_limit = ~0u;
bool g_pinned_fails = false;
double g_clock = 0.0;                 // ms
std::map<std::string, double> g_cost;  // of a step, by the log's names
char g_handle;

void note(const std::string &line) { g_log += line + "\n"; }

void spend(const char *kind, double steps = 1.0)
{
    auto it = g_cost.find(kind);
    g_clock += steps * (it == g_cost.end() ? 1.0 : it->second);
}

void launched(const char *kind, const lmx::Params &p)
{
    spend(kind);
    note(std::string(kind) + " t=" + std::to_string(p.ctl->timestep) + " packed=" + std::to_string(p.packed) + " N=" +
         std::to_string(p.N) + " R=" + std::to_string(p.R));
}

void stepped(const lmx::Params &p) { p.ctl->timestep++; }

template <class T>
T *handle()
{
    return reinterpret_cast<T *>(&g_handle);
}

}  // namespace

extern "C" {
void standin_reset(void)
{
    g_log.clear();
    g_limit = ~0u;
    g_pinned_fails = false;
    g_cost.clear();
}
void standin_clear_log(void) { g_log.clear(); }
const char *standin_log(void) { return g_log.c_str(); }
void standin_resident_limit(uint32_t steps) { g_limit = steps; }
void standin_pinned_fails(int fails) { g_pinned_fails = fails != 0; }
void standin_cost(const char *kind, double ms) { g_cost[kind] = ms; }

// ---- runtime
hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipSetDevice(int d) { note("device " + std::to_string(d)); return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { note("sync"); return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipMalloc(void **p, size_t n) { *p = calloc(n ? n : 1, 1); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    if (g_pinned_fails) return hipErrorOutOfMemory;
    return hipMalloc(p, n);
}
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { note("copy"); memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { memset(p, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { memset(p, v, n); return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { *s = handle<ihipStream_t>(); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { note("sync"); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = reinterpret_cast<hipEvent_t>(new double(0.0)); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<double *>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { *reinterpret_cast<double *>(e) = g_clock; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    *ms = (float)(*reinterpret_cast<double *>(b) - *reinterpret_cast<double *>(a));
    return hipSuccess;
}
}  // extern "C"

// ---- kernels
namespace lmx {

hipError_t launch_sweep(const Params &p, const uint32_t *, uint32_t *, int axis, hipStream_t)
{
    if (axis == 0) launched("sweep", p);
    return hipSuccess;
}
hipError_t launch_sweep_fast(const Params &p, const uint32_t *s, uint32_t *d, int axis, uint32_t, hipStream_t st) { return launch_sweep(p, s, d, axis, st); }
hipError_t launch_sweep_col(const Params &p, const uint32_t *s, uint32_t *d, int axis, uint32_t, hipStream_t st) { return launch_sweep(p, s, d, axis, st); }
hipError_t launch_sweep_tile(const Params &p, const uint32_t *s, uint32_t *d, int axis, bool, const ReactionList &, hipStream_t st) { return launch_sweep(p, s, d, axis, st); }
hipError_t launch_sweep_sparse(const Params &p, const uint32_t *s, uint32_t *d, int axis, bool, const ReactionList &, hipStream_t st) { return launch_sweep(p, s, d, axis, st); }
hipError_t launch_reaction(const Params &, uint32_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_reaction_fast(const Params &, uint32_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_reaction_list(const Params &, uint32_t *, const ReactionList &, int, hipStream_t) { return hipSuccess; }
hipError_t launch_resolve(const Params &p, uint32_t *, hipStream_t) { stepped(p); return hipSuccess; }
hipError_t launch_fused(const Params &p, const uint32_t *, uint32_t *, uint32_t, hipStream_t) { launched("fused", p); return hipSuccess; }
bool fast_path_ok(const Params &p) { return !p.word_particles && (p.X & 3u) == 0 && p.N >= 4; }
bool col_ok(const Params &, int, uint32_t) { return true; }
bool fused_ok(const Params &p) { return fast_path_ok(p) && p.X <= 256u; }
uint32_t fused_tile_rows(uint32_t, uint32_t) { return 8u; }
uint32_t x4_blocks(const Params &) { return 8u; }
uint32_t reaction_blocks(const Params &) { return 8u; }
uint32_t batch_list_shards(const TileGeom &, uint32_t) { return 8u; }
bool batch_list_by_block(uint32_t) { return false; }
uint32_t batch_list_blocks(uint32_t, uint32_t) { return 8u; }
uint32_t resident_gather_blocks(uint32_t) { return 1u; }
hipError_t launch_prob_tables(const Params &, float *, float *, hipStream_t) { note("tables"); return hipSuccess; }

static uint4 g_static[16];
hipError_t static_reaction_list(int, uint32_t, ReactionList *out)
{
    *out = ReactionList{g_static, 1u};
    return hipSuccess;
}

hipError_t launch_box_step(const Params &p, const BoxGeom &, const uint32_t *, uint32_t *, const uint32_t *, uint32_t *,
                           const CandList &rl, hipStream_t)
{
    launched("box", p);
    if (rl.site == reinterpret_cast<uint32_t *>(g_static)) note("static list");
    return hipSuccess;
}
hipError_t launch_box_reactions(const Params &p, const BoxGeom &, uint32_t *, const CandList &, hipStream_t) { stepped(p); return hipSuccess; }

static hipError_t resident(const ResidentJob &j)
{
    Control *ctl = j.p.ctl;
    note("resident t=" + std::to_string(j.start) + " steps=" + std::to_string(j.nsteps) + " packed=" + std::to_string(j.p.packed));
    if (ctl->timestep != j.start) return hipSuccess;
    const uint32_t done = j.nsteps < g_limit ? j.nsteps : g_limit;
    ctl->timestep += done;
    spend("resident", done);
    return hipSuccess;
}
hipError_t launch_resident(const ResidentJob &one, const ResidentJob *jobs, uint32_t n, uint32_t, uint32_t, bool, hipStream_t)
{
    for (uint32_t k = 0; k < n; k++) resident(jobs ? jobs[k] : one);
    return hipSuccess;
}
hipError_t launch_box_jobs(const BoxJob *jobs, const uint32_t *map, uint32_t boxes, uint32_t, uint32_t, hipStream_t)
{
    for (uint32_t k = 0; k < boxes; k++)
        if (k == 0 || map[k] != map[k - 1]) {
            launched("box", jobs[map[k]].p);
            stepped(jobs[map[k]].p);
        }
    return hipSuccess;
}
hipError_t launch_batch_sweeps(const Member *m, const uint32_t *const *, const uint32_t *const *, uint32_t n, const uint32_t *,
                               uint32_t, uint32_t, hipStream_t)
{
    for (uint32_t k = 0; k < n; k++) launched("sweep", m[k].p);
    return hipSuccess;
}
hipError_t launch_batch_resolve(Member *m, uint32_t n, hipStream_t)
{
    for (uint32_t k = 0; k < n; k++) stepped(m[k].p);
    return hipSuccess;
}
hipError_t launch_copy(const void *s, void *d, size_t n, int, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t launch_fill(uint32_t *p, size_t n, uint32_t v, hipStream_t)
{
    while (n--) *p++ = v;
    return hipSuccess;
}
hipError_t launch_validate(const Params &, const uint32_t *, hipStream_t) { return hipSuccess; }
hipError_t launch_counts(const uint32_t *, size_t, uint32_t nS, bool, uint32_t *, uint32_t *out, hipStream_t)
{
    memset(out, 0, nS * sizeof(uint32_t));
    return hipSuccess;
}
hipError_t launch_report(const ReportList &c, uint32_t *out, hipStream_t)
{
    note(out ? "report" : "report to null");
    for (uint32_t k = 0; out && k < c.n; k++) memcpy(out + k * kReportWords, c.ctl[k], kReportWords * sizeof(uint32_t));
    return hipSuccess;
}
hipError_t launch_exp(const double *, double *, size_t, hipStream_t) { return hipSuccess; }
hipError_t launch_prob(const float *, float *, size_t, hipStream_t) { return hipSuccess; }

}  // namespace lmx
