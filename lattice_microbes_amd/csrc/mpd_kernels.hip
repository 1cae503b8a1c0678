// MPD-RDME step kernels for gfx950 (CDNA4, wave64).
//
//  sweep_kernel     one diffusion sweep along x, y or z, one site per thread,
//                   any shape (mpd_{x,y,z}_kernel, MpdRdmeSolver.cu:1342-1490)
//  reaction_kernel  per-site reaction, one site per thread, any shape
//                   (precomp_reaction_kernel, MpdRdmeSolver.cu:1592-1675)
//  resolve_kernel   canonical-order overflow placement on the device (the
//                   classic host handler, MpdRdmeSolver.cu:1103-1189, or the
//                   relaxed correct_overflows, :1677-1761)
//  count_kernel     species counts (ByteLattice::getParticleCounts,
//                   IntLattice::getParticleCounts)
//
// Every per-particle decision depends only on (site index, slot, timestep,
// substep) through the counter-based hash, so the results do not depend on
// how sites are distributed over threads.
#include <algorithm>

#include "lmx_batch.h"
#include "lmx_device.h"
#include "lmx_kernels.h"
#include "lmx_resolve.h"
#include "lmx_site.h"

namespace lmx {

// ---------------------------------------------------------------------------
// Generic sweep: one site per thread, any lattice shape (the vector kernels in
// mpd_fast.hip need X % 4 == 0).
// ---------------------------------------------------------------------------
template <class L>
__global__ __launch_bounds__(256) void sweep_kernel(Params p, const uint32_t *__restrict__ src,
                                                    uint32_t *__restrict__ dst, uint32_t stride,
                                                    uint32_t len, uint32_t substep)
{
    constexpr int W = L::W;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p.N) return;
    const unsigned long long h = timestep_hash(p.seed32, p.ctl->timestep, substep);
    const uint32_t c = (i / stride) % len;
    const bool has_m = (c > 0) || (p.boundary == 0);
    const bool has_p = (c + 1 < len) || (p.boundary == 0);
    const uint32_t im = (c > 0) ? i - stride : i + (len - 1) * stride;
    const uint32_t ip = (c + 1 < len) ? i + stride : i - (len - 1) * stride;

    // The site types and word 0 of the three sites first; word k >= 1 of a
    // site only if word k-1 leaves room for it (L::need_next: its last slot
    // occupied, or the input may be unpacked).
    const uint32_t sti = p.sites[i];
    const uint32_t stm = has_m ? p.sites[im] : 0u;
    const uint32_t stp = has_p ? p.sites[ip] : 0u;
    uint32_t wi[W], wm[W], wp[W], out[W];
    uint32_t any = 0;
#pragma unroll
    for (int k = 0; k < W; k++) {
        wi[k] = (k == 0 || L::need_next(p, wi[k > 0 ? k - 1 : 0])) ? src[(size_t)k * p.N + i] : 0u;
        wm[k] = has_m && (k == 0 || L::need_next(p, wm[k > 0 ? k - 1 : 0])) ? src[(size_t)k * p.N + im] : 0u;
        wp[k] = has_p && (k == 0 || L::need_next(p, wp[k > 0 ? k - 1 : 0])) ? src[(size_t)k * p.N + ip] : 0u;
        any |= wi[k] | wm[k] | wp[k];
    }
    if (any == 0) {
#pragma unroll
        for (int k = 0; k < W; k++) dst[(size_t)k * p.N + i] = 0u;
        return;
    }
    pull_site_l<L>(p, i, im, ip, wi, wm, wp, sti, stm, stp, has_m, has_p, h, substep, out);
#pragma unroll
    for (int k = 0; k < W; k++) dst[(size_t)k * p.N + i] = out[k];
}

// Generic reaction phase: one site per thread, in place.
template <class L>
__global__ __launch_bounds__(256) void reaction_kernel(Params p, uint32_t *__restrict__ lat)
{
    constexpr int W = L::W;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= p.N) return;
    const uint32_t st = p.sites[i];
    uint32_t w[W];
#pragma unroll
    for (int k = 0; k < W; k++) w[k] = (k == 0 || L::need_next(p, w[k > 0 ? k - 1 : 0])) ? lat[(size_t)k * p.N + i] : 0u;
    const unsigned long long h = timestep_hash(p.seed32, p.ctl->timestep, 3);
    if (react_site_l<L>(p, i, st, w, h)) {
#pragma unroll
        for (int k = 0; k < W; k++) lat[(size_t)k * p.N + i] = w[k];
    }
}

__global__ __launch_bounds__(kResolveThreads) void resolve_kernel(Params p, uint32_t *lat)
{
    resolve_body<kResolveThreads>(p, lat);
}

// Batched resolver: block r resolves member r's step on its post-step buffer
// (lat[1]) and swaps the member's two buffers for the next step.
__global__ __launch_bounds__(kResolveThreads) void batch_resolve_kernel(Member *__restrict__ m)
{
    Member &M = m[blockIdx.x];
    uint32_t *const before = M.lat[0], *const after = M.lat[1];
    resolve_body<kResolveThreads>(M.p, after);
    __syncthreads();  // every wave has read both pointers (resolve_body returns block-uniformly)
    if (threadIdx.x == 0) {
        M.lat[0] = after;
        M.lat[1] = before;
        const uint32_t t = M.p.ctl->timestep;  // the next step's, written by this thread in resolve_body
        for (uint32_t s = 0; s < 3; s++) M.h[s] = timestep_hash(M.p.seed32, t, s);
    }
}

// Species counts: slot bytes up to a word's first empty one
// (ByteLattice::getParticleCounts, ByteLattice.cpp:495-520), or the words of
// the uint32 lattice (IntLattice::getParticleCounts, IntLattice.cpp:419-435:
// every nonzero word is one particle).  Reading the lattice bounds it, so a
// thread reads 16 bytes at a time and blocks count in LDS; counts has nS
// entries and the number of finished blocks behind them, all zero, and the
// block that ends last hands the counts to host memory and zeroes them again:
// one launch, and no copy, for what took three calls.
template <bool WORDS>
__global__ __launch_bounds__(256) void count_kernel(const uint32_t *__restrict__ lat, size_t nwords, uint32_t nS,
                                                    uint32_t *counts, uint32_t *out)
{
    constexpr uint32_t kCountBins = WORDS ? 1024u : 256u;
    __shared__ uint32_t hist[kCountBins], last;
    for (uint32_t k = threadIdx.x; k < kCountBins; k += blockDim.x) hist[k] = 0;
    __syncthreads();
    auto add = [&](uint32_t sp) {
        if (sp < kCountBins) atomicAdd(&hist[sp], 1u);
        else if (sp <= nS) atomicAdd(&counts[sp - 1], 1u);
    };
    auto word_of = [&](uint32_t word) {
        if (WORDS) {
            if (word) add(word);
            return;
        }
        while (word & 0xFFu) {
            add(word & 0xFFu);
            word >>= 8;
        }
    };
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x, threads = (size_t)gridDim.x * blockDim.x;
    const uint4 *lat4 = reinterpret_cast<const uint4 *>(lat);
    const size_t n4 = nwords / 4;
    for (size_t k = tid; k < n4; k += 2 * threads) {
        const bool two = k + threads < n4;
        const uint4 u = lat4[k], v = two ? lat4[k + threads] : make_uint4(0u, 0u, 0u, 0u);
        if (u.x | u.y | u.z | u.w) {
            word_of(u.x);
            word_of(u.y);
            word_of(u.z);
            word_of(u.w);
        }
        if (v.x | v.y | v.z | v.w) {
            word_of(v.x);
            word_of(v.y);
            word_of(v.z);
            word_of(v.w);
        }
    }
    for (size_t k = 4 * n4 + tid; k < nwords; k += threads) word_of(lat[k]);
    __syncthreads();
    for (uint32_t k = threadIdx.x + 1u; k < kCountBins && k <= nS; k += blockDim.x)
        if (hist[k]) atomicAdd(&counts[k - 1], hist[k]);
    wait_for_stores();  // the additions are done
    __syncthreads();
    if (threadIdx.x == 0) last = atomicAdd(&counts[nS], 1u) == gridDim.x - 1u ? 1u : 0u;
    __syncthreads();
    if (!last) return;
    for (uint32_t k = threadIdx.x; k < nS; k += blockDim.x) {
        out[k] = load_agent(&counts[k]);
        counts[k] = 0u;
    }
    if (threadIdx.x == 0) counts[nS] = 0u;
}

// The first words of solvers' control blocks to host memory.
__global__ void report_kernel(ReportList c, uint32_t *out)
{
    const uint32_t k = threadIdx.x % kReportWords;
    for (uint32_t m = threadIdx.x / kReportWords; m < c.n; m += blockDim.x / kReportWords)
        out[m * kReportWords + k] = load_agent(reinterpret_cast<const uint32_t *>(c.ctl[m]) + k);
}

// Range check of a lattice changed on the device by a caller: particle
// types at most nS, site types below nST (the kernels index their tables with
// them).  A violation is a sticky error, reported by the next synchronize.
__global__ __launch_bounds__(256) void validate_kernel(Params p, const uint32_t *__restrict__ lat, size_t nwords)
{
    bool bad = false;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t wi = (size_t)blockIdx.x * blockDim.x + threadIdx.x; wi < nwords; wi += stride) {
        const uint32_t v = lat[wi];
        if (p.word_particles) {
            bad |= v > p.nS;
            continue;
        }
#pragma unroll
        for (int b = 0; b < 4; b++) bad |= ((v >> (8 * b)) & 0xFFu) > p.nS;
    }
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < p.N; i += stride) bad |= p.sites[i] >= p.nST;
    if (bad) set_error(p.ctl, kErrInvalidLattice, p.ctl->timestep);
}

hipError_t launch_validate(const Params &p, const uint32_t *lat, hipStream_t st)
{
    hipLaunchKernelGGL(validate_kernel, dim3(1024), dim3(256), 0, st, p, lat, (size_t)p.N * p.W);
    return hipGetLastError();
}

// STREAM copy: one 16-byte load and store per thread, one pass (no
// grid-stride loop: on gfx950 a flat grid of n/256 blocks measures ~6.2 TB/s
// where a grid-stride loop over 8-64 blocks per CU stays near 4.5-4.8 TB/s);
// the measured copy peak that the sweeps' HBM rates are quoted against beside
// the 8 TB/s figure.
__global__ __launch_bounds__(256) void copy_kernel(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

hipError_t launch_copy(const void *src, void *dst, size_t bytes, int num_cu, hipStream_t st)
{
    (void)num_cu;
    const size_t n = bytes / sizeof(uint4);
    const size_t nb = (n + 255) / 256;
    if (nb == 0 || nb > 0x7fffffffu) return hipErrorInvalidValue;
    hipLaunchKernelGGL(copy_kernel, dim3((unsigned)nb), dim3(256), 0, st, reinterpret_cast<const uint4 *>(src),
                       reinterpret_cast<uint4 *>(dst), n);
    return hipGetLastError();
}

// Fills n words with a value (used instead of a memset node, so that work
// enqueued on a stream someone captures holds kernels only).
__global__ __launch_bounds__(256) void fill_kernel(uint32_t *__restrict__ ptr, size_t n, uint32_t value)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) ptr[i] = value;
}

hipError_t launch_fill(uint32_t *ptr, size_t n, uint32_t value, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    const size_t nb = std::min<size_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)nb), dim3(256), 0, st, ptr, n, value);
    return hipGetLastError();
}

__global__ void exp_kernel(const double *x, double *y, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = exp_proj(x[i]);
}

__global__ void prob_kernel(const float *a, float *y, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = reaction_probability(a[i]);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
static inline unsigned blocks_for(size_t n, unsigned bs) { return (unsigned)((n + bs - 1) / bs); }

template <class L>
static void sweep_launch(const Params &p, const uint32_t *src, uint32_t *dst, uint32_t stride, uint32_t len,
                         int axis, hipStream_t st)
{
    hipLaunchKernelGGL(sweep_kernel<L>, dim3(blocks_for(p.N, 256)), dim3(256), 0, st, p, src, dst, stride, len,
                       (uint32_t)axis);
}

hipError_t launch_sweep(const Params &p, const uint32_t *src, uint32_t *dst, int axis, hipStream_t st)
{
    const uint32_t stride = axis == 0 ? 1u : (axis == 1 ? p.X : p.XY);
    const uint32_t len = axis == 0 ? p.X : (axis == 1 ? p.Y : p.Z);
    const int key = p.word_particles ? 100 + (int)p.P : (int)p.W;
    switch (key) {
    case 1: sweep_launch<ByteSites<1>>(p, src, dst, stride, len, axis, st); break;
    case 2: sweep_launch<ByteSites<2>>(p, src, dst, stride, len, axis, st); break;
    case 4: sweep_launch<ByteSites<4>>(p, src, dst, stride, len, axis, st); break;
    case 104: sweep_launch<WordSites<4>>(p, src, dst, stride, len, axis, st); break;
    case 108: sweep_launch<WordSites<8>>(p, src, dst, stride, len, axis, st); break;
    case 116: sweep_launch<WordSites<16>>(p, src, dst, stride, len, axis, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_reaction(const Params &p, uint32_t *lat, hipStream_t st)
{
    const dim3 grid(blocks_for(p.N, 256)), block(256);
    const int key = p.word_particles ? 100 + (int)p.P : (int)p.W;
    switch (key) {
    case 1: hipLaunchKernelGGL(reaction_kernel<ByteSites<1>>, grid, block, 0, st, p, lat); break;
    case 2: hipLaunchKernelGGL(reaction_kernel<ByteSites<2>>, grid, block, 0, st, p, lat); break;
    case 4: hipLaunchKernelGGL(reaction_kernel<ByteSites<4>>, grid, block, 0, st, p, lat); break;
    case 104: hipLaunchKernelGGL(reaction_kernel<WordSites<4>>, grid, block, 0, st, p, lat); break;
    case 108: hipLaunchKernelGGL(reaction_kernel<WordSites<8>>, grid, block, 0, st, p, lat); break;
    case 116: hipLaunchKernelGGL(reaction_kernel<WordSites<16>>, grid, block, 0, st, p, lat); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_resolve(const Params &p, uint32_t *lat, hipStream_t st)
{
    hipLaunchKernelGGL(resolve_kernel, dim3(1), dim3(kResolveThreads), 0, st, p, lat);
    return hipGetLastError();
}

hipError_t launch_batch_resolve(Member *m, uint32_t n, hipStream_t st)
{
    hipLaunchKernelGGL(batch_resolve_kernel, dim3(n), dim3(kResolveThreads), 0, st, m);
    return hipGetLastError();
}

hipError_t launch_counts(const uint32_t *lat, size_t nwords, uint32_t nS, bool words, uint32_t *counts, uint32_t *out,
                         hipStream_t st)
{
    const unsigned g = std::min(std::max(blocks_for(nwords / 8, 256), 1u), 1024u);
    if (words)
        hipLaunchKernelGGL(count_kernel<true>, dim3(g), dim3(256), 0, st, lat, nwords, nS, counts, out);
    else
        hipLaunchKernelGGL(count_kernel<false>, dim3(g), dim3(256), 0, st, lat, nwords, nS, counts, out);
    return hipGetLastError();
}

hipError_t launch_report(const ReportList &c, uint32_t *out, hipStream_t st)
{
    const uint32_t threads = std::min((c.n * kReportWords + 63u) / 64u * 64u, 1024u);
    hipLaunchKernelGGL(report_kernel, dim3(1), dim3(threads), 0, st, c, out);
    return hipGetLastError();
}

hipError_t launch_exp(const double *x, double *y, size_t n, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(exp_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, x, y, n);
    return hipGetLastError();
}

hipError_t launch_prob(const float *a, float *y, size_t n, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(prob_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, a, y, n);
    return hipGetLastError();
}

}  // namespace lmx
