// The end of an Arnoldi step on the device: the norm of the new Krylov vector
// from the CGS update's partial sums, the Hessenberg / Givens update and the
// convergence test.  One workgroup of kCgsNT threads does it, either in a
// launch of its own (krylov.hip) or as an extra workgroup of the next step's
// fused J u + rFFT (spectral.hip), whose other workgroups form the vector's
// scale from the same partials by the same tree.  Nothing here is contracted,
// whatever the including unit's setting, so both give the same bits.
#pragma once

#include "vv1d_internal.h"
#include "wave_ops.h"

namespace vv {
namespace {

constexpr int kGdNT = 256;
constexpr int kGdNW = kGdNT / 64;

// Sum over the block, returned in every thread (fixed tree).
__device__ __forceinline__ double block_sum_all(double v, double *red)
{
    const double ws = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ws;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kGdNW; ++w) s += red[w];
    __syncthreads();
    return s;
}

// thread t's share of the norm partials: part[t], part[t + NT], ...
__device__ __forceinline__ double norm_share(const double *part, int nb)
{
    double a = 0.0;
    for (int b = threadIdx.x; b < nb; b += kGdNT) a += part[b];
    return a;
}

// the scale of the Krylov vector whose squared norm is tot (VecNormalize)
__host__ __device__ __forceinline__ double scale_of(double tot)
{
    const double tt = sqrt(tot);
    return tt != 0.0 ? 1.0 / tt : 1.0;
}

__host__ __device__ __forceinline__ int ksp_test(const GmresState *g, double res)
{
#pragma clang fp contract(off)
    if (!__builtin_isfinite(res)) return VV_KSP_DIVERGED_NANORINF;
    if (res <= g->ttol) return res < g->atol ? VV_KSP_CONVERGED_ATOL : VV_KSP_CONVERGED_RTOL;
    if (res >= g->dtol * g->st.rnorm0) return VV_KSP_DIVERGED_DTOL;
    return 0;
}

// The report the host polls: number and end of the cycle in one 32-bit word of
// mapped pinned memory, so no fence orders it (a system-scope release would
// write back the XCD's L2).
__device__ __forceinline__ void report(uint32_t *hout, uint32_t seq, bool done)
{
    __hip_atomic_store(hout, 2 * seq + (done ? 1u : 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The end of the cycle as the launch that carries update it + 1 takes it (it = -1:
// after the cycle's start); st.done is for every other launch.
__host__ __device__ __forceinline__ void set_skip(GmresState *g, int it, bool end) { g->skip[(it + 1) & 1] = end; }

// Whether a launch that carries the update or start `a` has nothing to do for
// instance b besides it: done as of the update before; at a start, not taking part.
// The launch's other workgroups ask while hess_update runs in its first one, so
// nothing that hess_update writes is read here: skip by the parity of the step
// (it writes the other one), at a restart what the solution update of the cycle
// before left, at a first start the instance mask.
__host__ __device__ __forceinline__ bool carried_skip(const HessArgs &a, const GmresState *g, int b)
{
    if (a.start == 2) return a.init.active != nullptr && a.init.active[b] == 0;
    if (a.start == 1) return g->over != 0;
    return g->skip[a.it & 1] != 0;
}

__device__ __forceinline__ bool hess_skip(const HessArgs &a) { return carried_skip(a, a.g + blockIdx.y, blockIdx.y); }

// Start of a cycle on V_0 of instance b with ||V_0||^2 = tot (KSPGMRESCycle
// entry: VecNormalize(VV(0)), zero-residual and convergence tests), by one thread.
__host__ __device__ __forceinline__ void cycle_start(const HessArgs &a, GmresState *g, int b, double tot)
{
#pragma clang fp contract(off)
    if (a.start == 2) {
        const int32_t act = a.init.active != nullptr ? a.init.active[b] : 1;
        g->st.its = 0;
        g->st.reason = 0;
        g->st.active = act;
        g->st.res = 0.0;
        g->st.rnorm0 = 0.0;
        g->rtol = a.init.rtol;
        g->atol = a.init.atol;
        g->dtol = a.init.dtol;
        g->haptol = 1.0e-30;     // PETSc gmres->haptol
        g->max_it = a.init.max_it;
        g->max_k = a.init.max_k;
    }
    g->st.it = 0;
    // an instance that is not solving, or whose solve has ended, stays done
    if (!g->st.active || g->st.reason != 0) {
        g->st.done = 1;
        set_skip(g, -1, true);
        return;
    }
    const double nrm = sqrt(tot);
    g->st.done = 0;
    set_skip(g, -1, false);
    g->scale[0] = scale_of(tot);
    g->grs[0] = nrm;
    g->st.res = nrm;
    if (nrm == 0.0) {
        g->st.reason = VV_KSP_CONVERGED_ATOL;
        g->st.done = 1;
        set_skip(g, -1, true);
        return;
    }
    if (a.start == 2) {
        g->st.rnorm0 = nrm;
        g->ttol = fmax(a.init.rtol * nrm, a.init.atol);
    }
    const int rsn = ksp_test(g, nrm);
    if (rsn != 0) {
        g->st.reason = rsn;
        g->st.done = 1;
        set_skip(g, -1, true);
    }
}

// VecNormalize of V_{it+1} from the maxpy partials, then
// KSPGMRESUpdateHessenberg (rotations, happy breakdown, residual estimate)
// and the convergence test of instance blockIdx.y; sets done when the cycle
// ends.  The Hessenberg column and the previous rotations are staged in LDS by
// the whole block (loads in flight together with the norm's partials), so the
// sequential rotation chain of thread 0 reads LDS, not dependent global loads.
// a.hout (optional): the report to the host.
__device__ __forceinline__ void hess_update(const HessArgs &a)
{
#pragma clang fp contract(off)
    GmresState *g = a.g + blockIdx.y;
    const double *part = a.part + blockIdx.y * a.pstride;
    uint32_t *hout = a.hout != nullptr ? a.hout + blockIdx.y : nullptr;
    if (a.start) {
        __shared__ double sred[kGdNW + 1];
        const double tot = block_sum_all(norm_share(part, a.nb), sred);
        if (threadIdx.x == 0) cycle_start(a, g, blockIdx.y, tot);
        return;
    }
    const int it = a.it;
    // every load of the block is issued before the early-exit test waits on
    // the flag's (reading the state of a finished cycle is harmless)
    const int32_t done = g->st.done;
    __shared__ double red[kGdNW + 1];
    __shared__ double s_h[kMaxRestart + 2], s_c[kMaxRestart], s_s[kMaxRestart];
    double *hh = g->hh + (size_t)it * (kMaxRestart + 1);
    const int t = threadIdx.x;
    const double h_t = t <= it ? hh[t] : 0.0;
    const double c_t = t < it ? g->cc[t] : 0.0;
    const double s_t = t < it ? g->ss[t] : 0.0;
    const double grs_it = g->grs[it];
    const double acc = norm_share(part, a.nb);
    if (done) {                        // uniform over the block, before any barrier
        if (t == 0) set_skip(g, it, true);
        if (hout && t == 0) report(hout, a.seq, true);
        return;
    }
    if (t <= it) s_h[t] = h_t;
    if (t < it) {
        s_c[t] = c_t;
        s_s[t] = s_t;
    }
    const double tot = block_sum_all(acc, red);        // barriers: the LDS stores above are visible
    if (t != 0) return;
    const double tt = sqrt(tot);
    s_h[it + 1] = tt;
    g->scale[it + 1] = scale_of(tot);
    // happy breakdown
    double hapbnd = fabs(tt / grs_it);
    if (hapbnd > g->haptol) hapbnd = g->haptol;
    const bool hapend = tt < hapbnd;
    // apply the previous rotations to the new column
    for (int q = 1; q <= it; ++q) {
        const double t0 = s_h[q - 1];
        s_h[q - 1] = s_c[q - 1] * t0 + s_s[q - 1] * s_h[q];
        s_h[q] = s_c[q - 1] * s_h[q] - s_s[q - 1] * t0;
    }
    double res;
    int reason = 0;
    if (!hapend) {
        const double d = sqrt(s_h[it] * s_h[it] + s_h[it + 1] * s_h[it + 1]);
        if (d == 0.0) {
            reason = VV_KSP_DIVERGED_BREAKDOWN;
            res = g->st.res;
        } else {
            const double cc = s_h[it] / d, ss = s_h[it + 1] / d;
            g->cc[it] = cc;
            g->ss[it] = ss;
            g->grs[it + 1] = -(ss * grs_it);
            g->grs[it] = cc * grs_it;
            s_h[it] = cc * s_h[it] + ss * s_h[it + 1];
            res = fabs(-(ss * grs_it));
        }
    } else {
        res = 0.0;
    }
    for (int q = 0; q <= it + 1; ++q) hh[q] = s_h[q];
    g->st.it = it + 1;
    g->st.its += 1;
    g->st.res = res;
    if (reason == 0) reason = ksp_test(g, res);
    if (hapend && reason == 0) reason = VV_KSP_DIVERGED_BREAKDOWN;
    if (reason == 0 && g->st.its >= g->max_it) reason = VV_KSP_DIVERGED_ITS;
    g->st.reason = reason;
    const bool end = reason != 0 || g->st.it >= g->max_k || g->st.its >= g->max_it;
    if (end) g->st.done = 1;
    set_skip(g, it, end);
    if (hout) report(hout, a.seq, end);
}

}  // namespace
}  // namespace vv
