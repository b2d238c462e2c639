// GMRES(m) with classical Gram-Schmidt -- the PETSc KSPGMRES defaults the
// reference runs (run_nonlinear_matrixfree_split_mp.py:47-53: restart 30,
// CGS without refinement, Givens rotations, zero initial guess) -- and the
// BLAS-1 reductions around it.
//
// The basis V_0..V_m is stored unnormalised: v_j = scale[j] * V_j, which is
// bit-identical to the reference's VecNormalize (x *= 1/||x||) because every
// reader multiplies V_j by scale[j] exactly as VecScale would have.  This
// saves the separate normalisation pass.
//
// Bandwidth layout of the CGS kernels (mdot, maxpy + norm, solution update):
// one thread owns EPT double2 elements (coalesced, NT apart) of every vector;
// vectors are streamed in groups of two whose 2*EPT loads are issued back to
// back, so each wavefront keeps 16 x 16 B in flight per lane (in groups of
// eight with 1 or 2 elements).  The grid
// covers N exactly once (no grid-stride loop), EPT in {1,2,4,8} chosen so the
// launch has >= 256 workgroups.
//
// All reductions have a fixed grid and a fixed summation tree, so results
// are reproducible run to run.  Each reduction kernel writes one partial per
// workgroup; one workgroup of a later launch sums them (for GMRES with the
// Hessenberg / Givens bookkeeping, mostly inside the next step's fused J u,
// gmres_dev.h).  The kernel boundary orders the partials before their sum, so no
// device-scope fence (an L2 write-back on this GPU) is needed inside the
// streaming kernels.
#include "cgs_vec.h"
#include "gmres_dev.h"

namespace vv {
namespace {

constexpr int NT = kCgsNT;
constexpr int NW = kCgsNW;

// Sum of part[0..nb) by the whole block (thread t adds t, t+NT, ...).
__device__ __forceinline__ double final_sum_1(const double *part, int nb, double *red)
{
    double a = 0.0;
    for (int b = threadIdx.x; b < nb; b += NT) a += part[b];
    return block_sum_all(a, red);
}

// Column sums of part[b*PV + v] (b < nb) for v < ncols (<= PV), by the whole
// block: the columns are padded to cols = max(8, next power of two), thread t
// owns column t % cols and rows b = t / cols (mod NT / cols), loads issued 16
// at a time (one round for nb <= 16 NT / cols).  Result in out[v].
template <int PV>
__device__ void final_sum_cols(const double *part, int nb, int ncols, double *out, double *red /*[NT]*/)
{
    int cols = 8;
    while (cols < ncols) cols <<= 1;
    const int RS = NT / cols;        // row streams
    const int v = threadIdx.x & (cols - 1), r0 = threadIdx.x / cols;
    double acc = 0.0;
    if (v < ncols) {
        for (int b0 = r0; b0 < nb; b0 += RS * 16) {
            double x[16];
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int b = b0 + q * RS;
                x[q] = (b < nb) ? part[(size_t)b * PV + v] : 0.0;
            }
#pragma unroll
            for (int q = 0; q < 16; ++q) acc += x[q];
        }
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x < ncols) {
        double s = 0.0;
        for (int r = 0; r < RS; ++r) s += red[r * cols + threadIdx.x];
        out[threadIdx.x] = s;
    }
    __syncthreads();
}

// Instance b of a batched context is blockIdx.y in every kernel below.
__global__ void gmres_init_kernel(GmresState *g, const int32_t *active, double rtol, double atol, double dtol,
                                  int max_it, int max_k)
{
    if (threadIdx.x != 0) return;
    g += blockIdx.y;
    const int32_t act = active != nullptr ? active[blockIdx.y] : 1;
    g->st.it = 0;
    g->st.its = 0;
    g->st.reason = 0;
    g->st.done = act ? 0 : 1;
    g->st.active = act;
    g->st.res = 0.0;
    g->st.rnorm0 = 0.0;
    g->rtol = rtol;
    g->atol = atol;
    g->dtol = dtol;
    g->haptol = 1.0e-30;     // PETSc gmres->haptol
    g->max_it = max_it;
    g->max_k = max_k;
}

// Per-block partial sums of x*y over len elements (x == y: sum of squares).
// Cross-block sums are finished by a one-block kernel: the kernel boundary
// makes the partials visible without device-scope fences.
__global__ __launch_bounds__(NT) void dot_partial_kernel(const double *__restrict__ x, const double *__restrict__ y,
                                                         int64_t len, int64_t xstride, double *partial,
                                                         int64_t pstride)
{
    __shared__ double red[NW + 1];
    x += blockIdx.y * xstride;
    y += blockIdx.y * xstride;
    partial += blockIdx.y * pstride;
    double acc = 0.0;
    for (int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x; e < len; e += (int64_t)gridDim.x * NT)
        acc += x[e] * y[e];
    const double s = block_sum_all(acc, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// *out = sqrt(sum) (VecNorm) or the sum (VecDot)
__global__ __launch_bounds__(NT) void reduce_finish_kernel(const double *partial, int nb, double *out, int root)
{
    __shared__ double red[NW + 1];
    const double tot = final_sum_1(partial, nb, red);
    if (threadIdx.x == 0) *out = root ? sqrt(tot) : tot;
}

// the norms of the B instances' fields from nb partials each, and their Poisson
// residuals, into host memory
__global__ __launch_bounds__(NT) void norms_finish_kernel(const double *partial, int nb, int64_t pstride,
                                                          const double *pres, double *host)
{
    __shared__ double red[NW + 1];
    const double tot = final_sum_1(partial + blockIdx.y * pstride, nb, red);
    if (threadIdx.x != 0) return;
    host[blockIdx.y] = sqrt(tot);
    if (pres != nullptr) host[gridDim.y + blockIdx.y] = pres[16 * (size_t)blockIdx.y];
}

// TAIL: N is not a multiple of the vector width L (odd grids such as 9 x 9;
// one instance only, a batched context needs N % 4 == 0).  Thread t < N - L
// nvv of workgroup 0 then also owns the scalar element L nvv + t.
template <typename S, bool TAIL>
__device__ __forceinline__ int64_t tail_element(int64_t N, int64_t nvv)
{
    constexpr int L = V16<S>::L;
    return (TAIL && blockIdx.x == 0 && (int64_t)threadIdx.x < N - nvv * L) ? nvv * L + threadIdx.x : -1;
}
// VecMDot of w = V_{col+1} against v_0..v_col, written as HH(:, col) and the
// VecMAXPY coefficients -HH(:, col).
template <int EPT, int PV, typename S, bool TAIL>
__global__ __launch_bounds__(NT) void mdot_kernel(CgsArgs<S> a, int col)
{
    using V = typename V16<S>::type;
    constexpr int L = V16<S>::L;
    GmresState *g = a.g + blockIdx.y;
    a.basis += blockIdx.y * a.N;
    a.part += blockIdx.y * a.pstride;
    if (g->st.done) return;
    __shared__ double red[NW][PV];
    __shared__ double s_scale[PV];
    const int nvec = col + 1;
    if (threadIdx.x < nvec) s_scale[threadIdx.x] = g->scale[threadIdx.x];
    __syncthreads();
    const int64_t nvv = a.N / L;
    const int64_t e0 = (int64_t)blockIdx.x * NT * EPT + threadIdx.x;
    const V *W = reinterpret_cast<const V *>(a.basis + (size_t)nvec * a.vstride);
    const int64_t et = tail_element<S, TAIL>(a.N, nvv);
    const double wt = (TAIL && et >= 0) ? (double)a.basis[(size_t)nvec * a.vstride + et] : 0.0;
    V w[EPT];
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        const int64_t e = e0 + (int64_t)q * NT;
        w[q] = (e < nvv) ? W[e] : V{};
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr int G = cgs_group<EPT>();
    for (int v = 0; v < nvec; v += G) {
        V x[G][EPT];
        load_group<EPT, G, S>(a.basis, a.vstride, v, nvec - v, e0, nvv, x);
#pragma unroll
        for (int gg = 0; gg < G; ++gg) {
            if (v + gg >= nvec) break;
            const double sv = s_scale[v + gg];
            double acc = dot_slice<EPT, S>(w, x[gg], sv);
            if (TAIL && et >= 0) acc = __builtin_fma(wt, (double)a.basis[(size_t)(v + gg) * a.vstride + et] * sv, acc);
            acc = wave_sum(acc);
            if (lane == 0) red[wave][v + gg] = acc;
        }
    }
    __syncthreads();
    if (threadIdx.x < PV) {
        double s = 0.0;
        if (threadIdx.x < nvec)
            for (int wv = 0; wv < NW; ++wv) s += red[wv][threadIdx.x];
        a.part[(size_t)blockIdx.x * PV + threadIdx.x] = s;
    }
}

// CGS update  V_{it+1} <- w - sum_j h_j v_j  (VecMAXPY with lhh = -h) and
// per-block partial sums of its squared norm (of the stored values).
// From the newest vector down, each XCD on the rows whose dots it has just
// formed: the dots went from the oldest up, so what they read last is in the
// caches still, and a basis past the 256 MB of the last one (15 vectors at
// 1024 x 2048) is not read in a cycle that evicts every line before its reuse:
// with 21 vectors 67.4 -> 62.4 us here and 68.3 -> 64.7 in the dots.  Up to 12
// vectors, at the cache's 7.1 TB/s (2.3 us a vector) either way.
template <int EPT, int PV, typename S, bool TAIL>
__global__ __launch_bounds__(NT) void maxpy_norm_kernel(CgsArgs<S> a, int it)
{
    using V = typename V16<S>::type;
    constexpr int L = V16<S>::L;
    GmresState *g = a.g + blockIdx.y;
    a.basis += blockIdx.y * a.N;
    a.part += blockIdx.y * a.pstride;
    if (g->st.done) return;
    __shared__ double red[NW + 1];
    __shared__ double s_coef[kMaxRestart + 1], s_scale[kMaxRestart + 1];
    __shared__ double s_red[NT], s_h[PV];
    const int nvec = it + 1;
    const int64_t nvv = a.N / L;
    const int64_t e0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * NT * EPT + threadIdx.x;
    S *Ws = const_cast<S *>(a.basis) + (size_t)nvec * a.vstride;
    V *W = reinterpret_cast<V *>(Ws);
    const int64_t et = tail_element<S, TAIL>(a.N, nvv);
    double wt = (TAIL && et >= 0) ? (double)Ws[et] : 0.0;
    // w's loads are issued first, in flight while the dot partials are summed
    V wl[EPT];
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        const int64_t e = e0 + (int64_t)q * NT;
        wl[q] = (e < nvv) ? W[e] : V{};
    }
    if (threadIdx.x < nvec) s_scale[threadIdx.x] = g->scale[threadIdx.x];
    // HH(:, it) = <w, v_j>: every workgroup sums the mdot partials in the same
    // order (so all hold the same values); workgroup 0 records the column
    final_sum_cols<PV>(a.part, a.nbd, nvec, s_h, s_red);
    if (threadIdx.x < nvec) {
        const double h = s_h[threadIdx.x];
        s_coef[threadIdx.x] = -h;            // VecMAXPY coefficients lhh = -HH(:, it)
        if (blockIdx.x == 0) g->hh[it * (kMaxRestart + 1) + threadIdx.x] = h;
    }
    __syncthreads();
    double w[EPT][L];
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
#pragma unroll
        for (int l = 0; l < L; ++l) w[q][l] = vget(wl[q], l);
    }
    constexpr int G = cgs_group<EPT>();
    const S *last = a.basis + (int64_t)it * a.vstride;
    for (int j = 0; j < nvec; j += G) {
        V x[G][EPT];
        load_group<EPT, G, S>(last, -a.vstride, j, nvec - j, e0, nvv, x);
#pragma unroll
        for (int gg = 0; gg < G; ++gg) {
            if (j + gg >= nvec) break;
            const double sj = s_scale[it - j - gg], cj = s_coef[it - j - gg];
#pragma unroll
            for (int q = 0; q < EPT; ++q) {
#pragma unroll
                for (int l = 0; l < L; ++l) w[q][l] = w[q][l] + cj * (vget(x[gg][q], l) * sj);
            }
            if (TAIL && et >= 0) wt = wt + cj * ((double)a.basis[(size_t)(it - j - gg) * a.vstride + et] * sj);
        }
    }
    double acc = 0.0;
    if (TAIL && et >= 0) {
        const S o = (S)wt;
        Ws[et] = o;
        acc += (double)o * (double)o;
    }
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        const int64_t e = e0 + (int64_t)q * NT;
        if (e < nvv) {
            V o;
#pragma unroll
            for (int l = 0; l < L; ++l) vset(o, l, w[q][l]);
            W[e] = o;
#pragma unroll
            for (int l = 0; l < L; ++l) {
                const double r = vget(o, l);
                acc += r * r;
            }
        }
    }
    const double s = block_sum_all(acc, red);
    if (threadIdx.x == 0) a.part[a.noff + blockIdx.x] = s;
}

// The end of an Arnoldi step, or the start of a cycle, in a launch of its own
// (gmres_dev.h).
__global__ __launch_bounds__(NT) void gmres_update_kernel(HessArgs a) { hess_update(a); }

// KSPGMRESBuildSoln, and what follows it, in one launch: y from the rotated
// (triangular) Hessenberg matrix, then x = V y (store) or x += V y
// (VEC_TEMP = 0 + sum_j nrs_j v_j; x = x + VEC_TEMP; x is FP64 for either
// basis type).  With f (one instance): f -= V y in place of the store where the
// solve converged (SNESSolve_KSPONLY's step); a cycle that ended without a
// reason stores x for the restarts.  hout: workgroup 0 also stores the
// instance's final status there.
// Every workgroup solves the triangle itself, in its first wavefront, while the
// first group of basis vectors is on its way: lane r holds row r's right-hand
// side, and each unknown found is taken off the rows above (n steps of one
// division and one FMA; by one thread in a launch of its own it was n^2 / 2
// dependent LDS reads, 8.5 us at n = 21 and 15 at 30).  With zeroing x, its
// read-back and f -= x in their own launches the end of a solve took 8.5 +
// 39.4 + 11.8 us at 1024 x 2048 and its start 6.5 more.
template <int EPT, typename S, bool TAIL>
__global__ __launch_bounds__(NT) void update_kernel(double *__restrict__ x, double *__restrict__ f, int store,
                                                    CgsArgs<S> a, GmresStatus *hout)
{
    using V = typename V16<S>::type;
    constexpr int L = V16<S>::L;
    GmresState *g = a.g + blockIdx.y;
    a.basis += blockIdx.y * a.N;
    x += blockIdx.y * a.N;
    const int n = g->st.it;
    int reason = g->st.reason;
    __shared__ double s_coef[kMaxRestart + 1], s_scale[kMaxRestart + 1];
    __shared__ double sh[kMaxRestart * kMaxRestart];        // column j at j n
    __shared__ int s_sing;
    const int t = threadIdx.x;
    const int64_t nvv = a.N / L;
    const int64_t e0 = (int64_t)blockIdx.x * NT * EPT + t;
    constexpr int G = cgs_group<EPT>();
    V v[G][EPT];
    load_group<EPT, G, S>(a.basis, a.vstride, 0, n, e0, nvv, v);
    for (int idx = t; idx < n * n; idx += NT) {
        const int col = idx / n, r = idx - col * n;
        sh[idx] = g->hh[(size_t)col * (kMaxRestart + 1) + r];
    }
    double rhs = t < n ? g->grs[t] : 0.0;
    if (t < n) s_scale[t] = g->scale[t];
    if (t == 0) s_sing = 0;
    __syncthreads();
    if (t < 64) {
        double coef = 0.0;
        for (int k = n - 1; k >= 0; --k) {
            const double d = sh[k * n + k], h = t < k ? sh[k * n + t] : 0.0;
            const double y = d != 0.0 ? __shfl(rhs, k) / d : 0.0;
            if (d == 0.0 && t == 0) s_sing = 1;
            if (t == k) coef = y;
            rhs = rhs - h * y;
        }
        if (t < n) s_coef[t] = coef;
    }
    __syncthreads();
    if (s_sing) {                      // alike in every workgroup, whatever `reason` was read as
        reason = VV_KSP_DIVERGED_BREAKDOWN;
        if (blockIdx.x == 0 && t == 0) g->st.reason = reason;
    }
    if (blockIdx.x == 0 && t == 0) g->over = !g->st.active || reason != 0;
    if (hout != nullptr && blockIdx.x == 0 && t == 0) {
        // per-field stores by one lane
        GmresStatus *ho = hout + blockIdx.y;
        ho->it = n;
        ho->its = g->st.its;
        ho->reason = reason;
        ho->done = g->st.done;
        ho->active = g->st.active;
        ho->res = g->st.res;
        ho->rnorm0 = g->st.rnorm0;
    }
    const bool step = f != nullptr && reason > 0;
    if (n <= 0 && (!store || f != nullptr) && reason != 0) return;
    const int64_t et = tail_element<S, TAIL>(a.N, nvv);
    double tt = 0.0;
    double acc[EPT][L];
#pragma unroll
    for (int q = 0; q < EPT; ++q)
#pragma unroll
        for (int l = 0; l < L; ++l) acc[q][l] = 0.0;
    for (int j = 0; j < n; j += G) {
        if (j > 0) load_group<EPT, G, S>(a.basis, a.vstride, j, n - j, e0, nvv, v);
#pragma unroll
        for (int gg = 0; gg < G; ++gg) {
            if (j + gg >= n) break;
            const double sj = s_scale[j + gg], cj = s_coef[j + gg];
#pragma unroll
            for (int q = 0; q < EPT; ++q) {
#pragma unroll
                for (int l = 0; l < L; ++l) acc[q][l] = acc[q][l] + cj * (vget(v[gg][q], l) * sj);
            }
            if (TAIL && et >= 0) tt = tt + cj * ((double)a.basis[(size_t)(j + gg) * a.vstride + et] * sj);
        }
    }
    // out = base + sign * acc
    double *out = step ? f : x;
    const double sign = step ? -1.0 : 1.0;
    const bool add = step || !store;
    if (TAIL && et >= 0) out[et] = (add ? out[et] : 0.0) + sign * tt;
    // x, f: FP64, pairs where both are 16-byte aligned
    const bool pairs = (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        const int64_t e = e0 + (int64_t)q * NT;
        if (e < nvv) {
#pragma unroll
            for (int h = 0; h < L / 2; ++h) {
                double *o = out + e * L + 2 * h;
                double2 xv{0.0, 0.0};
                if (pairs) {
                    if (add) xv = *reinterpret_cast<const double2 *>(o);
                } else if (add) {
                    xv.x = o[0];
                    xv.y = o[1];
                }
                xv.x = xv.x + sign * acc[q][2 * h];
                xv.y = xv.y + sign * acc[q][2 * h + 1];
                if (pairs) {
                    *reinterpret_cast<double2 *>(o) = xv;
                } else {
                    o[0] = xv.x;
                    o[1] = xv.y;
                }
            }
        }
    }
}

// V_0 of a cycle with the partial sums of its squares: MODE 0 V_0 = b (FP64),
// 1 V_0 = (float) r with ||r|| of the FP64 right-hand side, 2 V_0 = b - V_0
// (KSPInitialResidual after a restart: r = b - A x).
template <int MODE, typename S>
__global__ __launch_bounds__(NT) void start_kernel(const double *__restrict__ b, S *v0, int64_t len, double *partial,
                                                   int64_t pstride)
{
    __shared__ double red[NW + 1];
    b += blockIdx.y * len;
    v0 += blockIdx.y * len;
    double acc = 0.0;
    for (int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x; e < len; e += (int64_t)gridDim.x * NT) {
        double d = b[e];
        if (MODE == 2) d = d + (-1.0) * (double)v0[e];
        v0[e] = (S)d;
        acc += d * d;
    }
    const double s = block_sum_all(acc, red);
    if (threadIdx.x == 0) partial[blockIdx.y * pstride + blockIdx.x] = s;
}

// y = y + alpha*x (VecAXPY).  mode 1: only when the GMRES reason is positive
// (SNESSolve_KSPONLY takes the step unless the linear solve diverged).
__global__ __launch_bounds__(NT) void axpy_kernel(double alpha, const double *__restrict__ x, double *y, int64_t len,
                                                  const GmresState *g, int mode)
{
    x += blockIdx.y * len;
    y += blockIdx.y * len;
    if (mode == 1 && g[blockIdx.y].st.reason <= 0) return;
    for (int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x; e < len; e += (int64_t)gridDim.x * NT)
        y[e] = y[e] + alpha * x[e];
}

// y = b - y; instance blockIdx.y at b + blockIdx.y len, y + blockIdx.y ystride
__global__ __launch_bounds__(NT) void rsub_kernel(const double *__restrict__ b, double *y, int64_t len,
                                                  int64_t ystride)
{
    b += blockIdx.y * len;
    y += blockIdx.y * ystride;
    for (int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x; e < len; e += (int64_t)gridDim.x * NT)
        y[e] = b[e] + (-1.0) * y[e];
}

__global__ __launch_bounds__(NT) void copy_kernel(const double *__restrict__ x, double *__restrict__ y, int64_t len)
{
    for (int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x; e < len; e += (int64_t)gridDim.x * NT) y[e] = x[e];
}

// y[b][j][i] += alpha w[b][i] (an x-only field added to every v-row)
__global__ __launch_bounds__(NT) void xadd_kernel(double *__restrict__ y, const double *__restrict__ w, int nx,
                                                  int64_t N, double alpha)
{
    y += blockIdx.y * N;
    w += (size_t)blockIdx.y * nx;
    for (int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x; e < N; e += (int64_t)gridDim.x * NT)
        y[e] = y[e] + alpha * w[e % nx];
}

// y = 0 (a kernel rather than a memset node, so captured graphs replay it)
__global__ __launch_bounds__(NT) void zero_kernel(double *__restrict__ y, int64_t len)
{
    for (int64_t e = (int64_t)blockIdx.x * NT + threadIdx.x; e < len; e += (int64_t)gridDim.x * NT) y[e] = 0.0;
}

int grid_for(int64_t len)
{
    const int64_t want = (len + NT - 1) / NT;
    return (int)(want < kReduceBlocks ? (want > 0 ? want : 1) : kReduceBlocks);
}

// 16-byte vectors per thread of the CGS kernels: the context's tuned value,
// else the largest of 8,4,2,1 that still gives >= 256 workgroups (nvv:
// 16-byte vectors per basis vector)
int cgs_ept_v(const vv_ctx *c, int64_t nvv)
{
    if (c != nullptr && c->tune_cgs_ept > 0) return c->tune_cgs_ept;
    for (int ept = 8; ept > 1; ept >>= 1)
        if ((nvv + (int64_t)NT * ept - 1) / ((int64_t)NT * ept) >= 256) return ept;
    return 1;
}

int cgs_blocks_v(const vv_ctx *c, int64_t nvv)
{
    const int ept = cgs_ept_v(c, nvv);
    return (int)((nvv + (int64_t)NT * ept - 1) / ((int64_t)NT * ept));
}

// the maxpy norm partials sit after the dot partials (rows x kMaxRestart) in
// each instance's part_stride = rows x (kMaxRestart + 2) doubles
int64_t norm_partial_offset(const vv_ctx *c) { return c->part_stride / (kMaxRestart + 2) * kMaxRestart; }

}  // namespace

int cgs_ept(const vv_ctx *c, int64_t nvv) { return cgs_ept_v(c, nvv); }

// partial-sum rows the CGS kernels can need (one vector per thread)
int cgs_blocks_max(int64_t N) { return (int)(((N >> 1) + NT - 1) / NT); }

hipError_t launch_gmres_init(vv_ctx *c, double rtol, double atol, double dtol, int max_it)
{
    hipLaunchKernelGGL(gmres_init_kernel, dim3(1, c->B), dim3(64), 0, c->stream, c->gs, c->active, rtol, atol, dtol,
                       max_it, c->p.restart);
    return hipGetLastError();
}

double *norm_partials(vv_ctx *c) { return c->partial + norm_partial_offset(c); }

namespace {

template <int E, typename S, bool TAIL>
void cgs_launch(vv_ctx *c, const S *basis, int which, int arg, double *x, int dot_rows, double *f, GmresStatus *hout)
{
    const int nb = cgs_blocks_v(c, c->N / V16<S>::L);
    CgsArgs<S> a{basis, c->N, c->vs, c->partial, c->part_stride, c->gs, norm_partial_offset(c),
                 dot_rows > 0 ? dot_rows : nb};
    const dim3 grid(nb, c->B), block(NT);
    if (which == 0) {
        if (c->p.restart < 32) launch_timed(c, mdot_kernel<E, 32, S, TAIL>, grid, block, 0, a, arg);
        else launch_timed(c, mdot_kernel<E, 64, S, TAIL>, grid, block, 0, a, arg);
    } else if (which == 1) {
        if (c->p.restart < 32) launch_timed(c, maxpy_norm_kernel<E, 32, S, TAIL>, grid, block, 0, a, arg);
        else launch_timed(c, maxpy_norm_kernel<E, 64, S, TAIL>, grid, block, 0, a, arg);
    } else {
        launch_timed(c, update_kernel<E, S, TAIL>, grid, block, 0, x, f, arg, a, hout);
    }
}

template <typename S, bool TAIL>
void cgs_dispatch_e(vv_ctx *c, const S *basis, int which, int arg, double *x, int dot_rows, double *f,
                    GmresStatus *hout)
{
    switch (cgs_ept_v(c, c->N / V16<S>::L)) {
    case 8: cgs_launch<8, S, TAIL>(c, basis, which, arg, x, dot_rows, f, hout); break;
    case 4: cgs_launch<4, S, TAIL>(c, basis, which, arg, x, dot_rows, f, hout); break;
    case 2: cgs_launch<2, S, TAIL>(c, basis, which, arg, x, dot_rows, f, hout); break;
    default: cgs_launch<1, S, TAIL>(c, basis, which, arg, x, dot_rows, f, hout); break;
    }
}

template <typename S>
hipError_t cgs_dispatch(vv_ctx *c, const S *basis, int which, int arg, double *x, int dot_rows = 0,
                        double *f = nullptr, GmresStatus *hout = nullptr)
{
    if (c->N % V16<S>::L) cgs_dispatch_e<S, true>(c, basis, which, arg, x, dot_rows, f, hout);
    else cgs_dispatch_e<S, false>(c, basis, which, arg, x, dot_rows, f, hout);
    return hipGetLastError();
}

// CGS dots of w with V_0..V_col: per-workgroup partials only; their column
// sums are formed by every workgroup of the following maxpy_norm launch
template <typename S>
hipError_t mdot_t(vv_ctx *c, const S *basis, int col)
{
    return cgs_dispatch(c, basis, 0, col, nullptr);
}

template <typename S>
hipError_t maxpy_norm_t(vv_ctx *c, const S *basis, int it, int dot_rows)
{
    c->pend_it = it;
    c->pend_nb = cgs_blocks_v(c, c->N / V16<S>::L);
    return cgs_dispatch(c, basis, 1, it, nullptr, dot_rows);
}

}  // namespace

hipError_t launch_mdot(vv_ctx *c, int col) { return mdot_t<double>(c, c->basis, col); }
hipError_t launch_maxpy_norm(vv_ctx *c, int it, int dot_rows)
{
    return maxpy_norm_t<double>(c, c->basis, it, dot_rows);
}

HessArgs take_update(vv_ctx *c)
{
    const bool due = c->pend_it >= 0 || c->pend_start;
    const HessArgs a{norm_partials(c), c->part_stride, due ? c->pend_nb : 0, c->pend_it, c->gs,
                     c->pend_start ? nullptr : c->report_out, c->report_seq, c->pend_start, c->start};
    c->pend_it = -1;
    c->pend_start = 0;
    c->report_out = nullptr;
    return a;
}

hipError_t launch_update(vv_ctx *c)
{
    const HessArgs a = take_update(c);
    if (a.nb == 0) return hipSuccess;
    hipLaunchKernelGGL(gmres_update_kernel, dim3(1, c->B), dim3(NT), 0, c->stream, a);
    return hipGetLastError();
}

hipError_t launch_build_solution(vv_ctx *c, double *x, double *f, bool store, GmresStatus *hout)
{
    return cgs_dispatch(c, c->basis, 2, store ? 1 : 0, x, 0, f, hout);
}
hipError_t launch_mdot32(vv_ctx *c, int col) { return mdot_t<float>(c, c->basis32, col); }
hipError_t launch_maxpy_norm32(vv_ctx *c, int it, int dot_rows)
{
    return maxpy_norm_t<float>(c, c->basis32, it, dot_rows);
}
hipError_t launch_build_solution32(vv_ctx *c, double *x, double *f, bool store, GmresStatus *hout)
{
    return cgs_dispatch(c, c->basis32, 2, store ? 1 : 0, x, 0, f, hout);
}

namespace {
hipError_t start_due(vv_ctx *c, int nb, bool first)
{
    c->pend_it = -1;
    c->pend_nb = nb;
    c->pend_start = first ? 2 : 1;
    return hipGetLastError();
}
}  // namespace

hipError_t launch_start(vv_ctx *c, const double *b, bool first)
{
    const int nb = grid_for(c->N);
    hipLaunchKernelGGL((start_kernel<0, double>), dim3(nb, c->B), dim3(NT), 0, c->stream, b, c->basis, c->N,
                       norm_partials(c), c->part_stride);
    return start_due(c, nb, first);
}

hipError_t launch_start32(vv_ctx *c, const double *r, bool first)
{
    const int nb = grid_for(c->N);
    hipLaunchKernelGGL((start_kernel<1, float>), dim3(nb, c->B), dim3(NT), 0, c->stream, r, c->basis32, c->N,
                       norm_partials(c), c->part_stride);
    return start_due(c, nb, first);
}

hipError_t launch_restart(vv_ctx *c, const double *b)
{
    const int nb = grid_for(c->N);
    hipLaunchKernelGGL((start_kernel<2, double>), dim3(nb, c->B), dim3(NT), 0, c->stream, b, c->basis, c->N,
                       norm_partials(c), c->part_stride);
    return start_due(c, nb, false);
}

hipError_t launch_rsub(vv_ctx *c, const double *b, double *y)
{
    hipLaunchKernelGGL(rsub_kernel, dim3(grid_for(c->N), c->B), dim3(NT), 0, c->stream, b, y, c->N, c->N);
    return hipGetLastError();
}

hipError_t launch_norms(vv_ctx *c, const double *x, int nb, const double *pres, double *host)
{
    if (x != nullptr) {
        nb = grid_for(c->N);
        hipLaunchKernelGGL(dot_partial_kernel, dim3(nb, c->B), dim3(NT), 0, c->stream, x, x, c->N, c->N, c->partial,
                           c->part_stride);
    }
    hipLaunchKernelGGL(norms_finish_kernel, dim3(1, c->B), dim3(NT), 0, c->stream, c->partial, nb, c->part_stride,
                       pres, host);
    return hipGetLastError();
}

hipError_t launch_norm2(vv_ctx *c, const double *x, int64_t n, double *out_dev)
{
    const int nb = grid_for(n);
    hipLaunchKernelGGL(dot_partial_kernel, dim3(nb), dim3(NT), 0, c->stream, x, x, n, (int64_t)0, c->partial,
                       c->part_stride);
    hipLaunchKernelGGL(reduce_finish_kernel, dim3(1), dim3(NT), 0, c->stream, c->partial, nb, out_dev, 1);
    return hipGetLastError();
}

hipError_t launch_dot(vv_ctx *c, const double *x, const double *y, int64_t n, double *out_dev)
{
    const int nb = grid_for(n);
    hipLaunchKernelGGL(dot_partial_kernel, dim3(nb), dim3(NT), 0, c->stream, x, y, n, (int64_t)0, c->partial,
                       c->part_stride);
    hipLaunchKernelGGL(reduce_finish_kernel, dim3(1), dim3(NT), 0, c->stream, c->partial, nb, out_dev, 0);
    return hipGetLastError();
}

hipError_t launch_axpy(vv_ctx *c, double alpha, const double *x, double *y, int64_t n)
{
    hipLaunchKernelGGL(axpy_kernel, dim3(grid_for(n)), dim3(NT), 0, c->stream, alpha, x, y, n, c->gs, 0);
    return hipGetLastError();
}

hipError_t launch_axpy_cond(vv_ctx *c, double alpha, const double *x, double *y)
{
    hipLaunchKernelGGL(axpy_kernel, dim3(grid_for(c->N), c->B), dim3(NT), 0, c->stream, alpha, x, y, c->N, c->gs, 1);
    return hipGetLastError();
}

hipError_t launch_copy(vv_ctx *c, const double *x, double *y, int64_t n)
{
    hipLaunchKernelGGL(copy_kernel, dim3(grid_for(n)), dim3(NT), 0, c->stream, x, y, n);
    return hipGetLastError();
}

hipError_t launch_xadd(vv_ctx *c, double *y, const double *w, double alpha)
{
    hipLaunchKernelGGL(xadd_kernel, dim3(grid_for(c->N), c->B), dim3(NT), 0, c->stream, y, w, c->p.nx, c->N, alpha);
    return hipGetLastError();
}

hipError_t launch_zero(vv_ctx *c, double *y, int64_t n)
{
    hipLaunchKernelGGL(zero_kernel, dim3(grid_for(n)), dim3(NT), 0, c->stream, y, n);
    return hipGetLastError();
}

}  // namespace vv
