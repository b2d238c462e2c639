// Arakawa J1 / J2 / J4 Poisson-bracket kernels: the implicit-midpoint
// residual F(f), the Jacobian-vector product J u and the plain accumulation
// y += factor {x, H} (or y = 0 + factor {x, H}; the double-bracket
// dissipation terms are chains of these).
//
// This translation unit is compiled with -ffp-contract=off: the stencils of
// bracket_kernel keep the reference's IEEE operation order
// (PoissonBracket.pyx:100-113, 221-234, 360-389; C left-to-right), so what
// the callbacks return is bit-identical to the reference's unfused double
// arithmetic; bracket_sep_kernel forms the solver's own J u and F(f).
//
// Layout: natural order, element (i, j) at i + nx*j (x contiguous).
// Tiling: one workgroup computes a 64 (x) x TY (v) tile (TY = 16).  The tile
// of the bracket's first argument and of H_ave, both with a 2-cell halo, is
// staged in LDS (br_cell: a thread's own output cells first, then its share of
// the halo; F(f) at 2048 x 4096 61 -> 51 us against cells dealt in row order);
// every global load of a thread is issued before the first
// LDS store.  H_ave is composed on the fly from its 1D factors
// ((((h0_j + .5 h1p_i) + .5 h1h_i) + .5 h2p_i) + .5 h2h_i), exactly the
// value the reference's 2D Have vector holds (PETScVlasovSolver.pyx:145-149),
// so it costs no HBM traffic.  Each wavefront owns TY/4 consecutive rows;
// lane l computes column i0 + l (global loads and stores are 512-byte rows)
// and walks down its rows with the stencil values in a sliding register
// window.

#include "arakawa.h"
#include "gmres_dev.h"
#include "vv1d_internal.h"

namespace vv {
namespace {

constexpr int TX = kBrTX;
constexpr int TY = kBrTY;
constexpr int HX = kBrHX;
constexpr int HY = kBrHY;
constexpr int NT = 256;
constexpr int ROWS_PER_WAVE = TY / (NT / 64);
constexpr int NQ = kBrCells;
static_assert(ROWS_PER_WAVE == kBrOwn && TX == 64 && NT == 256, "br_cell's shape");

// MODE_TRANSPOSED: y = alpha u + factor {u~, H} on every row, u~ = u with the
// rows outside 2..nv-3 zeroed.  The Arakawa stencils are skew-symmetric in
// their first argument ({f, H} summed against g equals -{g, H} summed
// against f for fields that vanish outside the grid), so for the masked
// operator M u = R {u, H} (R: keep rows 2..nv-3) the transpose is
// M^T g = -{R g, H} evaluated on all rows: this mode with factor = -1.
enum { MODE_RESIDUAL = 0, MODE_JACOBIAN = 1, MODE_ACCUMULATE = 2, MODE_TRANSPOSED = 3 };

// T is the field type: double, or float (bracket_sep_kernel: J u of the FP32
// GMRES cycle of the mixed-precision solver, coefficients rounded once).
// Instance b of a batched context is blockIdx.y: its fields start at b * N,
// its x-factors of H at b * nx, its GMRES state b * gstride bytes after
// instance 0's (uscale, done), its hx-dependent factors in inst[b].
template <typename T>
struct BrArgs {
    int nx, nv;
    int64_t N;
    const T *f;            // residual: f; jacobian: u; accumulate: x
    const T *fh;           // residual: f at the previous time level
    const double *uscale;  // optional device scale of the first argument (unnormalised Krylov vector)
    T *y;
    const double *h0, *h1p, *h1h, *h2p, *h2h;
    const double *h2d;     // optional second argument as a 2D field (instead of H_ave)
    const double *hxv;     // optional second argument that depends on x only
    const InstConst *inst;
    double ht_inv, factor, alpha;
    const int32_t *done;   // optional early-exit flag (GMRES cycle finished)
    int64_t gstride;
    double *part;          // residual: per-workgroup sums of y^2 (null: none), pstride apart per instance
    int64_t pstride;
    int store;             // accumulate mode: y = 0 + factor {x, H} (the reference's
                           // Vec.set(0.) followed by PoissonBracket.function)
};

template <int KIND, int MODE>
__global__ __launch_bounds__(NT) void bracket_kernel(BrArgs<double> a)
{
    const int b = blockIdx.y;
    __shared__ double sF[HY][HX];
    __shared__ double sH[HY][HX];
    __shared__ double sX[4][HX];      // h1p, h1h, h2p, h2h (or the x-only H) of the tile's columns
    __shared__ double sV[HY];         // h0 of the tile's rows

    const int nx = a.nx, nv = a.nv;
    const BrTile tile = br_tile(blockIdx.x, nx, nv);
    const int i0 = tile.i0, j0 = tile.j0;
    const size_t fo = (size_t)b * a.N, xo = (size_t)b * nx;
    const double *__restrict__ fin = a.f + fo;
    const double *__restrict__ fhin = (MODE == MODE_RESIDUAL) ? a.fh + fo : nullptr;
    double *__restrict__ yout = a.y + fo;
    const double half = 0.5;
    const bool factors = (a.h2d == nullptr && a.hxv == nullptr);

    // Phase 1: every global load of the block is issued before anything waits
    // on one (the early-exit flag, the scale, the 1D factors and the tile), so
    // a block pays one memory latency, not one per dependent step.
    const int32_t dflag =
        (a.done != nullptr) ? *reinterpret_cast<const int32_t *>(reinterpret_cast<const char *>(a.done) + b * a.gstride)
                            : 0;
    // batched: a finished instance skips its loads (one instance keeps them
    // in flight with the flag's)
    if (gridDim.y > 1 && dflag) return;
    const double usd = (a.uscale != nullptr)
                           ? *reinterpret_cast<const double *>(reinterpret_cast<const char *>(a.uscale) + b * a.gstride)
                           : 1.0;
    double xf0 = 0.0, xf1 = 0.0, xf2 = 0.0, xf3 = 0.0, vf = 0.0;
    if (threadIdx.x < HX) {
        const int gi = br_halo_column(tile, (int)threadIdx.x, nx);
        if (a.hxv != nullptr) {
            xf0 = a.hxv[xo + gi];
        } else if (factors) {
            xf0 = a.h1p[xo + gi];
            xf1 = a.h1h[xo + gi];
            xf2 = a.h2p[xo + gi];
            xf3 = a.h2h[xo + gi];
        }
    } else if (threadIdx.x < HX + HY) {
        const int gj = br_halo_row(tile, (int)threadIdx.x - HX, nv);
        if (factors && gj >= 0) vf = a.h0[gj];
    }
    double fa[NQ], fb[NQ];
    double hq[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        int r, c;
        fa[q] = 0.0;
        fb[q] = 0.0;
        hq[q] = 0.0;
        if (br_cell(threadIdx.x, q, &r, &c)) {
            const int64_t o = br_halo_offset(tile, r, c, nx, nv);
            if (o >= 0) {
                fa[q] = fin[o];
                if (MODE == MODE_RESIDUAL) fb[q] = fhin[o];
                if (a.h2d != nullptr) hq[q] = a.h2d[fo + o];
            }
        }
    }

    // Phase 2: stage the 1D factors, then the tile of the first argument and of H
    if (dflag) return;                 // uniform over the block, before any barrier
    if (threadIdx.x < HX) {
        sX[0][threadIdx.x] = xf0;
        sX[1][threadIdx.x] = xf1;
        sX[2][threadIdx.x] = xf2;
        sX[3][threadIdx.x] = xf3;
    } else if (threadIdx.x < HX + HY) {
        sV[threadIdx.x - HX] = vf;
    }
    __syncthreads();

    const double us = usd;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        int r, c;
        if (br_cell(threadIdx.x, q, &r, &c)) {
            const int gj = br_halo_row(tile, r, nv);
            const bool in = gj >= 0;
            double fv;
            if (MODE == MODE_RESIDUAL) {
                fv = half * fb[q] + half * fa[q];            // Fave (PETScNLVlasovMP.pyx:44-46)
            } else if (MODE == MODE_TRANSPOSED) {
                fv = (gj >= 2 && gj < nv - 2) ? fa[q] * us : 0.0;
            } else if (MODE == MODE_JACOBIAN) {
                fv = fa[q] * us;                             // == VecScale'd Krylov vector
            } else {
                fv = (a.uscale != nullptr) ? fa[q] * us : fa[q];
            }
            sF[r][c] = fv;
            // ((((h0_j + .5 h1p_i) + .5 h1h_i) + .5 h2p_i) + .5 h2h_i)  (PETScVlasovSolver.pyx:145-149);
            // outside the grid H is 0: those cells only meet rows whose result
            // is not formed (j < 2 or j >= nv - 2) except in the transposed mode
            if (a.h2d != nullptr) {
                sH[r][c] = in ? hq[q] : 0.0;
            } else if (a.hxv != nullptr) {
                sH[r][c] = in ? sX[0][c] : 0.0;
            } else {
                sH[r][c] = in ? compose_have(sV[r], sX[0][c], sX[1][c], sX[2][c], sX[3][c]) : 0.0;
            }
        }
    }
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int i = i0 + lane;
    if (MODE != MODE_RESIDUAL && i >= nx) return;
    const int cx = lane + 2;
    double sq = 0.0;
    const double ht_inv = a.ht_inv, af1 = a.inst[b].af1, af2 = a.inst[b].af2, factor = a.factor;

    // Each lane walks down its column with the stencil values of F and H in
    // a sliding register window (arakawa.h).  Same values, same expressions.
    const int rr0 = wave * ROWS_PER_WAVE;
    const TileRd<double, HX> rF{&sF[0][0]}, rH{&sH[0][0]};
    ArakawaWin<double> win;
    win.load(rF, rH, rr0 + 2, cx);
#pragma unroll
    for (int q = 0; q < ROWS_PER_WAVE; ++q) {
        const int rr = rr0 + q;
        const int j = j0 + rr;
        if (j < nv && (MODE != MODE_RESIDUAL || i < nx)) {
            const size_t o = (size_t)j * nx + i;
            double base;
            if (MODE == MODE_RESIDUAL) {
                const double fder = fa[q] - fb[q];                   // Fder = (0 + F) - Fh
                base = 0.0 + ht_inv * fder;                     // Y = 0; Y += Fder/dt
            } else if (MODE == MODE_JACOBIAN) {
                base = jacobian_base(ht_inv, win.f0[2]);         // Y = 0; Y += u/dt
            } else if (MODE == MODE_TRANSPOSED) {
                base = a.alpha * (fa[q] * us);
            } else {
                base = a.store ? 0.0 : yout[o];
            }
            double out = base;
            if (MODE == MODE_TRANSPOSED || (j >= 2 && j < nv - 2))
                out = arakawa_add<KIND>(win, base, factor, af1, af2);
            yout[o] = out;
            if (MODE == MODE_RESIDUAL) sq += (double)out * (double)out;
        }
        // move the window one row down (rows stay inside the staged tile)
        if (q + 1 < ROWS_PER_WAVE) win.advance(rF, rH, rr + 3, cx);
    }
    // the residual's norm without another pass over it (6.8 us at 1024 x 2048)
    if (MODE == MODE_RESIDUAL && a.part != nullptr) {
        __shared__ double red[NT / 64];
        sq = wave_sum(sq);
        if (lane == 0) red[wave] = sq;
        __syncthreads();
        if (threadIdx.x == 0) {
            double s = 0.0;
            for (int w = 0; w < NT / 64; ++w) s += red[w];
            a.part[b * a.pstride + blockIdx.x] = s;
        }
    }
}

// J u and F(f) inside the solver: the same tiles with the bracket split into row
// and column coefficients (SepWin, arakawa.h), so one tile in LDS (12 KB: as
// many wavefronts a CU as there are slots for, against 24 with H beside it) and
// a quarter of the arithmetic.  F(f) at 1024 x 2048 18.6 us unfactored, 13.9 here;
// J u at 2048 x 1024 13.7, 9.6.  T is double, or float for the FP32 cycle.
template <int KIND, int MODE, typename T>
__global__ __launch_bounds__(NT) void bracket_sep_kernel(BrArgs<T> a)
{
    const int b = blockIdx.y;
    __shared__ T sF[HY][HX];
    __shared__ double sP[HX];                      // x-part of H of the tile's columns
    __shared__ __align__(16) T sA[TY][4];          // coefficients of its rows

    const int nx = a.nx, nv = a.nv, t = threadIdx.x;
    const BrTile tile = br_tile(blockIdx.x, nx, nv);
    const int i0 = tile.i0, j0 = tile.j0;
    const size_t fo = (size_t)b * a.N, xo = (size_t)b * nx;
    const T *__restrict__ fin = a.f + fo;
    const T *__restrict__ fhin = (MODE == MODE_RESIDUAL) ? a.fh + fo : nullptr;
    T *__restrict__ yout = a.y + fo;
    const T half = T(0.5);
    const int32_t dflag =
        (a.done != nullptr) ? *reinterpret_cast<const int32_t *>(reinterpret_cast<const char *>(a.done) + b * a.gstride)
                            : 0;
    // batched: a finished instance skips its loads (one instance keeps them
    // in flight with the flag's)
    if (gridDim.y > 1 && dflag) return;
    const double usd = (a.uscale != nullptr)
                           ? *reinterpret_cast<const double *>(reinterpret_cast<const char *>(a.uscale) + b * a.gstride)
                           : 1.0;
    double c1, c2;
    sep_weights(KIND, a.factor, a.inst[b].af1, a.inst[b].af2, c1, c2);
    T fa[NQ], fb[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        int r, c;
        fa[q] = T(0);
        fb[q] = T(0);
        if (br_cell(t, q, &r, &c)) {
            const int64_t o = br_halo_offset(tile, r, c, nx, nv);
            if (o >= 0) {
                fa[q] = fin[o];
                if (MODE == MODE_RESIDUAL) fb[q] = fhin[o];
            }
        }
    }
    double phi = 0.0;
    if (t < HX) {
        const size_t gi = xo + br_halo_column(tile, t, nx);
        phi = phi_ave(a.h1p[gi], a.h1h[gi], a.h2p[gi], a.h2h[gi]);
    }
    T k[4];
    const bool krow = t >= 128 && t < 128 + TY;
    if (krow) sep_row(a.h0, j0 + t - 128, nv, c1, c2, k);
    if (dflag) return;                 // uniform over the block, before any barrier
    const T us = (T)usd;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        int r, c;
        if (br_cell(t, q, &r, &c)) sF[r][c] = MODE == MODE_RESIDUAL ? half * fb[q] + half * fa[q] : fa[q];
    }
    if (t < HX) sP[t] = phi;
    if (krow) {
#pragma unroll
        for (int q = 0; q < 4; ++q) sA[t - 128][q] = k[q];
    }
    __syncthreads();
    const int lane = t & 63, wave = t >> 6;
    const int i = i0 + lane, cx = lane + 2, rr0 = wave * ROWS_PER_WAVE;
    if (i >= nx) return;
    const T ht_inv = (T)a.ht_inv;
    T B[4];
    sep_coef(sP[cx - 2], sP[cx - 1], sP[cx], sP[cx + 1], sP[cx + 2], c1, c2, B);
    const TileRd<T, HX> rF{&sF[0][0]};
    SepWin<T> win;
    win.load(rF, rr0 + 2, cx);
#pragma unroll
    for (int q = 0; q < ROWS_PER_WAVE; ++q) {
        const int rr = rr0 + q, j = j0 + rr;
        if (j < nv) {
            const size_t o = (size_t)j * nx + i;
            T out;
            if (MODE == MODE_RESIDUAL) out = T(0) + ht_inv * (fa[q] - fb[q]);
            else out = jacobian_base(ht_inv, win.f0[2]);
            if (j >= 2 && j < nv - 2) out += win.bracket(sA[rr], B, sep_near(KIND), sep_far(KIND));
            if (MODE == MODE_JACOBIAN) out = scaled(out, us);      // J is linear
            yout[o] = out;
        }
        if (q + 1 < ROWS_PER_WAVE) win.advance(rF, rr + 3, cx);
    }
}

// The transposed linearisation's two brackets in one launch: with u~ = u (times
// its scale) on rows 2..nv-3 and 0 elsewhere,
//   y = alpha u + factor {u~, H_ave} on all rows,  csum = sum_j {u~, g}_ij
// by 16-row bands (tile row t at csum[t nx + i], instances cstride apart): the
// coupling term needs only the column sums of its bracket (g = f_bar in a.h2d),
// so that field is neither stored nor read back.  u~ is staged once for both, and
// the bracket with H_ave is the factored one (SepWin: H is 0 outside the grid, where
// its coefficients only meet rows of u~ that are 0): two 20 x 68 tiles (22 KB of
// LDS).  hs: the previous step's Hessenberg
// update or the cycle's start, as in the fused J u + rFFT.  At 256 x 512 it
// replaces two bracket launches (5.2 us each), the density (3.7 us) and the
// update (3.6 us).
template <int KIND>
__global__ __launch_bounds__(NT) void bracket_pair_kernel(BrArgs<double> a, HessArgs hs, double *csum,
                                                          int64_t cstride)
{
    const int extra = hs.nb > 0 ? 1 : 0;
    if (extra && blockIdx.x == 0) {
        hess_update(hs);
        return;
    }
    const int b = blockIdx.y;
    __shared__ double sF[HY][HX], sG[HY][HX];
    __shared__ double sP[HX], sS[NT / 64][TX];
    __shared__ __align__(16) double sA[TY][4];
    __shared__ double red[kGdNW + 1];
    const int nx = a.nx, nv = a.nv;
    const BrTile tile = br_tile((int)blockIdx.x - extra, nx, nv);
    const size_t fo = (size_t)b * a.N, xo = (size_t)b * nx;
    const double *__restrict__ fin = a.f + fo;
    const double *__restrict__ gin = a.h2d + fo;
    const int32_t dflag = extra ? hess_skip(hs)
                          : a.done != nullptr
                              ? *reinterpret_cast<const int32_t *>(reinterpret_cast<const char *>(a.done) + b * a.gstride)
                              : 0;
    if (gridDim.y > 1 && dflag) return;
    const double nshare = extra ? norm_share(hs.part + b * hs.pstride, hs.nb) : 0.0;
    double us = a.uscale != nullptr && !extra
                    ? *reinterpret_cast<const double *>(reinterpret_cast<const char *>(a.uscale) + b * a.gstride)
                    : 1.0;
    double c1, c2, phi = 0.0;
    sep_weights(KIND, a.factor, a.inst[b].af1, a.inst[b].af2, c1, c2);
    if (threadIdx.x < HX) {
        const size_t gi = xo + br_halo_column(tile, (int)threadIdx.x, nx);
        phi = phi_ave(a.h1p[gi], a.h1h[gi], a.h2p[gi], a.h2h[gi]);
    }
    const int kr = (int)threadIdx.x - 128;
    const bool krow = kr >= 0 && kr < TY;
    double kc[4];
    if (krow) sep_row(a.h0, tile.j0 + kr, nv, c1, c2, kc);
    double fa[NQ], ga[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        int r, c;
        fa[q] = ga[q] = 0.0;
        if (br_cell(threadIdx.x, q, &r, &c)) {
            const int64_t o = br_halo_offset(tile, r, c, nx, nv);
            if (o >= 0) {
                fa[q] = fin[o];
                ga[q] = gin[o];
            }
        }
    }
    if (dflag) return;                 // uniform over the block, before any barrier
    if (extra) us = scale_of(block_sum_all(nshare, red));
    if (threadIdx.x < HX) sP[threadIdx.x] = phi;
    if (krow) {
#pragma unroll
        for (int q = 0; q < 4; ++q) sA[kr][q] = kc[q];
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        int r, c;
        if (br_cell(threadIdx.x, q, &r, &c)) {
            const int gj = br_halo_row(tile, r, nv);
            sF[r][c] = (gj >= 2 && gj < nv - 2) ? fa[q] * us : 0.0;
            sG[r][c] = ga[q];
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = tile.i0 + lane, cx = lane + 2, rr0 = wave * ROWS_PER_WAVE;
    const double af1 = a.inst[b].af1, af2 = a.inst[b].af2;
    const TileRd<double, HX> rF{&sF[0][0]}, rG{&sG[0][0]};
    double *__restrict__ yout = a.y + fo;
    double cs = 0.0;
    double B[4];
    sep_coef(sP[cx - 2], sP[cx - 1], sP[cx], sP[cx + 1], sP[cx + 2], c1, c2, B);
    SepWin<double> wh;
    ArakawaWin<double> wg;
    wh.load(rF, rr0 + 2, cx);
    wg.load(rF, rG, rr0 + 2, cx);
#pragma unroll
    for (int q = 0; q < ROWS_PER_WAVE; ++q) {
        const int j = tile.j0 + rr0 + q;
        if (j < nv && i < nx) {
            const size_t o = (size_t)j * nx + i;
            yout[o] = a.alpha * (fa[q] * us) + wh.bracket(sA[rr0 + q], B, sep_near(KIND), sep_far(KIND));
            cs += arakawa_add<KIND>(wg, 0.0, 1.0, af1, af2);
        }
        if (q + 1 < ROWS_PER_WAVE) {
            wh.advance(rF, rr0 + q + 3, cx);
            wg.advance(rF, rG, rr0 + q + 3, cx);
        }
    }
    sS[wave][lane] = cs;
    __syncthreads();
    if (wave == 0 && i < nx)
        csum[b * cstride + (size_t)(tile.j0 / TY) * nx + i] = ((sS[0][lane] + sS[1][lane]) + sS[2][lane]) + sS[3][lane];
}

template <int MODE>
hipError_t launch_mode(vv_ctx *c, const BrArgs<double> &a)
{
    dim3 grid(br_tiles(c->p.nx, c->p.nv), c->B), block(NT);
    switch (c->p.bracket) {
    case VV_BRACKET_J1:
        launch_timed(c, bracket_kernel<VV_BRACKET_J1, MODE>, grid, block, 0, a);
        break;
    case VV_BRACKET_J2:
        launch_timed(c, bracket_kernel<VV_BRACKET_J2, MODE>, grid, block, 0, a);
        break;
    default:
        launch_timed(c, bracket_kernel<VV_BRACKET_J4, MODE>, grid, block, 0, a);
        break;
    }
    return hipGetLastError();
}

template <int MODE, typename T>
hipError_t launch_sep(vv_ctx *c, BrArgs<T> a)
{
    const dim3 grid(br_tiles(c->p.nx, c->p.nv), c->B), block(NT);
    switch (c->p.bracket) {
    case VV_BRACKET_J1: launch_timed(c, bracket_sep_kernel<VV_BRACKET_J1, MODE, T>, grid, block, 0, a); break;
    case VV_BRACKET_J2: launch_timed(c, bracket_sep_kernel<VV_BRACKET_J2, MODE, T>, grid, block, 0, a); break;
    default: launch_timed(c, bracket_sep_kernel<VV_BRACKET_J4, MODE, T>, grid, block, 0, a); break;
    }
    return hipGetLastError();
}

template <typename T>
BrArgs<T> base_args(vv_ctx *c)
{
    BrArgs<T> a{};
    a.nx = c->p.nx;
    a.nv = c->p.nv;
    a.N = c->N;
    a.inst = c->inst;
    a.gstride = (int64_t)sizeof(GmresState);
    a.h0 = c->h0;
    a.h1p = c->h1p;
    a.h1h = c->h1h;
    a.h2p = c->h2p;
    a.h2h = c->h2h;
    a.ht_inv = c->ht_inv;
    return a;
}

}  // namespace

int residual_blocks(const vv_ctx *c) { return br_tiles(c->p.nx, c->p.nv); }

hipError_t launch_residual(vv_ctx *c, const double *f, const double *fh, double *y, double *part)
{
    BrArgs<double> a = base_args<double>(c);
    a.f = f;
    a.fh = fh;
    a.y = y;
    a.part = part;
    a.pstride = c->part_stride;
    a.factor = 1.0;                 // B(Fave, H, 1.0)  (PETScNLVlasovMP.pyx:55)
    return launch_mode<MODE_RESIDUAL>(c, a);
}

hipError_t launch_residual_sep(vv_ctx *c, const double *f, const double *fh, double *y)
{
    BrArgs<double> a = base_args<double>(c);
    a.f = f;
    a.fh = fh;
    a.y = y;
    a.factor = 1.0;
    return launch_sep<MODE_RESIDUAL>(c, a);
}

hipError_t launch_jacobian_plain(vv_ctx *c, const double *u, double *y)
{
    BrArgs<double> a = base_args<double>(c);
    a.f = u;
    a.y = y;
    a.factor = 0.5;                 // B(u, H, 0.5)  (PETScNLVlasovMP.pyx:37)
    return launch_mode<MODE_JACOBIAN>(c, a);
}

hipError_t launch_jacobian(vv_ctx *c, const double *u, const double *uscale, double *y)
{
    BrArgs<double> a = base_args<double>(c);
    a.f = u;
    a.uscale = uscale;
    a.y = y;
    a.factor = 0.5;
    a.done = uscale != nullptr ? &c->gs->st.done : nullptr;
    return launch_sep<MODE_JACOBIAN>(c, a);
}

hipError_t launch_bracket_add(vv_ctx *c, const double *x, double *y, double factor)
{
    BrArgs<double> a = base_args<double>(c);
    a.f = x;
    a.y = y;
    a.factor = factor;
    return launch_mode<MODE_ACCUMULATE>(c, a);
}

hipError_t launch_bracket_t(vv_ctx *c, const double *u, const double *uscale, const double *h2d, const double *hxv,
                            double *y, double alpha, double factor)
{
    BrArgs<double> a = base_args<double>(c);
    a.f = u;
    a.uscale = uscale;
    a.h2d = h2d;
    a.hxv = hxv;
    a.y = y;
    a.alpha = alpha;
    a.factor = factor;
    a.done = uscale != nullptr ? &c->gs->st.done : nullptr;
    return launch_mode<MODE_TRANSPOSED>(c, a);
}

int band_rows(int nv) { return (nv + TY - 1) / TY; }

hipError_t launch_bracket_pair(vv_ctx *c, const double *u, const double *uscale, const double *g, double *y,
                               double alpha, double factor, double *csum, int64_t cstride)
{
    BrArgs<double> a = base_args<double>(c);
    a.f = u;
    a.uscale = uscale;
    a.h2d = g;
    a.y = y;
    a.alpha = alpha;
    a.factor = factor;
    a.done = uscale != nullptr ? &c->gs->st.done : nullptr;
    HessArgs hs{};
    if (uscale != nullptr) hs = take_update(c);
    const dim3 grid(br_tiles(c->p.nx, c->p.nv) + (hs.nb > 0 ? 1 : 0), c->B), block(NT);
    switch (c->p.bracket) {
    case VV_BRACKET_J1: launch_timed(c, bracket_pair_kernel<VV_BRACKET_J1>, grid, block, 0, a, hs, csum, cstride); break;
    case VV_BRACKET_J2: launch_timed(c, bracket_pair_kernel<VV_BRACKET_J2>, grid, block, 0, a, hs, csum, cstride); break;
    default: launch_timed(c, bracket_pair_kernel<VV_BRACKET_J4>, grid, block, 0, a, hs, csum, cstride); break;
    }
    return hipGetLastError();
}

hipError_t launch_bracket_gen(vv_ctx *c, const double *x, const double *h2d, const double *hxv, double *y,
                              double factor)
{
    BrArgs<double> a = base_args<double>(c);
    a.f = x;
    a.h2d = h2d;
    a.hxv = hxv;
    a.y = y;
    a.factor = factor;
    return launch_mode<MODE_ACCUMULATE>(c, a);
}

hipError_t launch_bracket_acc(vv_ctx *c, const double *x, const double *xscale, const double *h2d, double *y,
                              double factor, bool store, const int32_t *done)
{
    BrArgs<double> a = base_args<double>(c);
    a.f = x;
    a.uscale = xscale;
    a.h2d = h2d;
    a.y = y;
    a.factor = factor;
    a.store = store ? 1 : 0;
    a.done = done;
    return launch_mode<MODE_ACCUMULATE>(c, a);
}

hipError_t launch_jacobian32(vv_ctx *c, const float *u, const double *uscale, float *y)
{
    BrArgs<float> a = base_args<float>(c);
    a.f = u;
    a.uscale = uscale;
    a.y = y;
    a.factor = 0.5;
    a.done = uscale != nullptr ? &c->gs->st.done : nullptr;
    return launch_sep<MODE_JACOBIAN>(c, a);
}

}  // namespace vv
