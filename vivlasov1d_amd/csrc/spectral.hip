// Kinetic tensor-product preconditioner  P^-1 x = irfft_x( T_k^-1 rfft_x(x) )
// (TensorProductKinetic.pyx:146-160; TensorProductKineticFast.pyx:102-224):
//
//  rfft_kernel    real rows x[j][0..nx) -> spectrum S[k][j], k = 0..nx/2.
//                 Two real rows are packed as one complex row and transformed
//                 by an in-LDS Stockham FFT (radix 8 after up to two stages of
//                 radix 4; length 1024 as 4 x 8 x 8 x 4); the output is written
//                 mode-major (the transpose the reference does with a
//                 VecScatter is folded into the store).
//  tridiag_lu_kernel  one workgroup per mode k solves T_k c = S[k][.] along v
//                 from reciprocal LU pivots formed once per context, which are
//                 streamed (16 bytes a row, FP64); the bands are rebuilt from the
//                 mode's eigenvalue and two per-row factors.
//  tridiag_wave_kernel, tridiag_kernel  the same without pivots, for the
//                 potential form, whose bands change every step: a wavefront or
//                 a workgroup per mode, partitioned Thomas (one chunk of M rows
//                 per lane or thread) whose reduced system is solved by parallel
//                 cyclic reduction on shuffles or in LDS.
//  irfft_kernel   spectrum -> real rows, backward-normalised like
//                 numpy.fft.irfft / pyFFTW (imaginary parts of the k = 0 and
//                 k = nx/2 coefficients are ignored, as in a c2r transform).
//
// The potential form (TensorProductPotential.pyx:157-173) has the roles of x and
// v exchanged: rFFT along v down the field's columns (rfft_cols_kernel; where that
// does not apply the field is transposed, transpose_kernel, and back), one
// tridiagonal system along x per v-mode with bands from phi differences
// (potential_bands_kernel), irFFT.  The transform geometry (length, rows, modes,
// band constants) comes from the context.
//
// Every kernel is a template on the real type: double for the FP64 path,
// float for the FP32 preconditioner inside the mixed-precision GMRES cycle
// (complex64 spectrum, float twiddles; T_k's coefficients are formed in FP64
// and rounded).
#include "fft_lds.h"
#include "gmres_dev.h"

namespace vv {
namespace {

// Transform variants of the kernels below: VP8 nx = 1024 by the radix-8 plan
// with preloaded twiddles; VTWL shorter powers of two, twiddles copied to LDS;
// VLONG longer ones, twiddles from the table.
enum { VTWL = 0, VP8 = 1, VLONG = 2 };
// threads of a variant's workgroup
constexpr int vthreads(int V) { return V == VLONG ? NTL : NT; }

// LF: log2 of the first stage's radix (fft_first), which runs in registers:
// butterfly (p, j) of complex row p (real rows 2p, 2p+1) takes z_p[j + m nx/2^LF],
// exactly the elements the thread loads (coalesced along j); its twiddles are
// 1.  Every global load of the thread is issued before anything waits.
template <typename T, int V, int LF>
__global__ __launch_bounds__(vthreads(V)) void rfft_kernel(FftArgs<T> a, const T *__restrict__ x, cx_t<T> *__restrict__ spec)
{
    using C = cx_t<T>;
    const int32_t dflag = cycle_done(a.done, a.gstride);
    if (gridDim.y > 1 && dflag) return;   // batched: a finished instance skips its loads
    x += blockIdx.y * a.N;
    spec += blockIdx.y * a.S;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C *buf = reinterpret_cast<C *>(lds_raw);
    const int nx = a.nx, R = a.rows;
    // XCD-aware row-block order: the mode-major segments of neighbouring row
    // blocks share L2 lines, so they are kept on one XCD
    const int j0 = xcd_tile(blockIdx.x, gridDim.x) * R;
    constexpr int NTH = vthreads(V), RAD = 1 << LF, QB = MAXE / RAD / NTH;    // butterflies per thread
    const int lq = a.logn - LF, nq = 1 << lq;
    const int total = (R >> 1) * nq;
    T xr[QB][RAD], xi[QB][RAD];
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        const int bq = threadIdx.x + q * NTH;
        const int p = bq >> lq, j = bq & (nq - 1);
        const bool ok = bq < total;
        const bool r0 = ok && j0 + 2 * p < a.nv, r1 = ok && j0 + 2 * p + 1 < a.nv;
        const T *x0 = x + (size_t)(j0 + 2 * p) * nx + j;
#pragma unroll
        for (int m = 0; m < RAD; ++m) {
            xr[q][m] = r0 ? x0[m * nq] : T(0);
            xi[q][m] = r1 ? x0[nx + m * nq] : T(0);
        }
        if (a.add != nullptr) {
            const T *ad = a.add + (size_t)blockIdx.y * nx + j;
#pragma unroll
            for (int m = 0; m < RAD; ++m) {
                const T w = a.gamma * ad[m * nq];
                xr[q][m] += r0 ? w : T(0);
                xi[q][m] += r1 ? w : T(0);
            }
        }
    }
    FftTw<false, C> pt;
    if (V == VP8) pt.load(a.tw);
    const C *tw = tw_table<V == VTWL>(a.tw, buf + (size_t)(R >> 1) * nx, nx);
    if (dflag) return;                 // uniform over the block, before any barrier
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        const int bq = threadIdx.x + q * NTH;
        if (bq < total) {
            const int p = bq >> lq, j = bq & (nq - 1);
            C v[RAD];
#pragma unroll
            for (int m = 0; m < RAD; ++m) v[m] = cmk<C>(xr[q][m], xi[q][m]);
            if constexpr (LF == 3) dft8<false>(v);
            else dft4<false>(v[0], v[1], v[2], v[3]);
            const int z = (p << a.logn) + (j << LF);    // first stage's outputs: RAD j + m
#pragma unroll
            for (int m = 0; m < RAD; ++m) buf[swz<V == VLONG>(z + m)] = v[m];
        }
    }
    __syncthreads();
    lds_fft<false, V == VP8, 4, NTH, V == VLONG>(buf, a.logn, R >> 1, tw, pt, LF, LdsSink<C>{buf});
    store_real_spectrum<NTH>(buf, nx, R, j0, a.nv, a.pitch, spec);
}

// Jacobian-vector product fused with the forward rFFT of its rows:
// X = J u (the bracket kernel's MODE_JACOBIAN, PETScNLVlasovMP.pyx:33-37:
// Y = 0; Y += u/dt; Y += 0.5 {u, H_ave} on rows 2..nv-3) is formed in LDS row
// block by row block and transformed there, so X never goes to HBM.
// The workgroup's R rows are computed in strips of NT columns: the strip of
// u with a 2-cell halo, (R+4) x (NT+4) cells, and the x-part of H_ave are
// staged in LDS, two strips in turn (one barrier each); thread t walks column t
// of the strip down the R rows (SepWin, arakawa.h; the result is multiplied by
// the Krylov vector's scale), the values of bracket_sep_kernel bit for bit.  The
// next strip's loads are in flight during the current strip's walk, and the
// results stay in registers until the last walk is done, so the FFT buffer
// reuses the strips' LDS.  nx = 4 NT: thread t's columns over the 4 strips,
// t + m NT, are exactly the inputs of radix-4 butterfly t of the first FFT
// stage, which then runs in registers as in rfft_kernel (the same
// arithmetic, bit for bit).  nx = NT, 2 NT: the rows go to the FFT buffer and
// the transform starts from LDS (its unit twiddles can change only the sign
// of an exact zero).  R in 2, 4, 8.  1024 x 2048: 22.5 us with H staged beside u
// and the unfactored stencil, 17.5 now (FP32 16.8, 14.3).
template <int R, typename T>
struct JacStrip {
    T u[R + 4];          // own column, rows j0-2 .. j0+R+1 (0 outside the grid)
    double x[4];         // own column's x-factors
    T eu;                // halo cell (threads t < 4 (R+4))
    double ex[4];
};

template <int R, typename T>
__device__ __forceinline__ void jac_strip_load(const T *__restrict__ u, const JacRows &jr, size_t xo, int nx, int nv,
                                               int j0, int cb, JacStrip<R, T> &g)
{
    constexpr int RH = R + 4;
    const int t = threadIdx.x;
    const int i = cb + t;                              // staged column t + 2 (inside the row: nx >= cb + NT)
#pragma unroll
    for (int r = 0; r < RH; ++r) {
        const int gj = jr_row(j0, r, nv);
        g.u[r] = gj >= 0 ? u[(size_t)gj * nx + i] : T(0);
    }
    g.x[0] = jr.h1p[xo + i];
    g.x[1] = jr.h1h[xo + i];
    g.x[2] = jr.h2p[xo + i];
    g.x[3] = jr.h2h[xo + i];
    if (t < 4 * RH) {
        int hr, tc;
        jr_halo_cell(t, RH, &hr, &tc);
        const int gi = jr_col(cb, tc, nx);
        const int gj = jr_row(j0, hr, nv);
        g.eu = gj >= 0 ? u[(size_t)gj * nx + gi] : T(0);
        if (hr == 0) {
            g.ex[0] = jr.h1p[xo + gi];
            g.ex[1] = jr.h1h[xo + gi];
            g.ex[2] = jr.h2p[xo + gi];
            g.ex[3] = jr.h2h[xo + gi];
        }
    }
}

// Thread t's column of the staged strip down the R output rows (tile rows
// 2 .. R+1): J u, or 0 on rows past nv (the rFFT's zero rows).
template <int KIND, int R, typename T, typename RF>
__device__ __forceinline__ void jac_walk(const RF &rF, const T (*sA)[4], const double *sP, double c1, double c2,
                                         int j0, int nv, T ht_inv, T us, T (&res)[R])
{
    const int cx = threadIdx.x + 2;
    T B[4];
    sep_coef(sP[cx - 2], sP[cx - 1], sP[cx], sP[cx + 1], sP[cx + 2], c1, c2, B);
    SepWin<T> win;
    win.load(rF, 2, cx);
#pragma unroll
    for (int q = 0; q < R; ++q) {
        const int j = j0 + q;
        T out = T(0);
        if (j < nv) {
            out = jacobian_base(ht_inv, win.f0[2]);
            if (j >= 2 && j < nv - 2) out += win.bracket(sA[q], B, sep_near(KIND), sep_far(KIND));
            out = scaled(out, us);                     // == J of the VecScale'd Krylov vector
        }
        res[q] = out;
        if (q + 1 < R) win.advance(rF, q + 3, cx);
    }
}

// hs: the Hessenberg update of the step before, when one is due, by an extra
// first workgroup while the others go on with the vector it normalises: each
// forms the scale from the norm partials itself (they come back with the
// strip's loads).  A launch of its own took 4.9 us a step at 1024 x 2048 and
// 3-4 us with its gap on small grids.  The step that follows an instance's
// convergence then runs this kernel in vain (its later kernels return at once).
template <typename T>
constexpr size_t jac_strip_lds(int R, int NS)
{
    return (NS > 1 ? 2 : 1) * ((size_t)(R + 4) * (NT + 4) * sizeof(T) + (NT + 4) * sizeof(double));
}

template <int KIND, int R, int NS, typename T>
__device__ __forceinline__ void jac_rfft_body(FftArgs<T> a, JacRows jr, HessArgs hs, const T *__restrict__ u,
                                              cx_t<T> *__restrict__ spec)
{
    using C = cx_t<T>;
    const int extra = hs.nb > 0 ? 1 : 0;
    if (extra && blockIdx.x == 0) {
        hess_update(hs);
        return;
    }
    static_assert(NT == kJrSW, "a strip is one column per thread");
    constexpr int RH = R + 4, SP = NT + 4, nx = NS * NT;
    const int32_t dflag = extra ? hess_skip(hs) : cycle_done(a.done, a.gstride);
    if (gridDim.y > 1 && dflag) return;   // batched: a finished instance skips its loads
    const int b = blockIdx.y;
    u += b * a.N;
    spec += b * a.S;
    const size_t xo = (size_t)b * nx;
    // the FFT buffer reuses the strips' LDS: the strips' results wait in
    // registers until the last walk is done
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C *buf = reinterpret_cast<C *>(lds_raw);
    T *sF = reinterpret_cast<T *>(lds_raw);
    constexpr int NBUF = NS > 1 ? 2 : 1;               // strips in turn: one barrier each
    constexpr size_t kStrip = jac_strip_lds<T>(R, NS), kLines = (size_t)(R >> 1) * nx * sizeof(C);
    double *sP = reinterpret_cast<double *>(lds_raw + NBUF * (size_t)RH * SP * sizeof(T));
    const int nv = a.nv, t = threadIdx.x;
    const int j0 = xcd_tile((int)blockIdx.x - extra, (int)gridDim.x - extra) * R;
    // nx = NT, 2 NT: the twiddles' copy lies behind the strips and the FFT buffer
    const C *tw = tw_table<NS != 4>(a.tw, reinterpret_cast<C *>(lds_raw + (kStrip > kLines ? kStrip : kLines)), nx);
    __shared__ double red[kGdNW + 1];
    __shared__ __align__(16) T sA[R][4];
    const double nshare = extra ? norm_share(hs.part + b * hs.pstride, hs.nb) : 0.0;
    double usd = jr.uscale != nullptr && !extra
                     ? *reinterpret_cast<const double *>(reinterpret_cast<const char *>(jr.uscale) + b * a.gstride)
                     : 1.0;
    double c1, c2;
    sep_weights(KIND, jr.factor, jr.inst[b].af1, jr.inst[b].af2, c1, c2);
    JacStrip<R, T> g;
    jac_strip_load<R>(u, jr, xo, nx, nv, j0, 0, g);
    if (t < R) sep_row(jr.h0, j0 + t, nv, c1, c2, sA[t]);
    if (dflag) return;                 // uniform over the block, before any barrier
    if (extra) {
        const double ws = wave_sum(nshare);            // summed after the first strip's barrier
        if ((t & 63) == 0) red[t >> 6] = ws;
    }
    const T ht_inv = (T)jr.ht_inv;
    T us = T(1);
    T res[NS][R];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        // stage the strip: u and the x-part of H_ave
        T *cF = sF + (s & (NBUF - 1)) * RH * SP;
        double *cP = sP + (s & (NBUF - 1)) * SP;
#pragma unroll
        for (int r = 0; r < RH; ++r) cF[r * SP + t + 2] = g.u[r];
        cP[t + 2] = phi_ave(g.x[0], g.x[1], g.x[2], g.x[3]);
        if (t < 4 * RH) {
            int hr, tc;
            jr_halo_cell(t, RH, &hr, &tc);
            cF[hr * SP + tc] = g.eu;
            if (hr == 0) cP[tc] = phi_ave(g.ex[0], g.ex[1], g.ex[2], g.ex[3]);
        }
        __syncthreads();
        if (s + 1 < NS) jac_strip_load<R>(u, jr, xo, nx, nv, j0, (s + 1) * NT, g);
        if (s == 0) {
            if (extra) {
                double tot = 0.0;
                for (int w = 0; w < kGdNW; ++w) tot += red[w];
                usd = scale_of(tot);
            }
            us = (T)usd;
        }
        jac_walk<KIND, R>(TileRd<T, SP>{cF}, sA, cP, c1, c2, j0, nv, ht_inv, us, res[s]);
    }
    __syncthreads();
    // twiddles in flight during the first stage (not held through the walks)
    FftTw<false, C> pt;
    if (NS == 4) pt.load(a.tw);
    if (NS == 4) {
        // stage 0 of the transform in registers, as rfft_kernel: butterfly
        // (p, t) of complex row p (real rows 2p, 2p+1) takes columns t + m NT
#pragma unroll
        for (int p = 0; p < (R >> 1); ++p) {
            const C v0 = cmk<C>(res[0][2 * p], res[0][2 * p + 1]), v1 = cmk<C>(res[1 % NS][2 * p], res[1 % NS][2 * p + 1]);
            const C v2 = cmk<C>(res[2 % NS][2 * p], res[2 % NS][2 * p + 1]);
            const C v3 = cmk<C>(res[3 % NS][2 * p], res[3 % NS][2 * p + 1]);
            const C a0 = cadd(v0, v2), a1 = csub(v0, v2), a2 = cadd(v1, v3), d = csub(v1, v3);
            const C a3 = cmk<C>(d.y, -d.x);             // (v1 - v3) * (-i)
            C *z = buf + (p << a.logn) + (t << 2);      // stage 0 outputs: 4t + r
            z[0] = cadd(a0, a2);
            z[1] = cadd(a1, a3);
            z[2] = csub(a0, a2);
            z[3] = csub(a1, a3);
        }
    } else {
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int p = 0; p < (R >> 1); ++p) buf[p * nx + s * NT + t] = cmk<C>(res[s][2 * p], res[s][2 * p + 1]);
    }
    __syncthreads();
    lds_fft<false, NS == 4, 4>(buf, a.logn, R >> 1, tw, pt, NS == 4 ? 2 : 0, LdsSink<C>{buf});
    store_real_spectrum(buf, nx, R, j0, nv, a.pitch, spec);
}

// LDS max(R/2 nx 16, 2 (R+5)(NT+4) 8) bytes (37 KB at R = 4), so three
// workgroups per CU fit when the registers do (R <= 4; four cost register
// spills and were slower)
template <int KIND, int R, int NS, typename T>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(R <= 4 ? 3 : 2))) void jac_rfft_kernel(
    FftArgs<T> a, JacRows jr, HessArgs hs, const T *__restrict__ u, cx_t<T> *__restrict__ spec)
{
    jac_rfft_body<KIND, R, NS>(a, jr, hs, u, spec);
}

// The potential form's rFFT along v straight from the field (nv rows of nx):
// a workgroup takes R consecutive x (R, nx even), whose lines run down the
// columns.  The packed complex line p, (x = i0 + 2p, i0 + 2p + 1), is 16 bytes
// a row of the field as it lies there, so it is loaded as such; the lines of a
// 128-byte segment belong to neighbouring workgroups of one XCD, which find it
// in its L2.  The spectrum goes out x-contiguous per mode, as rfft_kernel's.
// With the inverse below it replaces a transpose before and after (4.0 us each
// and a launch at 512 x 1024).
template <typename T, int V>
__global__ __launch_bounds__(NT) void rfft_cols_kernel(FftArgs<T> a, const T *__restrict__ x,
                                                       cx_t<T> *__restrict__ spec)
{
    using C = cx_t<T>;
    const int32_t dflag = cycle_done(a.done, a.gstride);
    if (gridDim.y > 1 && dflag) return;   // batched: a finished instance skips its loads
    x += blockIdx.y * a.N;
    spec += blockIdx.y * a.S;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C *buf = reinterpret_cast<C *>(lds_raw);
    const int n = a.nx, nc = a.nv, npair = a.rows >> 1;      // line length, columns, lines
    const int i0 = xcd_tile(blockIdx.x, gridDim.x) * a.rows;
    const int total = n * npair;
    constexpr int QL = MAXE / NT;
    C z[QL];
#pragma unroll
    for (int q = 0; q < QL; ++q) {
        const int idx = threadIdx.x + q * NT;
        const int m = idx / npair, i = i0 + 2 * (idx - m * npair);
        const bool ok = idx < total && i < nc;
        const C v = *reinterpret_cast<const C *>(x + (ok ? (size_t)m * nc + i : 0));
        z[q] = ok ? v : cmk<C>(T(0), T(0));
    }
    FftTw<false, C> pt;
    if (V == VP8) pt.load(a.tw);
    const C *tw = tw_table<V == VTWL>(a.tw, buf + (size_t)npair * n, n);
    if (dflag) return;                 // uniform over the block, before any barrier
#pragma unroll
    for (int q = 0; q < QL; ++q) {
        const int idx = threadIdx.x + q * NT;
        const int m = idx / npair;
        if (idx < total) buf[(idx - m * npair) * n + m] = z[q];
    }
    __syncthreads();
    lds_fft<false, V == VP8, 4>(buf, a.logn, npair, tw, pt, 0, LdsSink<C>{buf});
    store_real_spectrum(buf, n, a.rows, i0, nc, a.pitch, spec);
}

// the same columns back: line b of the workgroup to x = i0 + 2b, i0 + 2b + 1
template <typename T>
struct IrfftColSink {
    T *y;
    int i0, n, logn, nc;
    __device__ __forceinline__ void operator()(int pos, cx_t<T> z) const
    {
        const int b = pos >> logn, m = pos & (n - 1), i = i0 + 2 * b;
        const T inv_n = T(1) / (T)n;
        if (i < nc) *reinterpret_cast<cx_t<T> *>(y + (size_t)m * nc + i) = cmk<cx_t<T>>(z.x * inv_n, z.y * inv_n);
    }
};

// Real rows 2b, 2b+1 of an irFFT workgroup from its complex transform b
// (backward-normalised by 1/nx, exact: nx is a power of two).
template <typename T>
struct IrfftSink {
    T *y;
    int j0, nx, logn, nv;
    __device__ __forceinline__ void operator()(int pos, cx_t<T> z) const
    {
        const int b = pos >> logn, i = pos & (nx - 1);
        const T inv_n = T(1) / (T)nx;
        const int r = j0 + 2 * b;
        if (r < nv) y[(size_t)r * nx + i] = z.x * inv_n;
        if (r + 1 < nv) y[(size_t)(r + 1) * nx + i] = z.y * inv_n;
    }
};

template <typename T, int V, bool COLS>
__global__ __launch_bounds__(vthreads(V)) void irfft_kernel(FftArgs<T> a, const cx_t<T> *__restrict__ spec, T *__restrict__ y)
{
    using C = cx_t<T>;
    const int32_t dflag = cycle_done(a.done, a.gstride);
    if (gridDim.y > 1 && dflag) return;   // batched: a finished instance skips its loads
    spec += blockIdx.y * a.S;
    y += blockIdx.y * a.N;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C *buf = reinterpret_cast<C *>(lds_raw);
    const int nx = a.nx, R = a.rows, nh = nx >> 1;
    const int j0 = xcd_tile(blockIdx.x, gridDim.x) * R;   // as in rfft_kernel
    const int npair = R >> 1;
    // Z_k = A_k + i B_k (k <= nx/2) and its Hermitian extension for k > nx/2;
    // every global load of the thread is issued before the LDS stores.
    const int total = (nh + 1) * npair;
    // (nx/2 + 1) R/2 <= MAXE/2 + MAXE/nx: nx >= 8 for the short lines, else >= 1024
    constexpr int NTH = vthreads(V), PER = (MAXE / 2 + (V == VTWL ? MAXE / 8 : MAXE / N8) + NTH - 1) / NTH;
    const bool p2 = (npair & (npair - 1)) == 0;
    const int lp = __ffs(npair) - 1;
    C va[PER], vb[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        if (V == VTWL && q * NTH >= total) break;   // uniform: short blocks skip the rest
        const int idx = threadIdx.x + q * NTH;
        const int k = p2 ? idx >> lp : idx / npair;
        const int ja = j0 + 2 * (idx - k * npair);
        va[q] = load_or_zero(spec, (int64_t)k * a.pitch + ja, idx < total && ja < a.nv);
        vb[q] = load_or_zero(spec, (int64_t)k * a.pitch + ja + 1, idx < total && ja + 1 < a.nv);
    }
    FftTw<true, C> pt;
    if (V == VP8) pt.load(a.tw);
    const C *tw = tw_table<V == VTWL>(a.tw, buf + (size_t)npair * nx, nx);
    if (dflag) return;                 // uniform over the block, before any barrier
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int idx = threadIdx.x + q * NTH;
        if (idx < total) {
            const int k = p2 ? idx >> lp : idx / npair;
            const int p = idx - k * npair;
            C A = va[q], B = vb[q];
            if (k == 0 || k == nh) {
                A.y = T(0);
                B.y = T(0);
            }
            const int z = p * nx;
            buf[swz<V == VLONG>(z + k)] = cmk<C>(A.x - B.y, A.y + B.x);
            if (k != 0 && k != nh) buf[swz<V == VLONG>(z + nx - k)] = cmk<C>(A.x + B.y, B.x - A.y);
        }
    }
    __syncthreads();
    // the last stage's outputs (natural order) go straight to the output rows
    if constexpr (COLS) lds_fft<true, V == VP8, 4, NTH, V == VLONG>(buf, a.logn, npair, tw, pt, 0, IrfftColSink<T>{y, j0, nx, a.logn, a.nv});
    else lds_fft<true, V == VP8, 4, NTH, V == VLONG>(buf, a.logn, npair, tw, pt, 0, IrfftSink<T>{y, j0, nx, a.logn, a.nv});
}

// Real rows of the irFFT left in the workgroup's LDS buffer itself, natural
// order (row r of the block at wr[r nx + i]), backward-normalised as in
// IrfftSink.  The last FFT stage reads every input before its barrier, so
// the buffer can take its outputs.
template <typename T>
struct RealRowsSink {
    T *wr;
    int nx, logn;
    __device__ __forceinline__ void operator()(int pos, cx_t<T> z) const
    {
        const int b = pos >> logn, i = pos & (nx - 1);
        const T inv_n = T(1) / (T)nx;
        wr[(2 * b) * nx + i] = z.x * inv_n;
        wr[(2 * b + 1) * nx + i] = z.y * inv_n;
    }
};

// The Arnoldi step's irFFT fused with the classical Gram-Schmidt dots that
// follow it: w = V_{col+1} = irfft(spec) is written to the basis and, from
// the workgroup's LDS, dotted with v_0..v_col.  The workgroup's R rows are
// one CGS slice of NT EPT 16-byte vectors (R nx = NT EPT L, nv % R == 0);
// thread t takes the slice's vectors t + q NT, and the per-slice partials
// part[slice PV + j] are summed by maxpy_norm_kernel as mdot_kernel's are.
// Where EPT equals the CGS launches' own, w and the partials are
// bit-identical to irfft_kernel followed by mdot_kernel.  What the fusion
// saves: the second read of w, one launch, and the wait for the first basis
// vectors, whose loads are in flight while the FFT stages run.
// START (col = -1): the irFFT into V_0 = P^-1 F and its norm partials, at
// part[slice]: a solve's first vector without the copy and the norm pass (8.4 +
// 6.7 us at 1024 x 2048).
template <typename T, int EPT, int PV, bool P8, bool START>
__global__ __launch_bounds__(NT) void irfft_mdot_kernel(FftArgs<T> a, const cx_t<T> *__restrict__ spec,
                                                        CgsArgs<T> g, int col)
{
    using C = cx_t<T>;
    using V = typename V16<T>::type;
    const int32_t dflag = cycle_done(a.done, a.gstride);
    if (gridDim.y > 1 && dflag) return;   // batched: a finished instance skips its loads
    spec += blockIdx.y * a.S;
    const T *basis = g.basis + blockIdx.y * g.N;
    const GmresState *gs = g.g + blockIdx.y;
    double *part = g.part + blockIdx.y * g.pstride;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C *buf = reinterpret_cast<C *>(lds_raw);
    __shared__ double red[kCgsNW][PV];
    __shared__ double s_scale[PV];
    const int nx = a.nx, R = a.rows, nh = nx >> 1;
    const int slice = xcd_tile(blockIdx.x, gridDim.x);
    const int j0 = slice * R;
    const int npair = R >> 1;
    const int nvec = col + 1;
    const int total = (nh + 1) * npair;
    // the slice's points; mode pairs (nx/2 + 1) R/2 <= PTS/4 + PTS/16 (nx >= 8)
    constexpr int PTS = NT * EPT * V16<T>::L, PER = (5 * PTS / 16 + NT - 1) / NT;
    C va[PER], vb[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int idx = threadIdx.x + q * NT;
        const int k = idx / npair;
        const int ja = j0 + 2 * (idx - k * npair);
        va[q] = load_or_zero(spec, (int64_t)k * a.pitch + ja, idx < total);
        vb[q] = load_or_zero(spec, (int64_t)k * a.pitch + ja + 1, idx < total);
    }
    const double sc = (int)threadIdx.x < nvec ? gs->scale[threadIdx.x] : 0.0;
    FftTw<true, C> pt;
    if (P8) pt.load(a.tw);
    const C *tw = tw_table<!P8>(a.tw, buf + (size_t)npair * nx, nx);
    if (dflag) return;                 // uniform over the block, before any barrier
    // the first group of basis vectors is in flight while the FFT stages run
    const int64_t nvv = g.N / V16<T>::L;
    const int64_t e0 = (int64_t)slice * NT * EPT + threadIdx.x;
    constexpr int G = cgs_group<EPT>();
    V x[G][EPT];
    load_group<EPT, G, T>(basis, g.vstride, 0, nvec, e0, nvv, x);
    if ((int)threadIdx.x < PV) s_scale[threadIdx.x] = sc;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int idx = threadIdx.x + q * NT;
        if (idx < total) {
            const int k = idx / npair;
            const int p = idx - k * npair;
            C A = va[q], B = vb[q];
            if (k == 0 || k == nh) {
                A.y = T(0);
                B.y = T(0);
            }
            C *z = buf + p * nx;
            z[k] = cmk<C>(A.x - B.y, A.y + B.x);
            if (k != 0 && k != nh) z[nx - k] = cmk<C>(A.x + B.y, B.x - A.y);
        }
    }
    __syncthreads();
    T *wr = reinterpret_cast<T *>(buf);
    lds_fft<true, P8, (PTS / 2 + 1023) / 1024>(buf, a.logn, npair, tw, pt, 0, RealRowsSink<T>{wr, nx, a.logn});

    // w of the slice: to the basis, and into registers for the dots
    const V *wl = reinterpret_cast<const V *>(wr);
    V *W = reinterpret_cast<V *>(const_cast<T *>(basis) + (size_t)nvec * g.vstride);
    V w[EPT];
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        w[q] = wl[threadIdx.x + q * NT];
        W[e0 + (int64_t)q * NT] = w[q];
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if constexpr (START) {
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < EPT; ++q)
#pragma unroll
            for (int l = 0; l < V16<T>::L; ++l) acc = __builtin_fma(vget(w[q], l), vget(w[q], l), acc);
        acc = wave_sum(acc);
        if (lane == 0) red[wave][0] = acc;
        __syncthreads();
        if (threadIdx.x == 0) {
            double s = 0.0;
            for (int wv = 0; wv < kCgsNW; ++wv) s += red[wv][0];
            part[slice] = s;
        }
        return;
    }
    for (int v = 0; v < nvec; v += G) {
        if (v > 0) load_group<EPT, G, T>(basis, g.vstride, v, nvec - v, e0, nvv, x);
#pragma unroll
        for (int gg = 0; gg < G; ++gg) {
            if (v + gg >= nvec) break;
            double acc = dot_slice<EPT, T>(w, x[gg], s_scale[v + gg]);
            acc = wave_sum(acc);
            if (lane == 0) red[wave][v + gg] = acc;
        }
    }
    __syncthreads();
    if (threadIdx.x < PV) {
        double s = 0.0;
        if ((int)threadIdx.x < nvec)
            for (int wv = 0; wv < kCgsNW; ++wv) s += red[wv][threadIdx.x];
        part[(size_t)slice * PV + threadIdx.x] = s;
    }
}

// Transforms of a length n that is not a power of two (n = 100, 201, ...):
// a direct real DFT with exact twiddle indices (k m mod n into the table of
// exp(-2 pi i m/n)), same spectrum layout and c2r semantics as the FFT
// kernels above.  O(n) work per output; the workgroup's rows and, when they
// fit 32 KiB, the twiddles are staged in LDS.  Rows are not packed in pairs,
// so `rows` may be odd.
template <typename T, bool TWL>
__global__ __launch_bounds__(NT) void rdft_kernel(FftArgs<T> a, const T *__restrict__ x, cx_t<T> *__restrict__ spec)
{
    using C = cx_t<T>;
    if (cycle_done(a.done, a.gstride)) return;      // uniform over the block, before any barrier
    x += blockIdx.y * a.N;
    spec += blockIdx.y * a.S;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int n = a.nx, R = a.rows, ld = n | 1, nk = n / 2 + 1;
    C *stw = reinterpret_cast<C *>(lds_raw);
    T *sx = reinterpret_cast<T *>(lds_raw + (TWL ? (size_t)n * sizeof(C) : 0));
    const int j0 = blockIdx.x * R;
    const int nr = a.nv - j0 < R ? a.nv - j0 : R;   // rows of this block
    for (int e = threadIdx.x; e < nr * n; e += NT) {
        const int r = e / n;
        sx[r * ld + (e - r * n)] = x[(size_t)j0 * n + e];
    }
    if (TWL)
        for (int e = threadIdx.x; e < n; e += NT) stw[e] = a.tw[e];
    __syncthreads();
    const C *tw = TWL ? stw : a.tw;
    for (int o = threadIdx.x; o < nk * nr; o += NT) {
        const int k = o / nr, r = o - k * nr;
        const T *xr = sx + r * ld;
        T re = T(0), im = T(0);
        for (int m = 0, t = 0; m < n; ++m) {
            const C w = tw[t];
            re += xr[m] * w.x;
            im += xr[m] * w.y;
            t += k;
            if (t >= n) t -= n;
        }
        spec[(size_t)k * a.pitch + j0 + r] = cmk<C>(re, im);
    }
}

// y[j][m] = (Re X_0 + 2 sum_{k=1}^{(n-1)/2} Re(X_k e^{2 pi i k m/n}) [+ Re X_{n/2} (-1)^m]) / n
template <typename T, bool TWL>
__global__ __launch_bounds__(NT) void irdft_kernel(FftArgs<T> a, const cx_t<T> *__restrict__ spec, T *__restrict__ y)
{
    using C = cx_t<T>;
    if (cycle_done(a.done, a.gstride)) return;      // uniform over the block, before any barrier
    spec += blockIdx.y * a.S;
    y += blockIdx.y * a.N;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int n = a.nx, R = a.rows, nk = n / 2 + 1, K = (n - 1) / 2;
    C *stw = reinterpret_cast<C *>(lds_raw);
    C *ss = reinterpret_cast<C *>(lds_raw + (TWL ? (size_t)n * sizeof(C) : 0));
    const int j0 = blockIdx.x * R;
    const int nr = a.nv - j0 < R ? a.nv - j0 : R;
    for (int e = threadIdx.x; e < nk * nr; e += NT) {
        const int k = e / nr, r = e - k * nr;
        C v = spec[(size_t)k * a.pitch + j0 + r];
        if (k == 0 || 2 * k == n) v.y = T(0);
        ss[r * nk + k] = v;
    }
    if (TWL)
        for (int e = threadIdx.x; e < n; e += NT) stw[e] = a.tw[e];
    __syncthreads();
    const C *tw = TWL ? stw : a.tw;
    const T inv_n = T(1) / (T)n;
    for (int o = threadIdx.x; o < nr * n; o += NT) {
        const int r = o / n, m = o - r * n;
        const C *X = ss + r * nk;
        T acc = T(0);
        for (int k = 1, t = m; k <= K; ++k) {
            const C w = tw[t];
            acc += X[k].x * w.x + X[k].y * w.y;
            t += m;
            if (t >= n) t -= n;
        }
        T v = X[0].x + T(2) * acc;
        if (!(n & 1)) v += (m & 1) ? -X[n / 2].x : X[n / 2].x;
        y[(size_t)j0 * n + o] = v * inv_n;
    }
}

struct TriArgs {
    int nv;           // system size
    int P;            // chunks (threads), power of two
    int64_t S, pitch, gstride;
    const double2 *eigen;
    const double *gm, *g0, *gp;
    int64_t cstride;         // instance stride of gm/g0/gp (0: shared)
    double clo, cmid, chi;   // band constants (kinetic 0.5, 1.0, 0.5; potential 1.0, 2.0, 1.0)
    const InstConst *inst;   // band factor afpc of instance blockIdx.y
    double ht_inv;
    const int32_t *done;
};

// Row j of T_k (KineticFast.pyx:248-272): sub a_j = diagm[j] (j >= 1),
// diagonal b_j = diag[j], super c_j = diagp[j] (j <= nv-2); rows past nv are
// identity rows that pad the system to P*M unknowns.  The coefficients are
// formed in FP64 (as the reference forms its band matrix) and rounded to C.
// TR: row j of the conjugate transpose T_k^H (sub conj(c_{j-1}), diagonal
// conj(b_j), super conj(a_{j+1})), the mode-k block of the transposed real
// operator P^T (P^-T x = irfft(T_k^-H rfft(x)): transposing a real
// x-circulant operator maps its symbol at k to the conjugate at -k).
// the three real per-row factors row j of T_k (or of T_k^H, TR) uses
template <bool TR>
__device__ __forceinline__ void tri_load(const TriArgs &a, int j, double &lo, double &mid, double &hi)
{
    // Clamped addresses and no selects on the loaded values: nothing here
    // waits on a load, so the loads of all rows of a chunk are in flight
    // together.  Values loaded for rows outside the system are never used:
    // tri_row makes those rows identity rows and drops the sub-diagonal of
    // row 0 and the super-diagonal of row nv-1.
    const int jc = j < a.nv ? j : a.nv - 1;
    if (!TR) {
        lo = a.gm[jc];
        hi = a.gp[jc];
    } else {
        lo = a.gp[jc > 0 ? jc - 1 : 0];
        hi = a.gm[jc < a.nv - 1 ? jc + 1 : jc];
    }
    mid = a.g0[jc];
}

template <bool TR, typename C>
__device__ __forceinline__ void tri_row(const TriArgs &a, double af, double2 e, int j, double lo, double mid,
                                        double hi, C &aj, C &bj, C &cj)
{
    using R = typename C::value_type;
    const double ey = TR ? -e.y : e.y;
    if (j < a.nv) {
        aj = (j > 0) ? cmk<C>((R)(((e.x * a.clo) * lo) * af), (R)(((ey * a.clo) * lo) * af)) : cmk<C>(R(0), R(0));
        bj = cmk<C>((R)(((e.x * a.cmid) * mid) * af + a.ht_inv), (R)(((ey * a.cmid) * mid) * af));
        cj = (j < a.nv - 1) ? cmk<C>((R)(((e.x * a.chi) * hi) * af), (R)(((ey * a.chi) * hi) * af))
                            : cmk<C>(R(0), R(0));
    } else {
        aj = cmk<C>(R(0), R(0));
        bj = cmk<C>(R(1), R(0));
        cj = cmk<C>(R(0), R(0));
    }
}

template <int M, typename T, bool TR>
__global__ __launch_bounds__(NT) void tridiag_kernel(TriArgs a, cx_t<T> *__restrict__ spec)
{
    using C = cx_t<T>;
    const int32_t dflag = cycle_done(a.done, a.gstride);
    if (gridDim.y > 1 && dflag) return;   // batched: a finished instance skips its loads
    spec += blockIdx.y * a.S;
    a.gm += blockIdx.y * a.cstride;
    a.g0 += blockIdx.y * a.cstride;
    a.gp += blockIdx.y * a.cstride;
    const double af = a.inst[blockIdx.y].afpc;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C *sd = reinterpret_cast<C *>(lds_raw);   // P*(M+1): right-hand sides / solution, chunk c at c*(M+1)
    __shared__ C sa[NT], sb[NT], sc[NT], se[NT];
    const int k = blockIdx.x;
    const double2 e = a.eigen[k];
    const int P = a.P, n = P * M;
    const C zero = cmk<C>(T(0), T(0));
    C *S = spec + (size_t)k * a.pitch;
    const int c = threadIdx.x;
    double clo[M], cmid[M], chi[M];   // per-row factors of the thread's chunk
    {
        // n = P*M <= NT*M: every load of the thread in flight before the LDS stores
        C v[M];
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const int j = threadIdx.x + q * NT;
            v[q] = load_or_zero(S, j, j < a.nv);
        }
        if (dflag) return;             // uniform over the block, before any barrier
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const int j = threadIdx.x + q * NT;
            if (j < n) sd[j + j / M] = v[q];      // one pad slot per chunk: no bank conflicts
        }
    }
    __syncthreads();

    C Am[M], Cm[M], Dm[M];
    C ae, be, ce;          // coefficients of the chunk's last row
    if (c < P) {
        const int s = c * M, ls = c * (M + 1);
        // forward sweep: y_j + c'_j y_{j+1} = d'_j - a'_j y_{s-1}
        C aj, bj, cj;
        tri_load<TR>(a, s, clo[0], cmid[0], chi[0]);
        tri_row<TR>(a, af, e, s, clo[0], cmid[0], chi[0], aj, bj, cj);
        C r = crecip(bj);
        Cm[0] = cmul(cj, r);
        Dm[0] = cmul(sd[ls], r);
        Am[0] = cmul(aj, r);
#pragma unroll
        for (int q = 1; q < M; ++q) {
            tri_load<TR>(a, s + q, clo[q], cmid[q], chi[q]);
            tri_row<TR>(a, af, e, s + q, clo[q], cmid[q], chi[q], aj, bj, cj);
            if (q == M - 1) {
                ae = aj;
                be = bj;
                ce = cj;
            }
            if (q < M - 1) {
                r = crecip(csub(bj, cmul(aj, Cm[q - 1])));
                Cm[q] = cmul(cj, r);
                Dm[q] = cmul(csub(sd[ls + q], cmul(aj, Dm[q - 1])), r);
                Am[q] = cneg(cmul(cmul(aj, Am[q - 1]), r));
            }
        }
        // backward sweep over rows s..e-1: y_j = D_j - A_j y_{s-1} - C_j y_e
#pragma unroll
        for (int q = M - 3; q >= 0; --q) {
            Dm[q] = csub(Dm[q], cmul(Cm[q], Dm[q + 1]));
            Am[q] = csub(Am[q], cmul(Cm[q], Am[q + 1]));
            Cm[q] = cneg(cmul(Cm[q], Cm[q + 1]));
        }
        // publish the first row of the chunk for the neighbour below
        sa[c] = Am[0];
        sc[c] = Cm[0];
        se[c] = Dm[0];
    }
    __syncthreads();
    // reduced equation of chunk c in the chunk-last unknowns E:
    //   alpha E_{c-1} + beta E_c + gamma E_{c+1} = delta
    C al = zero, bt = cmk<C>(T(1), T(0)), gm = zero, dl = zero;
    if (c < P) {
        const C dE = sd[c * (M + 1) + M - 1];
        al = cneg(cmul(ae, Am[M - 2]));
        bt = csub(be, cmul(ae, Cm[M - 2]));
        dl = csub(dE, cmul(ae, Dm[M - 2]));
        if (c + 1 < P) {
            bt = csub(bt, cmul(ce, sa[c + 1]));
            gm = cneg(cmul(ce, sc[c + 1]));
            dl = csub(dl, cmul(ce, se[c + 1]));
        }
    }
    __syncthreads();
    // parallel cyclic reduction on the P reduced unknowns
    for (int st = 1; st < P; st <<= 1) {
        if (c < P) {
            sa[c] = al;
            sb[c] = bt;
            sc[c] = gm;
            se[c] = dl;
        }
        __syncthreads();
        if (c < P) {
            C nal = zero, ngm = zero;
            C nbt = bt, ndl = dl;
            if (c - st >= 0) {
                const C k1 = cdiv(al, sb[c - st]);
                nal = cneg(cmul(sa[c - st], k1));
                nbt = csub(nbt, cmul(sc[c - st], k1));
                ndl = csub(ndl, cmul(se[c - st], k1));
            }
            if (c + st < P) {
                const C k2 = cdiv(gm, sb[c + st]);
                ngm = cneg(cmul(sc[c + st], k2));
                nbt = csub(nbt, cmul(sa[c + st], k2));
                ndl = csub(ndl, cmul(se[c + st], k2));
            }
            al = nal;
            gm = ngm;
            bt = nbt;
            dl = ndl;
        }
        __syncthreads();
    }
    if (c < P) se[c] = cdiv(dl, bt);     // E_c = y at the chunk's last row
    __syncthreads();
    if (c < P) {
        const int ls = c * (M + 1);
        const C Eprev = (c > 0) ? se[c - 1] : zero;
        const C Eown = se[c];
#pragma unroll
        for (int q = 0; q < M - 1; ++q)
            sd[ls + q] = csub(csub(Dm[q], cmul(Am[q], Eprev)), cmul(Cm[q], Eown));
        sd[ls + M - 1] = Eown;
    }
    __syncthreads();
    for (int j = threadIdx.x; j < a.nv; j += NT) S[j] = sd[j + j / M];
}

// The same solve for systems of up to 64 M rows (M <= 8), a wavefront per mode
// and four modes a workgroup: lane c owns the chunk of M rows, and the reduced
// system of the 64 chunk-last unknowns is solved by parallel cyclic reduction
// on shuffles, six steps without a barrier (the workgroup form: eight steps of
// two barriers and twelve LDS accesses at 512 rows, 12.0 us for the 513 modes
// of 512 x 1024).  A lane past the end holds identity rows; the couplings of a
// lane without a neighbour at the step's distance are zero by then, so no step
// needs a branch.
template <typename C> __device__ __forceinline__ C shfl_up_cx(C v, int off)
{
    return cmk<C>(__shfl_up(v.x, off), __shfl_up(v.y, off));
}
template <typename C> __device__ __forceinline__ C shfl_down_cx(C v, int off)
{
    return cmk<C>(__shfl_down(v.x, off), __shfl_down(v.y, off));
}
template <int CTRL, int ROWS = 0xf, typename C> __device__ __forceinline__ C dpp_cx(C v)
{
    return cmk<C>(dpp_move<CTRL, ROWS>(v.x), dpp_move<CTRL, ROWS>(v.y));
}
template <typename C> __device__ __forceinline__ C lane_cx(C v, int lane)
{
    return cmk<C>(read_lane(v.x, lane), read_lane(v.y, lane));
}

__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <int M, typename T, bool TR>
__global__ __launch_bounds__(NT) void tridiag_wave_kernel(TriArgs a, int nmodes, cx_t<T> *__restrict__ spec)
{
    using C = cx_t<T>;
    const int32_t dflag = cycle_done(a.done, a.gstride);
    if (dflag) return;                    // uniform over the launch's instance
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int k = blockIdx.x * (NT / 64) + wave;
    if (k >= nmodes) return;              // whole wavefronts; no barrier below
    a.gm += blockIdx.y * a.cstride;
    a.g0 += blockIdx.y * a.cstride;
    a.gp += blockIdx.y * a.cstride;
    const double af = a.inst[blockIdx.y].afpc;
    __shared__ C lds[NT / 64][64 * (M + 1)];
    C *sd = lds[wave];                    // chunk c at c (M + 1)
    const double2 e = a.eigen[k];
    C *S = spec + blockIdx.y * a.S + (size_t)k * a.pitch;
    const C zero = cmk<C>(T(0), T(0));
    double lo[M], mid[M], hi[M];
    {
        C v[M];
#pragma unroll
        for (int q = 0; q < M; ++q) v[q] = load_or_zero(S, lane + 64 * q, lane + 64 * q < a.nv);
#pragma unroll
        for (int q = 0; q < M; ++q) tri_load<TR>(a, lane * M + q, lo[q], mid[q], hi[q]);
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const int j = lane + 64 * q;
            sd[j + j / M] = v[q];
        }
    }
    wave_lds_fence();
    const int ls = lane * (M + 1);
    C Am[M], Cm[M], Dm[M], ae, be, ce;
    {
        // forward sweep: y_j + c'_j y_{j+1} = d'_j - a'_j y_{s-1}
        C aj, bj, cj;
        tri_row<TR>(a, af, e, lane * M, lo[0], mid[0], hi[0], aj, bj, cj);
        C r = crecip(bj);
        Cm[0] = cmul(cj, r);
        Dm[0] = cmul(sd[ls], r);
        Am[0] = cmul(aj, r);
#pragma unroll
        for (int q = 1; q < M; ++q) {
            tri_row<TR>(a, af, e, lane * M + q, lo[q], mid[q], hi[q], aj, bj, cj);
            if (q < M - 1) {
                r = crecip(csub(bj, cmul(aj, Cm[q - 1])));
                Cm[q] = cmul(cj, r);
                Dm[q] = cmul(csub(sd[ls + q], cmul(aj, Dm[q - 1])), r);
                Am[q] = cneg(cmul(cmul(aj, Am[q - 1]), r));
            } else {
                ae = aj;
                be = bj;
                ce = cj;
            }
        }
        // backward sweep over the chunk but its last row: y_j = D_j - A_j y_{s-1} - C_j y_e
#pragma unroll
        for (int q = M - 3; q >= 0; --q) {
            Dm[q] = csub(Dm[q], cmul(Cm[q], Dm[q + 1]));
            Am[q] = csub(Am[q], cmul(Cm[q], Am[q + 1]));
            Cm[q] = cneg(cmul(Cm[q], Cm[q + 1]));
        }
    }
    // reduced equation of the chunk in the chunk-last unknowns E:
    //   al E_{c-1} + bt E_c + gm E_{c+1} = dl  (lane 63's next is its own, times ce = 0)
    const C na = shfl_down_cx(Am[0], 1), nc = shfl_down_cx(Cm[0], 1), nd = shfl_down_cx(Dm[0], 1);
    if (lane == 63) ce = zero;
    C al = cneg(cmul(ae, Am[M - 2]));
    C bt = csub(csub(be, cmul(ae, Cm[M - 2])), cmul(ce, na));
    C gm = cneg(cmul(ce, nc));
    C dl = csub(csub(sd[ls + M - 1], cmul(ae, Dm[M - 2])), cmul(ce, nd));
#pragma unroll 1
    for (int st = 1; st < 64; st <<= 1) {
        const C ri = crecip(bt);
        const C k1 = cmul(al, shfl_up_cx(ri, st)), k2 = cmul(gm, shfl_down_cx(ri, st));
        const C ua = shfl_up_cx(al, st), ug = shfl_up_cx(gm, st), ud = shfl_up_cx(dl, st);
        const C da = shfl_down_cx(al, st), dg = shfl_down_cx(gm, st), dd = shfl_down_cx(dl, st);
        bt = csub(csub(bt, cmul(ug, k1)), cmul(da, k2));
        dl = csub(csub(dl, cmul(ud, k1)), cmul(dd, k2));
        al = cneg(cmul(ua, k1));
        gm = cneg(cmul(dg, k2));
        if (lane < 2 * st) al = zero;
        if (lane + 2 * st > 63) gm = zero;
    }
    const C E = cdiv(dl, bt);             // y at the chunk's last row
    C Ep = shfl_up_cx(E, 1);
    if (lane == 0) Ep = zero;
#pragma unroll
    for (int q = 0; q < M - 1; ++q) sd[ls + q] = csub(csub(Dm[q], cmul(Am[q], Ep)), cmul(Cm[q], E));
    sd[ls + M - 1] = E;
    wave_lds_fence();
#pragma unroll
    for (int q = 0; q < M; ++q) {
        const int j = lane + 64 * q;
        if (j < a.nv) S[j] = sd[j + j / M];
    }
}

// ---- kinetic solve with precomputed pivots ---------------------------------
// The kinetic T_k do not change during a run, so their LU factors are formed
// once per context (KineticFast.pyx:88-90 factors once with zgbtrf as well):
// without pivoting (the bands are diagonally dominant: |Im b_j| is about
// twice |a_j| + |c_j|, so zgbtrf's partial pivoting swaps no rows),
//   u_0 = b_0,  u_j = b_j - (a_j / u_{j-1}) c_{j-1},   rp[k][j] = 1 / u_j,
// in FP64, one thread per mode (and instance), stored as C (FP64, or rounded
// for the FP32 solve).  The solve then has no divisions:
//   forward   y_j = d_j - (a_j rp_{j-1}) y_{j-1},
//   backward  x_j = rp_j (y_j - c_j x_{j+1}),
// a_j and c_j being rebuilt from e_k and the per-row factors as in tri_row.
template <typename T>
__global__ __launch_bounds__(NT) void tridiag_factor_kernel(TriArgs a, int nmodes, int TN, int M, cx_t<T> *__restrict__ rp)
{
    const int k = blockIdx.x * NT + threadIdx.x;
    if (k >= nmodes) return;
    const double af = a.inst[blockIdx.y].afpc;
    const double2 e = a.eigen[k];
    // chunk-interleaved: the pivot of row j = t M + q at q NT + t, so that the
    // solve's thread t, which owns rows t M .. t M + M - 1, loads them
    // coalesced; rows nv .. NT M - 1 hold zero
    const int L = TN * M;
    cx_t<T> *R = rp + ((size_t)blockIdx.y * nmodes + k) * L;
    double lo, mid, hi;
    double2 aj, bj, cj;
    tri_load<false>(a, 0, lo, mid, hi);
    tri_row<false>(a, af, e, 0, lo, mid, hi, aj, bj, cj);
    double2 r = crecip(bj);
    R[0] = cmk<cx_t<T>>((T)r.x, (T)r.y);
    for (int j = 1; j < a.nv; ++j) {
        const double2 cprev = cj;
        tri_load<false>(a, j, lo, mid, hi);
        tri_row<false>(a, af, e, j, lo, mid, hi, aj, bj, cj);
        r = crecip(csub(bj, cmul(cmul(aj, r), cprev)));
        R[(j % M) * TN + j / M] = cmk<cx_t<T>>((T)r.x, (T)r.y);
    }
    for (int j = a.nv; j < L; ++j) R[(j % M) * TN + j / M] = cmk<cx_t<T>>(T(0), T(0));
}

// The affine maps y -> A + B y of a wavefront's lanes composed: (ea, eb) the map
// of the lanes before this one (REV: after it) applied to the value entering
// the wavefront, and (ta, tb) that of all 64 lanes, in every lane.  Rows of 16 by DPP, then the four rows'
// maps, which every lane reads and composes itself: ~350 cycles where six steps
// of four-double shuffles took ~900.
template <bool REV, typename C>
__device__ __forceinline__ void affine_scan(C A, C B, int lane, C &ea, C &eb, C &ta, C &tb)
{
    using R = typename C::value_type;
    const C zero = cmk<C>(R(0), R(0)), one = cmk<C>(R(1), R(0));
    const int r = lane & 15, row = lane >> 4;
    constexpr int DIR = REV ? kDppShl : kDppShr;
    const int pos = REV ? 15 - r : r;              // lanes of the row that come before
    {
        const C pa = dpp_cx<DIR + 1>(A), pb = dpp_cx<DIR + 1>(B);
        if (pos >= 1) {
            A = cadd(A, cmul(B, pa));
            B = cmul(B, pb);
        }
    }
    {
        const C pa = dpp_cx<DIR + 2>(A), pb = dpp_cx<DIR + 2>(B);
        if (pos >= 2) {
            A = cadd(A, cmul(B, pa));
            B = cmul(B, pb);
        }
    }
    {
        const C pa = dpp_cx<DIR + 4>(A), pb = dpp_cx<DIR + 4>(B);
        if (pos >= 4) {
            A = cadd(A, cmul(B, pa));
            B = cmul(B, pb);
        }
    }
    {
        const C pa = dpp_cx<DIR + 8>(A), pb = dpp_cx<DIR + 8>(B);
        if (pos >= 8) {
            A = cadd(A, cmul(B, pa));
            B = cmul(B, pb);
        }
    }
    ea = dpp_cx<DIR + 1>(A);
    eb = dpp_cx<DIR + 1>(B);
    if (pos == 0) {
        ea = zero;
        eb = one;
    }
    // rows in the order the recurrence meets them: last lane of each holds its map
    C pa = zero, pb = one;                         // of the rows before this lane's
    ta = zero;
    tb = one;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int rr = REV ? 3 - q : q;
        if (row == rr) {
            pa = ta;
            pb = tb;
        }
        const int last = REV ? 16 * rr : 16 * rr + 15;
        const C ra = lane_cx(A, last), rb = lane_cx(B, last);
        ta = cadd(ra, cmul(rb, ta));
        tb = cmul(rb, tb);
    }
    ea = cadd(ea, cmul(eb, pa));
    eb = cmul(eb, pb);
}

// One workgroup of TN threads per mode (blockIdx.x) and instance (blockIdx.y);
// thread t owns the chunk of M rows [t M, t M + M), in registers.  The
// spectrum row turns from coalesced to chunks and back in each wavefront's own
// part of LDS; the pivots and the band factors lie in chunk-interleaved order
// (read in row order, the factors' 8 M-byte strides took 64 lines a load: 73 us
// at 2048 x 4096 where it is 42 now, 17.2 and 14.0 at 1024 x 2048).  Across
// chunks the recurrences are affine maps y_out = A + B y_in, composed by a scan
// over the wavefront's lanes (affine_scan) and over the wavefronts (one LDS
// exchange), first forward, then backward; no thread waits on a division.
// Bound by memory and by its phases, which the two or three workgroups of a CU
// go through nearly together: 50 MB in 14 us at 1024 x 2048, 201 MB in 42 at
// 2048 x 4096.
// M = 16: the backward sweep's factors are loaded after the forward scan, so
// the kernel keeps 256 registers and two workgroups a CU (111 us with spills, 54
// with one workgroup).
// TR: T_k^H x = d from the same pivots, U^H y = d then L^H x = y:
//   y_j = conj(rp_j) (d_j - conj(c_{j-1}) y_{j-1}),  x_j = y_j - conj(a_{j+1} rp_j) x_{j+1}
// (cyclic reduction with divisions took 7.7 us at 256 x 512, the forward solve
// 5.1).
template <int TN, int M, typename T, bool TR>
__global__ __launch_bounds__(TN) __attribute__((amdgpu_waves_per_eu(2))) void tridiag_lu_kernel(
    TriArgs a, const cx_t<T> *__restrict__ rp, cx_t<T> *__restrict__ spec)
{
    using C = cx_t<T>;
    const int32_t dflag = cycle_done(a.done, a.gstride);
    if (gridDim.y > 1 && dflag) return;   // batched: a finished instance skips its loads
    const int k = blockIdx.x;
    const double af = a.inst[blockIdx.y].afpc;
    const double2 e = a.eigen[k];
    C *S = spec + blockIdx.y * a.S + (size_t)k * a.pitch;
    // pivots and band factors in chunk-interleaved order: thread t's rows
    // t M + q at q TN + t, loaded coalesced straight into registers
    const C *Rg = rp + ((size_t)blockIdx.y * gridDim.x + k) * (TN * M);
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int NW = TN / 64;
    __shared__ C wa[2 * NW], wb[2 * NW];
    const C zero = cmk<C>(T(0), T(0));
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    // the wavefront's own 64 (M + 1) slots: its right-hand side, then its x
    C *sd = reinterpret_cast<C *>(lds_raw) + wave * (64 * (M + 1));
    const int w0 = wave * 64 * M + lane;          // first of the rows lane loads and stores: w0 + 64 q
    C rpv[M], d[M];                               // pivots of rows t M .. t M + M - 1; d, then y
    double gf[M], gb[M];                          // factors of the forward and the backward sweeps' diagonals (0: none)
    C rprev = zero;                               // pivot of row t M - 1 (last row of chunk t - 1)
    const double *gfw = TR ? a.gp : a.gm, *gbw = TR ? a.gm : a.gp;
    double gprev = 0.0, gnext = 0.0;              // TR: super-diagonal of row t M - 1, sub-diagonal of row t M + M
#pragma unroll
    for (int q = 0; q < M; ++q) {
        const int j = w0 + 64 * q;
        d[q] = load_or_zero(S, j, j < a.nv);
    }
#pragma unroll
    for (int q = 0; q < M; ++q) {
        rpv[q] = Rg[q * TN + t];
        gf[q] = gfw[q * TN + t];
        if (M < 16) gb[q] = gbw[q * TN + t];
    }
    if constexpr (TR) {
        gprev = a.gp[t > 0 ? (M - 1) * TN + t - 1 : TN * M - 1];
        gnext = a.gm[t < TN - 1 ? t + 1 : 0];   // row 0's is 0
    } else {
        rprev = load_or_zero(Rg, (M - 1) * TN + t - 1, t > 0);
    }
    if (dflag) return;                            // uniform over the block, before any barrier
#pragma unroll
    for (int q = 0; q < M; ++q) {
        const int j = lane + 64 * q;
        sd[j + j / M] = d[q];                     // one pad slot per chunk
    }
    wave_lds_fence();
    const int ls = lane * (M + 1);
#pragma unroll
    for (int q = 0; q < M; ++q) d[q] = sd[ls + q];
    const double exl = e.x * a.clo, eyl = e.y * a.clo, exh = e.x * a.chi, eyh = e.y * a.chi;
    auto sub = [&](double g) { return cmk<C>((T)((exl * g) * af), (T)((eyl * g) * af)); };
    auto sup = [&](double g) { return cmk<C>((T)((exh * g) * af), (T)((eyh * g) * af)); };
    // the recurrences' coefficients: y_j = w_j d_j - m_j y_{j-1} (w = 1 but for TR),
    // x_j = z_j y_j - n_j x_{j+1} (z = 1 for TR)
    auto mcoef = [&](int q) {
        if constexpr (TR) return cmul(cconj(rpv[q]), cconj(sup(q > 0 ? gf[q > 0 ? q - 1 : 0] : gprev)));
        else return cmul(sub(gf[q]), q > 0 ? rpv[q > 0 ? q - 1 : 0] : rprev);
    };
    auto ncoef = [&](int q) {
        if constexpr (TR) return cconj(cmul(sub(q < M - 1 ? gb[q < M - 1 ? q + 1 : q] : gnext), rpv[q]));
        else return cmul(rpv[q], sup(gb[q]));
    };
    if constexpr (TR) {
#pragma unroll
        for (int q = 0; q < M; ++q) d[q] = cmul(cconj(rpv[q]), d[q]);
    }
    // long chunks: the coefficients are formed again for each sweep (the
    // factors look changed) instead of held, 8 M more registers
    auto again = [&](double (&g)[M]) {
        if constexpr (M >= 8) {
#pragma unroll
            for (int q = 0; q < M; ++q) asm volatile("" : "+v"(g[q]));
        }
    };
    // forward map of the chunk: y_{s+M-1} = A + B y_{s-1}
    C A = d[0], B = cneg(mcoef(0));
#pragma unroll
    for (int q = 1; q < M; ++q) {
        const C m = mcoef(q);
        A = csub(d[q], cmul(m, A));
        B = cneg(cmul(m, B));
    }
    again(gf);
    C ea, eb, ta, tb;                             // maps of lanes 0 .. lane-1, of the wavefront
    affine_scan<false>(A, B, lane, ea, eb, ta, tb);
    if (lane == 0) {
        wa[wave] = ta;
        wb[wave] = tb;
    }
    __syncthreads();
    C y = zero;                                   // y at the end of the previous wavefronts' rows
    for (int w = 0; w < wave; ++w) y = cadd(wa[w], cmul(wb[w], y));
    y = cadd(ea, cmul(eb, y));                    // y_{s-1}
    if constexpr (M >= 16) {                      // on their way during the sweep
#pragma unroll
        for (int q = 0; q < M; ++q) gb[q] = gbw[q * TN + t];
    }
#pragma unroll
    for (int q = 0; q < M; ++q) {
        y = csub(d[q], cmul(mcoef(q), y));
        d[q] = y;
    }
    // backward map of the chunk: x_s = G + D x_{s+M}
    auto zy = [&](int q) {
        if constexpr (TR) return d[q];
        else return cmul(rpv[q], d[q]);
    };
    C G = zy(M - 1), D = cneg(ncoef(M - 1));
#pragma unroll
    for (int q = M - 2; q >= 0; --q) {
        const C rc = ncoef(q);
        G = csub(zy(q), cmul(rc, G));
        D = cneg(cmul(rc, D));
    }
    again(gb);
    C xa, xb;                                     // maps of lanes lane+1 .. 63
    affine_scan<true>(G, D, lane, xa, xb, ta, tb);
    if (lane == 0) {
        wa[NW + wave] = ta;
        wb[NW + wave] = tb;
    }
    __syncthreads();
    C x = zero;                                   // x at the first row of the next wavefronts
    for (int w = NW - 1; w > wave; --w) x = cadd(wa[NW + w], cmul(wb[NW + w], x));
    x = cadd(xa, cmul(xb, x));                    // x_{s+M}
#pragma unroll
    for (int q = M - 1; q >= 0; --q) {
        if constexpr (TR) x = csub(d[q], cmul(ncoef(q), x));
        else x = cmul(rpv[q], csub(d[q], cmul(sup(gb[q]), x)));
        sd[ls + q] = x;
    }
    wave_lds_fence();
#pragma unroll
    for (int q = 0; q < M; ++q) {
        const int j = lane + 64 * q;
        if (w0 + 64 * q < a.nv) S[w0 + 64 * q] = sd[j + j / M];
    }
}

// out = in^T for every instance (blockIdx.z): in holds R rows of C, out C
// rows of R.  32x32 tiles through LDS (one pad column), loads and stores
// coalesced along the contiguous axis of each side; clamped addresses for the
// edge tiles.  The potential preconditioner transforms along v, so it works on
// the transposed field.
template <typename T>
__global__ __launch_bounds__(NT) void transpose_kernel(const T *__restrict__ in, T *__restrict__ out, int R, int C,
                                                       int64_t N, const int32_t *done, int64_t gstride)
{
    const int b = blockIdx.z;
    if (done != nullptr && *reinterpret_cast<const int32_t *>(reinterpret_cast<const char *>(done) + b * gstride))
        return;
    in += (size_t)b * N;
    out += (size_t)b * N;
    __shared__ T tile[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;      // 32 x 8
    T v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = r0 + ty + 8 * q, cc = c0 + tx;
        const bool ok = r < R && cc < C;
        const T t = in[(size_t)(ok ? r : 0) * C + (ok ? cc : 0)];
        v[q] = ok ? t : T(0);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) tile[ty + 8 * q][tx] = v[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int oc = c0 + ty + 8 * q, orr = r0 + tx;
        if (oc < C && orr < R) out[(size_t)oc * R + orr] = tile[tx][ty + 8 * q];
    }
}

// The phi differences of the potential bands (TensorProductPotentialFast.pyx:
// 243-252): gm_i = phi_i - phi_{i-1}, g0_i = phi_{i+1} - phi_{i-1},
// gp_i = phi_{i+1} - phi_i, indices mod nx, per instance (blockIdx.y).
__global__ __launch_bounds__(NT) void potential_bands_kernel(const double *__restrict__ phi, int nx,
                                                             double *__restrict__ gm, double *__restrict__ g0,
                                                             double *__restrict__ gp)
{
    const size_t o = (size_t)blockIdx.y * nx;
    const int i = blockIdx.x * NT + threadIdx.x;
    if (i >= nx) return;
    const int im = i == 0 ? nx - 1 : i - 1, ip = i == nx - 1 ? 0 : i + 1;
    gm[o + i] = phi[o + i] - phi[o + im];
    g0[o + i] = phi[o + ip] - phi[o + im];
    gp[o + i] = phi[o + ip] - phi[o + i];
}

template <typename T>
hipError_t transpose_t(vv_ctx *c, const T *in, T *out, bool back, const int32_t *done)
{
    const int R = back ? c->p.nx : c->p.nv, C = back ? c->p.nv : c->p.nx;
    dim3 grid((C + 31) / 32, (R + 31) / 32, c->B);
    hipLaunchKernelGGL(transpose_kernel<T>, grid, dim3(NT), 0, c->stream, in, out, R, C, c->N, done,
                       (int64_t)sizeof(GmresState));
    return hipGetLastError();
}

// v-rows per FFT workgroup: the context's tuned value, else the largest that
// fits 64 KiB of LDS while the launch keeps >= 512 workgroups
int fft_rows(const vv_ctx *c)
{
    if (c->tune_fft_rows > 0) return c->tune_fft_rows;
    const int nx = c->fft_n, nv = c->fft_rows;
    int R = 2;
    while (2 * R * nx <= 8192) R *= 2;
    if (R < 2) R = 2;
    while (R > 2 && (nv + R - 1) / R < 512) R >>= 1;
    return R;
}

// The DFT kernels' launch: rows per workgroup = fft_rows(c) capped so that
// the rows take <= 32 KiB of LDS; twiddles in LDS when they fit 32 KiB.
template <typename T>
FftArgs<T> dft_args(vv_ctx *c, const cx_t<T> *tw, const int32_t *done, bool *twl, size_t *lds)
{
    const int n = c->fft_n;
    const size_t row_bytes = (size_t)(n + 2) * sizeof(T);   // >= (n | 1) reals and >= (n/2 + 1) complex
    int R = fft_rows(c);
    const int cap = (int)(32768 / row_bytes);
    if (R > cap) R = cap > 1 ? cap : 1;
    *twl = (size_t)n * sizeof(cx_t<T>) <= 32768;
    *lds = (*twl ? (size_t)n * sizeof(cx_t<T>) : 0) + (size_t)R * row_bytes;
    return FftArgs<T>{n, 0, c->fft_rows, R, c->N, spec_stride(c), spec_pitch(c), (int64_t)sizeof(GmresState), tw, done};
}

// LDS of an FFT kernel: the packed rows, and the twiddles' copy below 1024
template <typename T>
size_t fft_lds(const FftArgs<T> &a)
{
    return ((size_t)(a.rows >> 1) * a.nx + (a.nx < N8 ? a.nx : 0)) * sizeof(cx_t<T>);
}

// Lines that the direct real DFT transforms at least as fast as the row blocks:
// those of a single stage, and short ones on small grids, where a pass over LDS
// between two barriers costs more than a sum of n terms.  rFFT up to 64 points
// (direct and row blocks, us: 50 x 128 4.2 and 5.0, 50 x 4096 5.5 and 6.0, 63 x 128
// 4.6 and 5.0; 72 x 128 5.0 and 4.9, 80 x 1024 6.3 and 5.3), irFFT up to 96 (36 x 4096
// 4.1 and 5.4, 80 x 1024 5.1 and 6.4, 96 x 128 4.9 and 5.1; 99 x 1024 5.9 and 5.1), both
// up to 2^23 products (irFFT 63 x 2048 4.6 and 4.9; 50 x 4096 5.2 and 4.6, 80 x 2048 6.7
// and 6.2).
constexpr int kDirectFwd = 64, kDirectInv = 96;
bool direct_lines(const vv_ctx *c, int longest)
{
    const int64_t n = c->fft_n;
    return !dft_rows(c) || (n <= longest && n * n * c->fft_rows * c->B <= 1 << 23);
}

// the row-block transforms of lengths with a plan
hipError_t row_rfft(vv_ctx *c, const double *x, double2 *spec, const int32_t *done, const double *add, double gamma)
{
    return launch_row_rfft(c, x, spec, done, add, gamma);
}
hipError_t row_rfft(vv_ctx *c, const float *x, float2 *spec, const int32_t *done, const float *, float)
{
    return launch_row_rfft32(c, x, spec, done);
}
hipError_t row_irfft(vv_ctx *c, const double2 *spec, double *y, const int32_t *done) { return launch_row_irfft(c, spec, y, done); }
hipError_t row_irfft(vv_ctx *c, const float2 *spec, float *y, const int32_t *done) { return launch_row_irfft32(c, spec, y, done); }

template <typename T>
hipError_t rdft_t(vv_ctx *c, const cx_t<T> *tw, const T *x, cx_t<T> *spec, const int32_t *done)
{
    bool twl;
    size_t lds;
    const FftArgs<T> a = dft_args<T>(c, tw, done, &twl, &lds);
    const dim3 grid((a.nv + a.rows - 1) / a.rows, c->B);
    if (twl) launch_timed(c, rdft_kernel<T, true>, grid, dim3(NT), (uint32_t)lds, a, x, spec);
    else launch_timed(c, rdft_kernel<T, false>, grid, dim3(NT), (uint32_t)lds, a, x, spec);
    return hipGetLastError();
}

template <typename T>
hipError_t irdft_t(vv_ctx *c, const cx_t<T> *tw, const cx_t<T> *spec, T *y, const int32_t *done)
{
    bool twl;
    size_t lds;
    const FftArgs<T> a = dft_args<T>(c, tw, done, &twl, &lds);
    const dim3 grid((a.nv + a.rows - 1) / a.rows, c->B);
    if (twl) launch_timed(c, irdft_kernel<T, true>, grid, dim3(NT), (uint32_t)lds, a, spec, y);
    else launch_timed(c, irdft_kernel<T, false>, grid, dim3(NT), (uint32_t)lds, a, spec, y);
    return hipGetLastError();
}

template <typename T>
hipError_t rfft_t(vv_ctx *c, const cx_t<T> *tw, const T *x, cx_t<T> *spec, const int32_t *done,
                  const T *add = nullptr, T gamma = T(0))
{
    if (dft_rows(c) && (add != nullptr || !direct_lines(c, kDirectFwd))) return row_rfft(c, x, spec, done, add, gamma);
    if (c->fft_n & (c->fft_n - 1)) return add != nullptr ? hipErrorInvalidValue : rdft_t<T>(c, tw, x, spec, done);
    FftArgs<T> a{c->fft_n, c->logn, c->fft_rows, fft_rows(c), c->N, spec_stride(c), spec_pitch(c),
                 (int64_t)sizeof(GmresState), tw, done, add, gamma};
    const int nb = (a.nv + a.rows - 1) / a.rows;
    const uint32_t lds = (uint32_t)fft_lds<T>(a);
    const dim3 grid(nb, c->B), block(NT);
    const bool first8 = fft_first(a.logn) == 3;
    if (a.nx == N8) launch_timed(c, rfft_kernel<T, VP8, 2>, grid, block, lds, a, x, spec);
    else if (a.nx < N8 && first8) launch_timed(c, rfft_kernel<T, VTWL, 3>, grid, block, lds, a, x, spec);
    else if (a.nx < N8) launch_timed(c, rfft_kernel<T, VTWL, 2>, grid, block, lds, a, x, spec);
    else if (first8) launch_timed(c, rfft_kernel<T, VLONG, 3>, grid, dim3(NTL), lds, a, x, spec);
    else launch_timed(c, rfft_kernel<T, VLONG, 2>, grid, dim3(NTL), lds, a, x, spec);
    return hipGetLastError();
}

template <int KIND, int R, int NS, typename T>
void jac_rfft_launch(vv_ctx *c, const FftArgs<T> &a, const JacRows &jr, const T *u, cx_t<T> *spec)
{
    const size_t fft = (size_t)(R >> 1) * a.nx * sizeof(cx_t<T>);
    const size_t strip = jac_strip_lds<T>(R, NS);
    HessArgs hs{};
    if (jr.uscale != nullptr) hs = take_update(c);     // a Krylov vector: its scale is due
    const dim3 grid((a.nv + R - 1) / R + (hs.nb > 0 ? 1 : 0), c->B);
    const size_t tws = NS != 4 ? a.nx * sizeof(cx_t<T>) : 0;
    launch_timed(c, jac_rfft_kernel<KIND, R, NS, T>, grid, dim3(NT), (uint32_t)((fft > strip ? fft : strip) + tws), a,
                 jr, hs, u, spec);
}

template <int KIND, int R, typename T>
void jac_rfft_width(vv_ctx *c, const FftArgs<T> &a, const JacRows &jr, const T *u, cx_t<T> *spec)
{
    if (a.nx == 4 * NT) jac_rfft_launch<KIND, R, 4>(c, a, jr, u, spec);
    else if (a.nx == 2 * NT) jac_rfft_launch<KIND, R, 2>(c, a, jr, u, spec);
    else jac_rfft_launch<KIND, R, 1>(c, a, jr, u, spec);
}

template <int R, typename T>
void jac_rfft_kind(vv_ctx *c, const FftArgs<T> &a, const JacRows &jr, const T *u, cx_t<T> *spec)
{
    switch (c->p.bracket) {
    case VV_BRACKET_J1: jac_rfft_width<VV_BRACKET_J1, R>(c, a, jr, u, spec); break;
    case VV_BRACKET_J2: jac_rfft_width<VV_BRACKET_J2, R>(c, a, jr, u, spec); break;
    default: jac_rfft_width<VV_BRACKET_J4, R>(c, a, jr, u, spec); break;
    }
}

template <typename T>
hipError_t jac_rfft_t(vv_ctx *c, const cx_t<T> *tw, const T *u, const double *uscale, cx_t<T> *spec,
                      const int32_t *done)
{
    const int R = jac_rfft_rows(c);
    const FftArgs<T> a{c->fft_n, c->logn, c->fft_rows, R, c->N, spec_stride(c), spec_pitch(c), (int64_t)sizeof(GmresState), tw, done};
    const JacRows jr{uscale, c->h0, c->h1p, c->h1h, c->h2p, c->h2h, c->inst, c->ht_inv, 0.5};
    switch (R) {
    case 2: jac_rfft_kind<2>(c, a, jr, u, spec); break;
    case 4: jac_rfft_kind<4>(c, a, jr, u, spec); break;
    case 8: jac_rfft_kind<8>(c, a, jr, u, spec); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename T>
hipError_t irfft_t(vv_ctx *c, const cx_t<T> *tw, const cx_t<T> *spec, T *y, const int32_t *done)
{
    // the row blocks store pairs: a y that is not aligned for them takes the direct DFT too
    if (!direct_lines(c, kDirectInv) && (reinterpret_cast<uintptr_t>(y) & (2 * sizeof(T) - 1)) == 0)
        return row_irfft(c, spec, y, done);
    if (c->fft_n & (c->fft_n - 1)) return irdft_t<T>(c, tw, spec, y, done);
    FftArgs<T> a{c->fft_n, c->logn, c->fft_rows, fft_rows(c), c->N, spec_stride(c), spec_pitch(c),
                 (int64_t)sizeof(GmresState), tw, done};
    const int nb = (a.nv + a.rows - 1) / a.rows;
    const uint32_t lds = (uint32_t)fft_lds<T>(a);
    const dim3 grid(nb, c->B), block(NT);
    if (a.nx == N8) launch_timed(c, irfft_kernel<T, VP8, false>, grid, block, lds, a, spec, y);
    else if (a.nx < N8) launch_timed(c, irfft_kernel<T, VTWL, false>, grid, block, lds, a, spec, y);
    else launch_timed(c, irfft_kernel<T, VLONG, false>, grid, dim3(NTL), lds, a, spec, y);
    return hipGetLastError();
}

// The potential form's transforms on the field's columns: lines of a power of
// two, pairs of columns aligned in every row.
template <typename T>
bool cols_apply(const vv_ctx *c, const T *f)
{
    return c->tb != nullptr && c->dft.n == 0 && (c->fft_n & (c->fft_n - 1)) == 0 && (c->fft_rows & 1) == 0 &&
           (reinterpret_cast<uintptr_t>(f) & (2 * sizeof(T) - 1)) == 0;
}

template <typename T>
hipError_t rfft_cols_t(vv_ctx *c, const cx_t<T> *tw, const T *x, cx_t<T> *spec, const int32_t *done)
{
    FftArgs<T> a{c->fft_n, c->logn, c->fft_rows, fft_rows(c), c->N, spec_stride(c), spec_pitch(c), (int64_t)sizeof(GmresState), tw, done};
    const uint32_t lds = (uint32_t)fft_lds<T>(a);
    const dim3 grid((a.nv + a.rows - 1) / a.rows, c->B), block(NT);
    if (a.nx == N8) launch_timed(c, rfft_cols_kernel<T, VP8>, grid, block, lds, a, x, spec);
    else if (a.nx < N8) launch_timed(c, rfft_cols_kernel<T, VTWL>, grid, block, lds, a, x, spec);
    else launch_timed(c, rfft_cols_kernel<T, VLONG>, grid, block, lds, a, x, spec);
    return hipGetLastError();
}

template <typename T>
hipError_t irfft_cols_t(vv_ctx *c, const cx_t<T> *tw, const cx_t<T> *spec, T *y, const int32_t *done)
{
    FftArgs<T> a{c->fft_n, c->logn, c->fft_rows, fft_rows(c), c->N, spec_stride(c), spec_pitch(c), (int64_t)sizeof(GmresState), tw, done};
    const uint32_t lds = (uint32_t)fft_lds<T>(a);
    const dim3 grid((a.nv + a.rows - 1) / a.rows, c->B), block(NT);
    if (a.nx == N8) launch_timed(c, irfft_kernel<T, VP8, true>, grid, block, lds, a, spec, y);
    else if (a.nx < N8) launch_timed(c, irfft_kernel<T, VTWL, true>, grid, block, lds, a, spec, y);
    else launch_timed(c, irfft_kernel<T, VLONG, true>, grid, dim3(NTL), lds, a, spec, y);
    return hipGetLastError();
}

// 16-byte vectors per thread of the slice one irFFT workgroup covers when the
// fused irFFT + dots kernel applies (power-of-two nx <= 4 NT, the kinetic
// form, full workgroups, R nx = NT EPT L with EPT in 1, 2, 4, 8), else 0
template <typename T>
int irfft_mdot_ept(const vv_ctx *c)
{
    const int nx = c->fft_n;
    constexpr int L = V16<T>::L;
    if (!c->fuse || (nx & (nx - 1)) || nx > 4 * NT || c->tb != nullptr) return 0;
    const int R = fft_rows(c);
    if (c->fft_rows % R || c->N % L) return 0;
    const int64_t pts = (int64_t)R * nx;
    if (pts % (NT * L)) return 0;
    const int64_t ept = pts / (NT * L);
    return (ept == 1 || ept == 2 || ept == 4 || ept == 8) ? (int)ept : 0;
}

template <typename T, int EPT>
void irfft_mdot_launch(vv_ctx *c, const FftArgs<T> &a, dim3 grid, size_t lds, const cx_t<T> *spec,
                       const CgsArgs<T> &g, int col)
{
    const bool p8 = a.nx == N8;
    const uint32_t l = (uint32_t)lds;
    if constexpr (sizeof(T) == 8) {
        if (col < 0) {
            if (p8) launch_timed(c, irfft_mdot_kernel<T, EPT, 32, true, true>, grid, dim3(NT), l, a, spec, g, col);
            else launch_timed(c, irfft_mdot_kernel<T, EPT, 32, false, true>, grid, dim3(NT), l, a, spec, g, col);
            return;
        }
    }
    if (c->p.restart < 32) {
        if (p8) launch_timed(c, irfft_mdot_kernel<T, EPT, 32, true, false>, grid, dim3(NT), l, a, spec, g, col);
        else launch_timed(c, irfft_mdot_kernel<T, EPT, 32, false, false>, grid, dim3(NT), l, a, spec, g, col);
    } else {
        if (p8) launch_timed(c, irfft_mdot_kernel<T, EPT, 64, true, false>, grid, dim3(NT), l, a, spec, g, col);
        else launch_timed(c, irfft_mdot_kernel<T, EPT, 64, false, false>, grid, dim3(NT), l, a, spec, g, col);
    }
}

template <typename T>
hipError_t irfft_mdot_t(vv_ctx *c, const cx_t<T> *tw, const cx_t<T> *spec, const T *basis, int col,
                        const int32_t *done)
{
    const int ept = irfft_mdot_ept<T>(c);
    FftArgs<T> a{c->fft_n, c->logn, c->fft_rows, fft_rows(c), c->N, spec_stride(c), spec_pitch(c),
                 (int64_t)sizeof(GmresState), tw, done};
    const int nb = a.nv / a.rows;
    const size_t lds = fft_lds<T>(a);
    const CgsArgs<T> g{basis, c->N, c->vs, col < 0 ? norm_partials(c) : c->partial, c->part_stride, c->gs, 0, nb};
    const dim3 grid(nb, c->B);
    switch (ept) {
    case 8: irfft_mdot_launch<T, 8>(c, a, grid, lds, spec, g, col); break;
    case 4: irfft_mdot_launch<T, 4>(c, a, grid, lds, spec, g, col); break;
    case 2: irfft_mdot_launch<T, 2>(c, a, grid, lds, spec, g, col); break;
    case 1: irfft_mdot_launch<T, 1>(c, a, grid, lds, spec, g, col); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename T>
const cx_t<T> *lu_factors(const vv_ctx *c);
template <> const double2 *lu_factors<double>(const vv_ctx *c) { return c->lu64; }
template <> const float2 *lu_factors<float>(const vv_ctx *c) { return c->lu32; }

template <typename T, bool TR>
hipError_t tridiag_lu_t(vv_ctx *c, cx_t<T> *spec, const int32_t *done)
{
    TriArgs a{c->fft_rows, NT, spec_stride(c), spec_pitch(c), (int64_t)sizeof(GmresState), c->eigen, c->lu_gm, nullptr, c->lu_gp,
              c->coef_stride, c->cf_lo, c->cf_mid, c->cf_hi, c->inst, c->ht_inv, done};
    const int TN = lu_threads(c->fft_rows), M = lu_rows(c->fft_rows);
    const size_t lds = (size_t)TN * (M + 1) * sizeof(cx_t<T>);
    const cx_t<T> *rp = lu_factors<T>(c);
    dim3 grid(c->nmodes, c->B), block(TN);
#define VV_TRI(TN_, M_) launch_timed(c, tridiag_lu_kernel<TN_, M_, T, TR>, grid, block, (uint32_t)lds, a, rp, spec)
    if (TN == 64) {
        if (M == 1) VV_TRI(64, 1);
        else VV_TRI(64, 2);
    } else if (TN == 128) {
        if (M == 2) VV_TRI(128, 2);
        else VV_TRI(128, 4);
    } else {
        if (M == 4) VV_TRI(256, 4);
        else if (M == 8) VV_TRI(256, 8);
        else VV_TRI(256, 16);
    }
#undef VV_TRI
    return hipGetLastError();
}

template <typename T, bool TR>
hipError_t tridiag_wave_t(vv_ctx *c, cx_t<T> *spec, const int32_t *done)
{
    TriArgs a{c->fft_rows, 64, spec_stride(c), spec_pitch(c), (int64_t)sizeof(GmresState), c->eigen, c->gm, c->g0, c->gp,
              c->coef_stride, c->cf_lo, c->cf_mid, c->cf_hi, c->inst, c->ht_inv, done};
    const dim3 grid((c->nmodes + NT / 64 - 1) / (NT / 64), c->B), block(NT);
    if (c->fft_rows <= 128) launch_timed(c, tridiag_wave_kernel<2, T, TR>, grid, block, 0, a, c->nmodes, spec);
    else if (c->fft_rows <= 256) launch_timed(c, tridiag_wave_kernel<4, T, TR>, grid, block, 0, a, c->nmodes, spec);
    else launch_timed(c, tridiag_wave_kernel<8, T, TR>, grid, block, 0, a, c->nmodes, spec);
    return hipGetLastError();
}

template <typename T, bool TR = false>
hipError_t tridiag_t(vv_ctx *c, cx_t<T> *spec, const int32_t *done)
{
    if (lu_factors<T>(c) != nullptr) return tridiag_lu_t<T, TR>(c, spec, done);
    if (c->fft_rows <= 512) return tridiag_wave_t<T, TR>(c, spec, done);
    const int P = 256, m = (c->fft_rows + 255) / 256, M = m <= 4 ? 4 : (m <= 8 ? 8 : 16);
    TriArgs a{c->fft_rows, P, spec_stride(c), spec_pitch(c), (int64_t)sizeof(GmresState), c->eigen, c->gm, c->g0, c->gp,
              c->coef_stride, c->cf_lo, c->cf_mid, c->cf_hi, c->inst, c->ht_inv, done};
    const size_t lds = (size_t)P * (M + 1) * sizeof(cx_t<T>);
    dim3 grid(c->nmodes, c->B), block(NT);
    switch (M) {
    case 4: launch_timed(c, tridiag_kernel<4, T, TR>, grid, block, (uint32_t)lds, a, spec); break;
    case 8: launch_timed(c, tridiag_kernel<8, T, TR>, grid, block, (uint32_t)lds, a, spec); break;
    default: launch_timed(c, tridiag_kernel<16, T, TR>, grid, block, (uint32_t)lds, a, spec); break;
    }
    return hipGetLastError();
}

}  // namespace

// The pivoted solve's threads per mode and rows per thread.  Every wavefront
// pays for two scans whatever its rows, so short systems take few wavefronts
// (64 x 128: 4.0 us by one of 2 rows a lane, 4.5 by 256 threads of which half
// hold no row; 1025 modes of 256 rows: 6.9 by 128 threads, 9.2 by 256; of 512:
// 10.0 and 11.2), long ones 256 threads (513 modes of 2048 rows: 14.0 us by 256
// threads of 8 rows, 15.7 by 512 of 4, 16.1 by 128 of 16; 1025 of 4096: 42, 56
// by 512 of 8).
int lu_threads(int nv) { return nv <= 128 ? 64 : nv <= 512 ? 128 : NT; }

int lu_rows(int nv)
{
    const int m = (nv + lu_threads(nv) - 1) / lu_threads(nv);
    return m <= 1 ? 1 : m <= 2 ? 2 : m <= 4 ? 4 : m <= 8 ? 8 : 16;
}

// pivots stored per mode (threads x rows per thread, chunk-interleaved)
int lu_pivots_per_mode(int nv) { return lu_threads(nv) * lu_rows(nv); }

int fft_rows_of(const vv_ctx *c) { return fft_rows(c); }

int fft_blocks(vv_ctx *c)
{
    const int R = fft_rows(c);
    return (c->fft_rows + R - 1) / R;
}

hipError_t launch_rfft(vv_ctx *c, const double *x, double2 *spec, const int32_t *done, const double *add, double gamma)
{
    return rfft_t<double>(c, c->twiddle, x, spec, done, add, gamma);
}

// Rows per workgroup of the fused J u + rFFT (its own choice: the spectrum's
// layout does not depend on it): the largest of 8, 4, 2 that still leaves
// >= 6 workgroups per CU (fewer halo rows per output row; batched contexts),
// else the FFT kernels' rows when those are 2, 4 or 8, else 2.  Measured at
// 512x1024 with 22 instances: 108 / 82 / 80 us at 2 / 4 / 8 rows (unfactored
// stencil); a single 1024x2048 instance: 21.0 / 17.2 us at 2 / 4 rows.
int jac_rfft_rows(const vv_ctx *c)
{
    const int nx = c->fft_n;
    if (!c->fuse || c->tb != nullptr || nx != c->p.nx || (nx & (nx - 1)) || nx < NT || nx > 4 * NT) return 0;
    for (int R = 8; R >= 2; R >>= 1)
        if ((int64_t)((c->fft_rows + R - 1) / R) * c->B >= 6 * 256) return R;
    const int R = fft_rows(c);
    return (R == 2 || R == 4 || R == 8) ? R : 2;
}

hipError_t launch_jac_rfft(vv_ctx *c, const double *u, const double *uscale, double2 *spec, const int32_t *done)
{
    return jac_rfft_t<double>(c, c->twiddle, u, uscale, spec, done);
}

hipError_t launch_jac_rfft32(vv_ctx *c, const float *u, const double *uscale, float2 *spec, const int32_t *done)
{
    return jac_rfft_t<float>(c, c->twiddle32, u, uscale, spec, done);
}

hipError_t launch_irfft(vv_ctx *c, const double2 *spec, double *y, const int32_t *done)
{
    return irfft_t<double>(c, c->twiddle, spec, y, done);
}

int irfft_mdot_rows(const vv_ctx *c, bool fp32)
{
    return (fp32 ? irfft_mdot_ept<float>(c) : irfft_mdot_ept<double>(c)) > 0 ? c->fft_rows / fft_rows(c) : 0;
}

hipError_t launch_irfft_mdot(vv_ctx *c, const double2 *spec, int col, const int32_t *done)
{
    return irfft_mdot_t<double>(c, c->twiddle, spec, c->basis, col, done);
}

hipError_t launch_irfft_start(vv_ctx *c, const double2 *spec)
{
    return irfft_mdot_t<double>(c, c->twiddle, spec, c->basis, -1, nullptr);
}

hipError_t launch_irfft_mdot32(vv_ctx *c, const float2 *spec, int col, const int32_t *done)
{
    return irfft_mdot_t<float>(c, c->twiddle32, spec, c->basis32, col, done);
}

hipError_t launch_tridiag_k(vv_ctx *c, double2 *spec, const int32_t *done)
{
    return tridiag_t<double>(c, spec, done);
}

hipError_t launch_tridiag_t(vv_ctx *c, double2 *spec, const int32_t *done)
{
    return tridiag_t<double, true>(c, spec, done);
}

hipError_t launch_rfft32(vv_ctx *c, const float *x, float2 *spec, const int32_t *done)
{
    return rfft_t<float>(c, c->twiddle32, x, spec, done);
}

hipError_t launch_irfft32(vv_ctx *c, const float2 *spec, float *y, const int32_t *done)
{
    return irfft_t<float>(c, c->twiddle32, spec, y, done);
}

hipError_t launch_tridiag32(vv_ctx *c, float2 *spec, const int32_t *done)
{
    return tridiag_t<float>(c, spec, done);
}

hipError_t launch_tridiag_factor(vv_ctx *c, double2 *rp64, float2 *rp32)
{
    TriArgs a{c->fft_rows, NT, spec_stride(c), spec_pitch(c), (int64_t)sizeof(GmresState), c->eigen, c->gm, c->g0, c->gp,
              c->coef_stride, c->cf_lo, c->cf_mid, c->cf_hi, c->inst, c->ht_inv, nullptr};
    dim3 grid((c->nmodes + NT - 1) / NT, c->B);
    const int M = lu_rows(c->fft_rows);
    if (rp64) hipLaunchKernelGGL(tridiag_factor_kernel<double>, grid, dim3(NT), 0, c->stream, a, c->nmodes, lu_threads(c->fft_rows), M, rp64);
    if (rp32) hipLaunchKernelGGL(tridiag_factor_kernel<float>, grid, dim3(NT), 0, c->stream, a, c->nmodes, lu_threads(c->fft_rows), M, rp32);
    return hipGetLastError();
}

hipError_t launch_transpose(vv_ctx *c, const double *in, double *out, bool back, const int32_t *done)
{
    return transpose_t<double>(c, in, out, back, done);
}

hipError_t launch_transpose32(vv_ctx *c, const float *in, float *out, bool back, const int32_t *done)
{
    return transpose_t<float>(c, in, out, back, done);
}

bool potential_cols(const vv_ctx *c, const double *f) { return cols_apply<double>(c, f); }
bool potential_cols32(const vv_ctx *c, const float *f) { return cols_apply<float>(c, f); }
hipError_t launch_rfft_cols(vv_ctx *c, const double *x, double2 *spec, const int32_t *done)
{
    return rfft_cols_t<double>(c, c->twiddle, x, spec, done);
}
hipError_t launch_irfft_cols(vv_ctx *c, const double2 *spec, double *y, const int32_t *done)
{
    return irfft_cols_t<double>(c, c->twiddle, spec, y, done);
}
hipError_t launch_rfft_cols32(vv_ctx *c, const float *x, float2 *spec, const int32_t *done)
{
    return rfft_cols_t<float>(c, c->twiddle32, x, spec, done);
}
hipError_t launch_irfft_cols32(vv_ctx *c, const float2 *spec, float *y, const int32_t *done)
{
    return irfft_cols_t<float>(c, c->twiddle32, spec, y, done);
}

hipError_t launch_potential_bands(vv_ctx *c, const double *phi)
{
    hipLaunchKernelGGL(potential_bands_kernel, dim3((c->p.nx + NT - 1) / NT, c->B), dim3(NT), 0, c->stream, phi,
                       c->p.nx, c->gm, c->g0, c->gp);
    return hipGetLastError();
}

}  // namespace vv
