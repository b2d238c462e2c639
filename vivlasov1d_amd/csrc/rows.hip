// Row blocks of the kinetic preconditioner for short x-lengths (powers of two
// up to 512) and for composite ones up to 2048 (primes: see rows_apply): a
// workgroup owns RW consecutive v-rows (all of x), forms what is to be
// transformed in LDS (J u, the residual F(f), or rows as they are), transforms
// it there and stores the spectrum mode-major; and back: spectrum -> rows,
// written once and dotted with the Krylov basis from LDS.
//
// The pairs of rows are packed as complex lines.  Powers of two go through the
// Stockham FFT of fft_lds.h; any other length through a mixed-radix one of the
// same shape whose stages sum their r inputs directly (radices up to 64, or
// the prime where it is larger), twiddles from an LDS copy of the table of
// exp(-2 pi i m/n) at exact indices m: n sum(r) complex products a line, so of
// two real rows (201 = 3 x 67: 70 a point of the line), where a direct real DFT
// takes n^2 real by complex ones for the two.  A prime's single stage does twice
// the direct one's arithmetic.
//
// The strip kernel of spectral.hip keeps nx = 256, 512, 1024 (compile-time
// width, the first FFT stage in registers) for J u; this one serves the rest:
// 64 x 128 to 128 x 256 grids and the decimal and odd ones, whose steps are bound
// by the number of launches.
#include <vector>

#include "fft_lds.h"
#include "gmres_dev.h"

namespace vv {
namespace {

// ---- mixed-radix transform --------------------------------------------------

// x / d for x < 2^14, d <= 2^12 (m = floor(2^32 / d) + 1: the excess x (m d -
// 2^32) <= x d < 2^32 never carries)
__device__ __forceinline__ int div_by(int x, uint32_t m) { return (int)__umulhi((uint32_t)x, m); }

// nb lines of length n = p.n in src, through the plan's stages between src and
// dst (LDS buffers of nb n); the last stage's outputs go to `last` (line,
// natural index, value), which may write the buffer it does not read.  Stage
// with radix r after sub-transforms of length Ns:
//   out[(t - k) r + k + p Ns] = sum_q in[t + q n/r] W_n^(q (k + p Ns) n/(Ns r)),
// k = t mod Ns, t < n/r, p < r; consecutive threads take consecutive t, so the
// inputs are read without bank conflicts.
template <bool INV, typename C, typename Sink>
__device__ __forceinline__ void dft_lines(C *src, C *dst, int nb, const DftPlan &p, const C *tw, const Sink &last)
{
    using R = typename C::value_type;
    const int n = p.n, total = nb * n;
    for (int s = 0; s < p.stages; ++s) {
        const int r = p.r[s], Ns = p.ns[s], nr = p.nr[s], step0 = p.step[s];
        const bool fin = s == p.stages - 1;
        for (int idx = threadIdx.x; idx < total; idx += NT) {
            const int b = div_by(idx, p.mn), o = idx - b * n;
            const int pp = nr > 1 ? div_by(o, p.mnr[s]) : o, t = o - pp * nr;
            const int k = Ns > 1 ? t - div_by(t, p.mns[s]) * Ns : 0;
            const int e = (k + pp * Ns) * step0;          // < n
            const C *x = src + b * n + t;
            R re0 = x[0].x, im0 = x[0].y, re1 = R(0), im1 = R(0);
            int i = e;                                     // q e mod n
            int q = 1;
            for (; q + 8 <= r; q += 8) {                   // 16 LDS reads in flight
                C v[8], w[8];
#pragma unroll
                for (int m = 0; m < 8; ++m) {
                    v[m] = x[(q + m) * nr];
                    w[m] = tw[i];
                    i += e;
                    i = i >= n ? i - n : i;
                }
#pragma unroll
                for (int m = 0; m < 8; m += 2) {
                    const R wa = INV ? -w[m].y : w[m].y, wb = INV ? -w[m + 1].y : w[m + 1].y;
                    re0 += v[m].x * w[m].x - v[m].y * wa;
                    im0 += v[m].x * wa + v[m].y * w[m].x;
                    re1 += v[m + 1].x * w[m + 1].x - v[m + 1].y * wb;
                    im1 += v[m + 1].x * wb + v[m + 1].y * w[m + 1].x;
                }
            }
            for (; q < r; ++q) {
                const C v = x[q * nr], w = tw[i];
                const R wy = INV ? -w.y : w.y;
                re0 += v.x * w.x - v.y * wy;
                im0 += v.x * wy + v.y * w.x;
                i += e;
                i = i >= n ? i - n : i;
            }
            const C v = cmk<C>(re0 + re1, im0 + im1);
            const int to = (t - k) * r + k + pp * Ns;
            if (fin) last(b, to, v);
            else dst[b * n + to] = v;
        }
        __syncthreads();
        C *h = src;
        src = dst;
        dst = h;
    }
}

// The transform of a row kernel by its kind: powers of two up to 512, or mixed radix.
constexpr int kFftPre = 0, kDft = 1;

template <typename C>
struct LineSink {
    C *buf;
    int n;
    __device__ __forceinline__ void operator()(int b, int i, C v) const { buf[b * n + i] = v; }
};

// R real rows' spectra from their packed transforms, any length
template <typename C>
__device__ __forceinline__ void store_rows_spectrum(const C *buf, int n, int R, int j0, int nv, int64_t pitch,
                                                    C *__restrict__ spec)
{
    using T = typename C::value_type;
    const int nk = n / 2 + 1;
    const T half = T(0.5);
    const uint32_t mR = 0xffffffffu / (uint32_t)R + 1;
    for (int idx = threadIdx.x; idx < nk * R; idx += NT) {
        const int k = div_by(idx, mR);
        const int r = idx - k * R;
        if (j0 + r >= nv) continue;
        const C *z = buf + (r >> 1) * n;
        const C zk = z[k];
        const C zm = z[k == 0 ? 0 : n - k];
        C out;
        if ((r & 1) == 0) out = cmk<C>((zk.x + zm.x) * half, (zk.y - zm.y) * half);
        else out = cmk<C>((zk.y + zm.y) * half, (zm.x - zk.x) * half);
        spec[(size_t)k * pitch + j0 + r] = out;
    }
}

// ---- forward ----------------------------------------------------------------

enum { F_JAC = 0, F_RES = 1, F_PLAIN = 2 };

// Row-block geometry: strips of W columns (all of x when nx <= 256, else 256),
// NS of them; G groups of R rows side by side in the workgroup when a row is
// shorter than the workgroup; RW = G R rows, at most 16.
struct RowGeom {
    int W, G, NS, RW;
    uint32_t mW, mSP;      // reciprocals of W and W + 4 (div_by)
    int fft_off, tw_off;   // LDS byte offsets of the transform buffer and the twiddle copy
};

template <typename T>
struct RowFwd {
    const T *u, *fh;               // JAC: u; RES: f, fh; PLAIN: x
    JacRows jr;
    int kind;                      // VV_BRACKET_*
    // collision term of J u (null n: none): y += drag_fac drag + diff_fac diff
    const double *cn, *cU, *ca, *cv;
    double drag_fac, diff_fac;
    int coll_e;
};

struct PitchRd {                   // cell (r, cx + d) of a tile of runtime pitch
    template <typename T>
    struct Of {
        const T *p;
        int P;
        __device__ __forceinline__ T operator()(int r, int cx, int d) const { return p[r * P + cx + d]; }
    };
};

// the collision term at the window's centre, as collision_kernel adds it
__device__ __forceinline__ double add_collision(double y, double fm, double f0, double fp, double vp, double vm,
                                                double n, double U, double a, double drag_fac, double diff_fac,
                                                bool e)
{
#pragma clang fp contract(off)
    const double u = U / n;
    double drag, diff;
    if (!e) {
        drag = ((vp - u) * fp - (vm - u) * fm) * a;
        diff = (fp - 2. * f0) + fm;
    } else {
        drag = (vp - u) * fp - (vm - u) * fm;
        diff = ((fp - 2. * f0) + fm) / a;
    }
    return y + (drag_fac * drag + diff_fac * diff);
}

// The base and factor of the two operators: J u = u/dt + .5 {u, H},
// F = (f - fh)/dt + {.5 fh + .5 f, H} (PETScNLVlasovMP.pyx:33-58), unfused.
template <typename T>
__device__ __forceinline__ T fave(T f, T fh)
{
#pragma clang fp contract(off)
    return T(0.5) * fh + T(0.5) * f;
}
template <typename T>
__device__ __forceinline__ T residual_base(T ht_inv, T f, T fh)
{
#pragma clang fp contract(off)
    const T d = f - fh;
    return T(0) + ht_inv * d;
}
// One workgroup: RW rows.  Per strip the tile of the bracket's first argument
// with a 2-cell halo and the x-part of H_ave are staged in LDS (every load of a
// thread issued before the first store), thread t walks column t % W of row group
// t / W down its R rows (SepWin), and the results, times the Krylov vector's
// scale (known one barrier later than the tile), go to the packed lines.  hs: as
// in the strip kernel.  Measured at 64 x 128: J u 5.1 + rFFT 4.1 + update 2.9 us
// and their gaps as launches of their own, 8.0 us here with the unfactored
// stencil, 7.3 now; 201 x 401: 5.6 + 9.3 + 3.3, 11.4, 10.4; 16 x (128 x 256): 11.4,
// 10.0.
// NEAR: the kind has nearest neighbours (not J2; as a branch a point 10.4 -> 10.8 us
// at 201 x 401).
template <int MODE, int R, int FK, bool NEAR, typename T>
__global__ __launch_bounds__(NT) void row_fwd_kernel(FftArgs<T> a, RowGeom g, RowFwd<T> p, HessArgs hs, DftPlan plan,
                                                     cx_t<T> *__restrict__ spec)
{
    using C = cx_t<T>;
    const int extra = hs.nb > 0 ? 1 : 0;
    if (extra && blockIdx.x == 0) {
        hess_update(hs);
        return;
    }
    const int32_t dflag = extra ? hess_skip(hs) : cycle_done(a.done, a.gstride);
    if (gridDim.y > 1 && dflag) return;   // batched: a finished instance skips its loads
    const int b = blockIdx.y, t = threadIdx.x;
    const int nx = a.nx, nv = a.nv, RW = g.RW, RH = RW + 4, W = g.W, SP = W + 4;
    const T *__restrict__ u = p.u + b * a.N;
    const T *__restrict__ fh = MODE == F_RES ? p.fh + b * a.N : nullptr;
    spec += b * a.S;
    const size_t xo = (size_t)b * nx;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    __shared__ double red[kGdNW + 1];
    __shared__ __align__(16) T sA[16][4];      // the rows' coefficients of the bracket
    C *buf = reinterpret_cast<C *>(lds_raw + g.fft_off);
    C *stw = reinterpret_cast<C *>(lds_raw + g.tw_off);
    const int j0 = xcd_tile((int)blockIdx.x - extra, (int)gridDim.x - extra) * RW;
    const double nshare = extra ? norm_share(hs.part + b * hs.pstride, hs.nb) : 0.0;
    tw_table<true>(a.tw, stw, nx);        // read after the barriers below
    if (MODE == F_PLAIN) {
        if (dflag) return;                // uniform over the block, before any barrier
        const uint32_t mnx = 0xffffffffu / (uint32_t)nx + 1;
        for (int idx = t; idx < RW * nx; idx += NT) {
            const int r = div_by(idx, mnx), i = idx - r * nx;
            T v = j0 + r < nv ? u[(size_t)(j0 + r) * nx + i] : T(0);
            if (a.add != nullptr && j0 + r < nv) v += a.gamma * a.add[xo + i];
            T *z = reinterpret_cast<T *>(buf + (r >> 1) * nx + i);
            z[r & 1] = v;
        }
    } else {
        T *sF = reinterpret_cast<T *>(lds_raw);
        double *sP = reinterpret_cast<double *>(lds_raw + (((size_t)RH * SP * sizeof(T) + 15) & ~(size_t)15));
        double usd = MODE == F_JAC && p.jr.uscale != nullptr && !extra
                         ? *reinterpret_cast<const double *>(reinterpret_cast<const char *>(p.jr.uscale) +
                                                             b * a.gstride)
                         : 1.0;
        const T ht_inv = (T)p.jr.ht_inv;
        double c1, c2;
        sep_weights(p.kind, p.jr.factor, p.jr.inst[b].af1, p.jr.inst[b].af2, c1, c2);
        const bool far = sep_far(p.kind);
        const int grp = g.G > 1 ? div_by(t, g.mW) : 0, col = t - grp * W;
        T us = T(1);
        for (int s = 0; s < g.NS; ++s) {
            const int cb = s * W;
            // the strip's cells: RH x SP <= 8 x 260 or 20 x 68 (R = 4), 6 x 260 (R = 2)
            constexpr int NQ = R == 4 ? 9 : 7;
            T fa[NQ], fb[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int idx = t + q * NT;
                const int r = div_by(idx, g.mSP), c = idx - r * SP;
                const int gj = idx < RH * SP ? jr_row(j0, r, nv) : -1;
                const int gi = jr_col(cb, c, nx);
                const size_t o = gj >= 0 ? (size_t)gj * nx + gi : 0;
                const T v = u[o];
                fa[q] = gj >= 0 ? v : T(0);
                fb[q] = T(0);
                if (MODE == F_RES) {
                    const T h = fh[o];
                    fb[q] = gj >= 0 ? h : T(0);
                }
            }
            double xf[2][4];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int c = t + q * NT;
                const size_t gi = xo + (c < SP ? jr_col(cb, c, nx) : 0);
                xf[q][0] = p.jr.h1p[gi];
                xf[q][1] = p.jr.h1h[gi];
                xf[q][2] = p.jr.h2p[gi];
                xf[q][3] = p.jr.h2h[gi];
            }
            if (s == 0 && t < RW) sep_row(p.jr.h0, j0 + t, nv, c1, c2, sA[t]);
            if (s == 0) {
                if (dflag) return;         // uniform over the block, before any barrier
                if (extra) {               // summed after the tile's barrier
                    const double ws = wave_sum(nshare);
                    if ((t & 63) == 0) red[t >> 6] = ws;
                }
            } else {
                __syncthreads();           // the last strip's walk is done
            }
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int c = t + q * NT;
                if (c < SP) sP[c] = phi_ave(xf[q][0], xf[q][1], xf[q][2], xf[q][3]);
            }
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int idx = t + q * NT;
                if (idx < RH * SP) sF[idx] = MODE == F_RES ? fave(fa[q], fb[q]) : fa[q];
            }
            __syncthreads();
            if (s == 0) {
                if (extra) {
                    double tot = 0.0;
                    for (int w = 0; w < kGdNW; ++w) tot += red[w];
                    usd = scale_of(tot);
                }
                us = (T)usd;
            }
            const int i = cb + col;
            if (grp < g.G && col < W && i < nx) {
                const int cx = col + 2, r0 = grp * R;
                const PitchRd::Of<T> rF{sF, SP};
                T B[4];
                sep_coef(sP[cx - 2], sP[cx - 1], sP[cx], sP[cx + 1], sP[cx + 2], c1, c2, B);
                SepWin<T> win;
                win.load(rF, r0 + 2, cx);
                double cn = 1.0, cU = 0.0, ca = 1.0;
                const bool coll = MODE == F_JAC && sizeof(T) == 8 && p.cn != nullptr;
                if (coll) {
                    cn = p.cn[i];
                    cU = p.cU[i];
                    ca = p.ca[i];
                }
                T *z = reinterpret_cast<T *>(buf + (r0 >> 1) * nx + i);
#pragma unroll
                for (int q = 0; q < R; ++q) {
                    const int j = j0 + r0 + q;
                    T out = T(0);
                    if (j < nv) {
                        T base;
                        if (MODE == F_RES) base = residual_base(ht_inv, u[(size_t)j * nx + i], fh[(size_t)j * nx + i]);
                        else base = jacobian_base(ht_inv, win.f0[2]);
                        out = base;
                        if (j >= 2 && j < nv - 2) {
                            out = base + win.bracket(sA[r0 + q], B, NEAR, far);
                            if (coll)
                                out = (T)add_collision((double)out, (double)win.f0[1], (double)win.f0[2],
                                                       (double)win.f0[3], p.cv[j + 1], p.cv[j - 1], cn, cU, ca,
                                                       p.drag_fac, p.diff_fac, p.coll_e != 0);
                        }
                    }
                    z[(q >> 1) * 2 * nx + (q & 1)] = MODE == F_JAC ? scaled(out, us) : out;
                    if (q + 1 < R) win.advance(rF, r0 + q + 3, cx);
                }
            }
        }
    }
    __syncthreads();
    const C *out = buf;
    if constexpr (FK == kDft) {
        C *other = buf + (RW >> 1) * nx;
        out = (plan.stages & 1) ? other : buf;
        dft_lines<false>(buf, other, RW >> 1, plan, (const C *)stw, LineSink<C>{const_cast<C *>(out), nx});
    } else {
        lds_fft<false, false, 1>(buf, a.logn, RW >> 1, (const C *)stw, FftTw<false, C>{}, 0, LdsSink<C>{buf});
    }
    store_rows_spectrum(out, nx, RW, j0, nv, a.pitch, spec);
}

// ---- inverse ----------------------------------------------------------------

// natural-order real rows of the workgroup: row r at wr[r nx + i], scaled by 1/n
template <typename T>
struct RowsOut {
    T *wr;
    int nx;
    T inv_n;
    __device__ __forceinline__ void operator()(int b, int i, cx_t<T> z) const
    {
        wr[(2 * b) * nx + i] = z.x * inv_n;
        wr[(2 * b + 1) * nx + i] = z.y * inv_n;
    }
};
template <typename T>
struct RowsOutPos {
    RowsOut<T> o;
    int logn;
    __device__ __forceinline__ void operator()(int pos, cx_t<T> z) const
    {
        o(pos >> logn, pos & (o.nx - 1), z);
    }
};

template <typename T> struct V2;
template <> struct V2<double> { using type = double2; };
template <> struct V2<float> { using type = float2; };

// The pair v of a block's cnt elements; the pair past the end reads the last
// one (inside the allocation) and elements past cnt count as 0.
template <typename T>
__device__ __forceinline__ typename V2<T>::type load_pair(const T *p, int v, int cnt)
{
    const int last = (cnt - 1) >> 1;
    typename V2<T>::type x = reinterpret_cast<const typename V2<T>::type *>(p)[v < last ? v : last];
    x.x = 2 * v < cnt ? x.x : T(0);
    x.y = 2 * v + 1 < cnt ? x.y : T(0);
    return x;
}

// irFFT of the workgroup's RI rows into w = V_{col+1}, and the dots of w with
// v_0 .. v_col from LDS, partials per block as irfft_mdot_kernel's; col = -1:
// into y, with the block's sum of squares at part[block] when part is given.  RI is even, so a block starts on an even element and is
// read in pairs (thread t the pairs t + 256 q, q < EPT); the last block may be
// short, and odd.  Replaces irFFT + mdot: 4.9 + 3.3 us at 64 x 128 and 9.3 +
// 4.6 us at 201 x 401 with a launch between.
template <typename T, int EPT, int FK>
__global__ __launch_bounds__(NT) void row_inv_kernel(FftArgs<T> a, const cx_t<T> *__restrict__ spec, DftPlan plan,
                                                     CgsArgs<T> g, int col, int pitch, T *y)
{
    using C = cx_t<T>;
    using V = typename V2<T>::type;
    const int32_t dflag = cycle_done(a.done, a.gstride);
    if (gridDim.y > 1 && dflag) return;   // batched: a finished instance skips its loads
    const int bi = blockIdx.y;
    spec += bi * a.S;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C *buf = reinterpret_cast<C *>(lds_raw);
    __shared__ double red[kCgsNW][kMaxRestart];
    __shared__ double s_scale[kMaxRestart];
    const int nx = a.nx, RI = a.rows, nk = nx / 2 + 1, npair = RI >> 1, nvec = col + 1, t = threadIdx.x;
    const int blk = xcd_tile(blockIdx.x, gridDim.x);
    const int j0 = blk * RI;
    const int rows = a.nv - j0 < RI ? a.nv - j0 : RI;
    const int cnt = rows * nx;
    const T *basis = nvec > 0 ? g.basis + bi * g.N + (size_t)j0 * nx : nullptr;
    T *W = nvec > 0 ? const_cast<T *>(basis) + (size_t)nvec * g.vstride : y + bi * a.N + (size_t)j0 * nx;
    const int total = nk * npair;
    // mode pairs (nx/2 + 1) RI/2 <= PTS/4 + PTS/16 (nx >= 8)
    constexpr int PTS = 2 * NT * EPT, PER = (5 * PTS / 16 + NT - 1) / NT;
    const uint32_t mp = 0xffffffffu / (uint32_t)npair + 1;      // npair = 1: wraps to 0, handled below
    C va[PER], vb[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int idx = t + q * NT;
        const int k = npair > 1 ? div_by(idx, mp) : idx;
        const int ja = j0 + 2 * (idx - k * npair);
        va[q] = load_or_zero(spec, (int64_t)k * a.pitch + ja, idx < total && ja < a.nv);
        vb[q] = load_or_zero(spec, (int64_t)k * a.pitch + ja + 1, idx < total && ja + 1 < a.nv);
    }
    const double sc = t < nvec ? (g.g + bi)->scale[t] : 0.0;
    C *stw = buf + (FK == kDft ? 2 : 1) * (size_t)npair * nx;
    tw_table<true>(a.tw, stw, nx);
    if (dflag) return;                    // uniform over the block, before any barrier
    // the first group of basis vectors is in flight while the transform runs
    constexpr int G = cgs_group<EPT>();
    V x[G][EPT];
    auto load_vectors = [&](int v) {
#pragma unroll
        for (int gg = 0; gg < G; ++gg) {
            if (v + gg >= nvec) break;    // uniform
#pragma unroll
            for (int q = 0; q < EPT; ++q)
                x[gg][q] = load_pair<T>(basis + (size_t)(v + gg) * g.vstride, t + q * NT, cnt);
        }
    };
    load_vectors(0);
    if (t < kMaxRestart) s_scale[t] = sc;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int idx = t + q * NT;
        if (idx < total) {
            const int k = npair > 1 ? div_by(idx, mp) : idx;
            const int p = idx - k * npair;
            const bool self = k == 0 || 2 * k == nx;
            C A = va[q], B = vb[q];
            if (self) {
                A.y = T(0);
                B.y = T(0);
            }
            C *z = buf + p * nx;
            z[k] = cmk<C>(A.x - B.y, A.y + B.x);
            if (!self) z[nx - k] = cmk<C>(A.x + B.y, B.x - A.y);
        }
    }
    __syncthreads();
    T *wr;
    if constexpr (FK == kDft) {
        C *other = buf + (size_t)npair * nx;
        wr = reinterpret_cast<T *>((plan.stages & 1) ? other : buf);
        dft_lines<true>(buf, other, npair, plan, (const C *)stw, RowsOut<T>{wr, nx, T(1) / (T)nx});
    } else {
        wr = reinterpret_cast<T *>(buf);
        lds_fft<true, false, (PTS / 2 + 1023) / 1024>(buf, a.logn, npair, (const C *)stw, FftTw<true, C>{}, 0,
                                                   RowsOutPos<T>{RowsOut<T>{wr, nx, T(1) / (T)nx}, a.logn});
    }
    // w of the block: to memory, and into registers for the dots
    V w[EPT];
#pragma unroll
    for (int q = 0; q < EPT; ++q) {
        const int v = t + q * NT;
        w[q] = load_pair<T>(wr, v, cnt);
        if (2 * v + 1 < cnt) reinterpret_cast<V *>(W)[v] = w[q];
        else if (2 * v < cnt) W[2 * v] = w[q].x;
    }
    const int lane = t & 63, wave = t >> 6;
    if (nvec == 0) {
        if (g.part == nullptr) return;
        double acc = 0.0;
#pragma unroll
        for (int q = 0; q < EPT; ++q) {
            acc = __builtin_fma((double)w[q].x, (double)w[q].x, acc);
            acc = __builtin_fma((double)w[q].y, (double)w[q].y, acc);
        }
        acc = wave_sum(acc);
        if (lane == 0) red[wave][0] = acc;
        __syncthreads();
        if (t == 0) {
            double s = 0.0;
            for (int wv = 0; wv < kCgsNW; ++wv) s += red[wv][0];
            (g.part + bi * g.pstride)[blk] = s;
        }
        return;
    }
    for (int v = 0; v < nvec; v += G) {
        if (v > 0) load_vectors(v);
#pragma unroll
        for (int gg = 0; gg < G; ++gg) {
            if (v + gg >= nvec) break;
            const double sv = s_scale[v + gg];
            double acc = 0.0;
#pragma unroll
            for (int q = 0; q < EPT; ++q) {
                acc = __builtin_fma((double)w[q].x, (double)x[gg][q].x * sv, acc);
                acc = __builtin_fma((double)w[q].y, (double)x[gg][q].y * sv, acc);
            }
            acc = wave_sum(acc);
            if (lane == 0) red[wave][v + gg] = acc;
        }
    }
    __syncthreads();
    if (t < nvec) {
        double s = 0.0;
        for (int wv = 0; wv < kCgsNW; ++wv) s += red[wv][t];
        (g.part + bi * g.pstride)[(size_t)blk * pitch + t] = s;
    }
}

// ---- host -------------------------------------------------------------------

bool pow2(int n) { return (n & (n - 1)) == 0; }

int fft_kind(int nx) { return pow2(nx) ? kFftPre : kDft; }

template <typename T> const cx_t<T> *twiddles(const vv_ctx *c);
template <> const double2 *twiddles<double>(const vv_ctx *c) { return c->twiddle; }
template <> const float2 *twiddles<float>(const vv_ctx *c) { return c->twiddle32; }

// geometry for R rows per thread
template <typename T>
RowGeom geom_for(const vv_ctx *c, int mode, int R, size_t *lds)
{
    const int nx = c->fft_n;
    RowGeom g{};
    g.W = nx < NT ? nx : NT;
    g.NS = (nx + NT - 1) / NT;
    const int most = 16 / R, fit = NT / nx;
    g.G = fit < 1 ? 1 : fit < most ? fit : most;
    g.RW = g.G * R;
    g.mW = 0xffffffffu / (uint32_t)g.W + 1;
    g.mSP = 0xffffffffu / (uint32_t)(g.W + 4) + 1;
    const int RH = g.RW + 4, SP = g.W + 4;
    size_t strip = (((size_t)RH * SP * sizeof(T) + 15) & ~(size_t)15) + (size_t)SP * sizeof(double);
    strip = (strip + 15) & ~(size_t)15;
    const bool dft = fft_kind(nx) == kDft;
    const size_t lines = (size_t)(g.RW >> 1) * nx * sizeof(cx_t<T>) * (dft ? 2 : 1);
    g.fft_off = mode == F_PLAIN ? 0 : (int)strip;
    const size_t end = g.fft_off + lines;
    g.tw_off = (int)end;
    *lds = end + (size_t)nx * sizeof(cx_t<T>);
    return g;
}

// rows per thread of the forward kernel: 4 (fewer halo rows) where that still
// leaves two workgroups a CU, in number and in LDS, else 2 (at most 113 KB, at
// nx = 2047)
template <typename T>
RowGeom row_geom(const vv_ctx *c, int mode, int *R, size_t *lds)
{
    *R = 4;
    const RowGeom g = geom_for<T>(c, mode, 4, lds);
    if ((int64_t)((c->fft_rows + g.RW - 1) / g.RW) * c->B >= 512 && *lds <= 65536) return g;
    *R = 2;
    return geom_for<T>(c, mode, 2, lds);
}

template <int MODE, int R, typename T>
void fwd_launch(vv_ctx *c, const FftArgs<T> &a, const RowGeom &g, const RowFwd<T> &p, const HessArgs &hs, dim3 grid,
                size_t lds, cx_t<T> *spec)
{
    const dim3 block(NT);
#define VV_FWD(FK_, NEAR_) \
    launch_timed(c, row_fwd_kernel<MODE, R, FK_, NEAR_, T>, grid, block, (uint32_t)lds, a, g, p, hs, c->dft, spec)
    if constexpr (MODE == F_PLAIN) {      // powers of two have kernels of their own
        VV_FWD(kDft, true);
    } else {
        const bool near = sep_near(p.kind);
        if (fft_kind(a.nx) == kFftPre) {
            if (near) VV_FWD(kFftPre, true);
            else VV_FWD(kFftPre, false);
        } else {
            if (near) VV_FWD(kDft, true);
            else VV_FWD(kDft, false);
        }
    }
#undef VV_FWD
}

template <int MODE, typename T>
hipError_t row_fwd_t(vv_ctx *c, RowFwd<T> p, cx_t<T> *spec, const int32_t *done, const T *add = nullptr,
                     T gamma = T(0))
{
    int R;
    size_t lds;
    const RowGeom g = row_geom<T>(c, MODE, &R, &lds);
    FftArgs<T> a{c->fft_n, c->logn, c->fft_rows, g.RW, c->N, spec_stride(c), spec_pitch(c), (int64_t)sizeof(GmresState),
                 twiddles<T>(c), done, add, gamma};
    HessArgs hs{};
    if (MODE == F_JAC && p.jr.uscale != nullptr) hs = take_update(c);    // a Krylov vector: its scale is due
    const dim3 grid((a.nv + g.RW - 1) / g.RW + (hs.nb > 0 ? 1 : 0), c->B);
    if (R == 4) fwd_launch<MODE, 4, T>(c, a, g, p, hs, grid, lds, spec);
    else fwd_launch<MODE, 2, T>(c, a, g, p, hs, grid, lds, spec);
    return hipGetLastError();
}

// rows of an inverse workgroup: the FFT kernels' rows, brought to at least 384
// and at most 4096 elements
int inv_rows(const vv_ctx *c)
{
    int R = fft_rows_of(c);
    R += R & 1;
    while (R * c->fft_n < 384 && R < c->fft_rows) R *= 2;
    while (R * c->fft_n > 4096 && R > 2) R = (R / 2 + 1) & ~1;
    return R;
}

template <typename T, int EPT>
void inv_launch(vv_ctx *c, const FftArgs<T> &a, const cx_t<T> *spec, const CgsArgs<T> &g, int col, int pitch, T *y,
                dim3 grid, size_t lds)
{
    const dim3 block(NT);
    switch (fft_kind(a.nx)) {
    case kFftPre: launch_timed(c, row_inv_kernel<T, EPT, kFftPre>, grid, block, (uint32_t)lds, a, spec, c->dft, g, col, pitch, y); break;
    default: launch_timed(c, row_inv_kernel<T, EPT, kDft>, grid, block, (uint32_t)lds, a, spec, c->dft, g, col, pitch, y); break;
    }
}

template <typename T>
hipError_t row_inv_t(vv_ctx *c, const T *basis, const cx_t<T> *spec, int col, T *y, double *part, const int32_t *done)
{
    const int RI = inv_rows(c);
    FftArgs<T> a{c->fft_n, c->logn, c->fft_rows, RI, c->N, spec_stride(c), spec_pitch(c), (int64_t)sizeof(GmresState),
                 twiddles<T>(c), done};
    const int nb = (a.nv + RI - 1) / RI;
    const bool dft = fft_kind(a.nx) == kDft;
    const size_t lds = (size_t)(RI >> 1) * a.nx * sizeof(cx_t<T>) * (dft ? 2 : 1) + (size_t)a.nx * sizeof(cx_t<T>);
    const CgsArgs<T> g{basis, c->N, c->vs, part, c->part_stride, c->gs, 0, nb};
    const int pitch = c->p.restart < 32 ? 32 : 64;
    const dim3 grid(nb, c->B);
    const int pts = RI * a.nx;
    if (pts <= 512) inv_launch<T, 1>(c, a, spec, g, col, pitch, y, grid, lds);
    else if (pts <= 1024) inv_launch<T, 2>(c, a, spec, g, col, pitch, y, grid, lds);
    else if (pts <= 2048) inv_launch<T, 4>(c, a, spec, g, col, pitch, y, grid, lds);
    else inv_launch<T, 8>(c, a, spec, g, col, pitch, y, grid, lds);
    return hipGetLastError();
}

}  // namespace

// Powers of two from 1024 on stay with the separate launches here: their runtime
// strips, 25 KB beside 32 KB and more of lines, leave one or two workgroups a
// CU (F(f) + rFFT at 1024 x 2048: 44.8 us against 18.6 + 13.0; J u + rFFT at
// 2048 x 1024: 41 against 12.8 + 13.2).
// Lengths of a single stage (primes, 9, 10, 12, 14, 15) are transformed by the
// direct real DFT (dft_rows), half the arithmetic; fusing J u and the dots with the
// line sum still saves more launches than that costs on grids of one strip and
// up to 2^25 products.  A solve of 8 iterations, fused and separate: 211 x 512
// 345 and 391 us, 101 x 2048 306 and 345, but 101 x 4096 460 and 447, 151 x 2048
// 537 and 512, 257 x 128 577 and 502, 1999 x 2048 39.2 ms and 25.6.
bool rows_apply(const vv_ctx *c)
{
    if (!c->fuse || c->p.precond != VV_PRECOND_TENSOR_KINETIC) return false;
    const int nx = c->p.nx;
    if (pow2(nx)) return nx <= 512;
    return dft_rows(c) || (c->dft.n > 0 && nx <= NT && (int64_t)nx * nx * c->fft_rows * c->B <= 1 << 25);
}

int row_inv_blocks(const vv_ctx *c)
{
    const int RI = inv_rows(c);
    return (c->fft_rows + RI - 1) / RI;
}

hipError_t launch_row_jac(vv_ctx *c, const double *u, const double *uscale, const CollTerm *coll, double2 *spec,
                          const int32_t *done)
{
    RowFwd<double> p{};
    p.u = u;
    p.jr = JacRows{uscale, c->h0, c->h1p, c->h1h, c->h2p, c->h2h, c->inst, c->ht_inv, 0.5};
    p.kind = c->p.bracket;
    if (coll != nullptr) {
        p.cn = coll->n;
        p.cU = coll->U;
        p.ca = coll->a;
        p.cv = c->vgrid;
        p.drag_fac = coll->drag_fac;
        p.diff_fac = coll->diff_fac;
        p.coll_e = coll->e;
    }
    return row_fwd_t<F_JAC, double>(c, p, spec, done);
}

hipError_t launch_row_jac32(vv_ctx *c, const float *u, const double *uscale, float2 *spec, const int32_t *done)
{
    RowFwd<float> p{};
    p.u = u;
    p.jr = JacRows{uscale, c->h0, c->h1p, c->h1h, c->h2p, c->h2h, c->inst, c->ht_inv, 0.5};
    p.kind = c->p.bracket;
    return row_fwd_t<F_JAC, float>(c, p, spec, done);
}

hipError_t launch_row_res(vv_ctx *c, const double *f, const double *fh, double2 *spec)
{
    RowFwd<double> p{};
    p.u = f;
    p.fh = fh;
    p.jr = JacRows{nullptr, c->h0, c->h1p, c->h1h, c->h2p, c->h2h, c->inst, c->ht_inv, 1.0};
    p.kind = c->p.bracket;
    return row_fwd_t<F_RES, double>(c, p, spec, nullptr);
}

// rows as they are (dft_rows); y of the inverse 16-byte aligned
hipError_t launch_row_rfft(vv_ctx *c, const double *x, double2 *spec, const int32_t *done, const double *add,
                           double gamma)
{
    RowFwd<double> p{};
    p.u = x;
    return row_fwd_t<F_PLAIN, double>(c, p, spec, done, add, gamma);
}

hipError_t launch_row_rfft32(vv_ctx *c, const float *x, float2 *spec, const int32_t *done)
{
    RowFwd<float> p{};
    p.u = x;
    return row_fwd_t<F_PLAIN, float>(c, p, spec, done);
}

hipError_t launch_row_irfft(vv_ctx *c, const double2 *spec, double *y, const int32_t *done)
{
    return row_inv_t<double>(c, nullptr, spec, -1, y, nullptr, done);
}

hipError_t launch_row_irfft32(vv_ctx *c, const float2 *spec, float *y, const int32_t *done)
{
    return row_inv_t<float>(c, nullptr, spec, -1, y, nullptr, done);
}

hipError_t launch_row_inv_start(vv_ctx *c, const double2 *spec)
{
    return row_inv_t<double>(c, nullptr, spec, -1, c->basis, norm_partials(c), nullptr);
}

hipError_t launch_row_inv(vv_ctx *c, const double2 *spec, int col, const int32_t *done)
{
    return row_inv_t<double>(c, c->basis, spec, col, nullptr, c->partial, done);
}

hipError_t launch_row_inv32(vv_ctx *c, const float2 *spec, int col, const int32_t *done)
{
    return row_inv_t<float>(c, c->basis32, spec, col, nullptr, c->partial, done);
}

// Radices of a length that is no power of two: the divisors' product that
// costs least, a radix r counted r products a point plus 8 for its pass over
// LDS; a prime above 64 stands alone.
DftPlan make_dft_plan(int n)
{
    DftPlan p{};
    p.n = n;
    std::vector<int> best, cur;
    int bestc = 1 << 30;
    auto rec = [&](auto &&self, int m, int from, int cost) -> void {
        if (cost >= bestc) return;
        if (m == 1) {
            bestc = cost;
            best = cur;
            return;
        }
        if ((int)cur.size() == kDftStages) return;
        bool prime = true;
        for (int d = 2; d * d <= m; ++d)
            if (m % d == 0) prime = false;
        for (int d = from; d <= m; ++d) {
            if (m % d || (d > 64 && !(d == m && prime))) continue;
            cur.push_back(d);
            self(self, m / d, d, cost + d + 8);
            cur.pop_back();
        }
    };
    rec(rec, n, 2, 0);
    p.stages = (int)best.size();
    int ns = 1;
    for (int s = 0; s < p.stages; ++s) {
        const int r = best[s];
        p.r[s] = r;
        p.ns[s] = ns;
        p.nr[s] = n / r;
        p.step[s] = n / (ns * r);
        p.mnr[s] = n / r > 1 ? 0xffffffffu / (uint32_t)(n / r) + 1 : 0;
        p.mns[s] = ns > 1 ? 0xffffffffu / (uint32_t)ns + 1 : 0;
        ns *= r;
    }
    p.mn = 0xffffffffu / (uint32_t)n + 1;
    return p;
}

}  // namespace vv
