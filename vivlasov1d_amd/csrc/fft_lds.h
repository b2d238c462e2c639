// In-LDS transforms of real v-rows (Stockham FFT of power-of-two lengths), the
// spectrum's mode-major store and small helpers, shared by the spectral units.
#pragma once

#include "arakawa.h"
#include "cgs_vec.h"

namespace vv {
namespace {

constexpr int NT = 256;
constexpr int MAXE = 4096;   // complex elements of one FFT workgroup (64 KiB of LDS)
// threads of the long lines' kernels (64 KB of LDS, two workgroups a CU): with 256
// rfft and irfft take 46.5 us at 2048 x 4096, with 512 and the swizzle below 44.6
constexpr int NTL = 512;

// complex arithmetic on double2 / float2
template <typename C> __device__ __forceinline__ C cmk(typename C::value_type re, typename C::value_type im)
{
    C r;
    r.x = re;
    r.y = im;
    return r;
}
template <typename C> __device__ __forceinline__ C cadd(C a, C b) { return cmk<C>(a.x + b.x, a.y + b.y); }
template <typename C> __device__ __forceinline__ C csub(C a, C b) { return cmk<C>(a.x - b.x, a.y - b.y); }
template <typename C> __device__ __forceinline__ C cmul(C a, C b)
{
    return cmk<C>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
template <typename C> __device__ __forceinline__ C cneg(C a) { return cmk<C>(-a.x, -a.y); }
template <typename C> __device__ __forceinline__ C cconj(C a) { return cmk<C>(a.x, -a.y); }
// 1/d for the complex divisions of the tridiagonal solve: the hardware
// reciprocal estimate refined by two Newton steps r <- r (2 - d r) instead of
// the IEEE division sequence.  The dependent chain of the Thomas sweep is
// shorter (21.5 -> 20.9 us per solve at 1024 x 2048); P^-1 moves by about
// one ulp (2.8e-16 relative).  The pivots are O(1/dt), far from the
// denormal and overflow ranges.
__device__ __forceinline__ double rcp_of(double d)
{
    double r = __builtin_amdgcn_rcp(d);
    r = r * (2.0 - d * r);
    r = r * (2.0 - d * r);
    return r;
}
__device__ __forceinline__ float rcp_of(float d) { return 1.0f / d; }

template <typename C> __device__ __forceinline__ C cdiv(C z, C w)
{
    const auto inv = rcp_of(w.x * w.x + w.y * w.y);
    return cmk<C>((z.x * w.x + z.y * w.y) * inv, (z.y * w.x - z.x * w.y) * inv);
}
template <typename C> __device__ __forceinline__ C crecip(C w)
{
    const auto inv = rcp_of(w.x * w.x + w.y * w.y);
    return cmk<C>(w.x * inv, -w.y * inv);
}

// p[i] when ok, else zero.  The address is clamped to p[0] instead of
// selecting between p + i and a local zero, so the load stays an
// unconditional global load that can be in flight with the others.
template <typename C> __device__ __forceinline__ C load_or_zero(const C *__restrict__ p, int64_t i, bool ok)
{
    const C v = p[ok ? i : 0];
    return ok ? v : cmk<C>(typename C::value_type(0), typename C::value_type(0));
}

// complex type of a real type
template <typename T> struct CxOf;
template <> struct CxOf<double> { using type = double2; };
template <> struct CxOf<float> { using type = float2; };
template <typename T> using cx_t = typename CxOf<T>::type;

template <bool INV, typename C>
__device__ __forceinline__ C twiddle(const C *__restrict__ tw, int m)
{
    const C t = tw[m];
    return INV ? cmk<C>(t.x, -t.y) : t;
}

// Twiddles of the n = 1024 plan 4 x 8 x 8 x 4 (see lds_fft1024), loaded once by
// each thread before the transform: every butterfly it owns, in any transform
// of the block and any stage, has the index j = threadIdx.x mod n/4 (n/8), so
// 17 of them cover it; their loads are in flight with the tile's own instead of
// being waited on after every barrier.  w: 0..6 and 7..13 for the radix-8 stages
// with sub-transforms of 4 and 32, 14..16 for the last radix-4 stage.
constexpr int N8 = 1024;
template <bool INV, typename C>
struct FftTw {
    C w[17];
    __device__ __forceinline__ void load(const C *__restrict__ tw)
    {
        const int t = threadIdx.x, ka = t & 3, kb = t & 31, kc = t & 255;
#pragma unroll
        for (int r = 1; r < 8; ++r) {
            w[r - 1] = twiddle<INV>(tw, r * ka * 32);
            w[6 + r] = twiddle<INV>(tw, r * kb * 4);
        }
#pragma unroll
        for (int r = 1; r < 4; ++r) w[13 + r] = twiddle<INV>(tw, r * kc);
    }
};

// Where the last stage of lds_fft puts its outputs: back into the LDS buffer
// (the default), or wherever a kernel wants them (the irFFT stores them to
// its output rows directly).  pos = transform * n + natural index.
template <typename C>
struct LdsSink {
    C *buf;
    __device__ __forceinline__ void operator()(int pos, C v) const { buf[pos] = v; }
};

// The radix-4 butterfly of the Stockham stages (outputs in natural order of
// the 4-point DFT; forward (v1 - v3)(-i), inverse (v1 - v3)(+i)).
template <bool INV, typename C>
__device__ __forceinline__ void dft4(C &v0, C &v1, C &v2, C &v3)
{
    const C a0 = cadd(v0, v2), a1 = csub(v0, v2), a2 = cadd(v1, v3), d = csub(v1, v3);
    const C a3 = INV ? cmk<C>(-d.y, d.x) : cmk<C>(d.y, -d.x);
    v0 = cadd(a0, a2);
    v1 = cadd(a1, a3);
    v2 = csub(a0, a2);
    v3 = csub(a1, a3);
}

// 8-point DFT in place: the radix-4 DFTs of the even and the odd samples,
// combined with W8^m (forward W8 = (1 - i)/sqrt 2, inverse its conjugate).
template <bool INV, typename C>
__device__ __forceinline__ void dft8(C (&v)[8])
{
    using R = typename C::value_type;
    const R h = R(0.70710678118654752440);
    C e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    C o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    dft4<INV>(e0, e1, e2, e3);
    dft4<INV>(o0, o1, o2, o3);
    o1 = INV ? cmk<C>((o1.x - o1.y) * h, (o1.x + o1.y) * h) : cmk<C>((o1.x + o1.y) * h, (o1.y - o1.x) * h);
    o2 = INV ? cmk<C>(-o2.y, o2.x) : cmk<C>(o2.y, -o2.x);
    o3 = INV ? cmk<C>(-(o3.x + o3.y) * h, (o3.x - o3.y) * h) : cmk<C>((o3.y - o3.x) * h, -(o3.x + o3.y) * h);
    v[0] = cadd(e0, o0);
    v[4] = csub(e0, o0);
    v[1] = cadd(e1, o1);
    v[5] = csub(e1, o1);
    v[2] = cadd(e2, o2);
    v[6] = csub(e2, o2);
    v[3] = cadd(e3, o3);
    v[7] = csub(e3, o3);
}

// One radix-8 Stockham stage of the n = 1024 plan: sub-transforms of length
// NS (4 or 32) combined into 8 NS; butterfly j takes elements j + 128 r,
// twiddled by W_1024^(r k 1024 / (8 NS)), k = j mod NS (= threadIdx.x mod NS
// for every butterfly of the thread, so the thread's twiddles are preloaded:
// flat index OFF + r - 1 of FftTw), and stores output m at 8 (j - k) + k + m NS.
template <bool INV, int NS, int OFF, typename C>
__device__ __forceinline__ void stage8_1024(C *buf, int nb, const FftTw<INV, C> &pt)
{
    constexpr int nq = N8 / 8;
    const int total = nb * nq;
    C v[2][8];
    int dst[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int bq = threadIdx.x + q * NT;
        dst[q] = -1;
        if (bq < total) {
            const int b = bq >> 7, j = bq & (nq - 1), k = j & (NS - 1);
            const C *src = buf + b * N8;
#pragma unroll
            for (int r = 0; r < 8; ++r) v[q][r] = src[j + r * nq];
#pragma unroll
            for (int r = 1; r < 8; ++r) v[q][r] = cmul(v[q][r], pt.w[OFF + r - 1]);
            dft8<INV>(v[q]);
            dst[q] = b * N8 + ((j - k) << 3) + k;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 2; ++q)
        if (dst[q] >= 0) {
#pragma unroll
            for (int m = 0; m < 8; ++m) buf[dst[q] + m * NS] = v[q][m];
        }
    __syncthreads();
}

// n = 1024 as 4 x 8 x 8 x 4: the first radix-4 stage (from LDS when s0 == 0;
// s0 == 1: the caller ran it in registers), two radix-8 stages and a last
// radix-4 stage whose outputs go to `last` -- four passes over LDS instead of
// the five of the radix-4 plan.  nb <= 4 transforms (MAXE elements).
template <bool INV, typename C, typename Sink>
__device__ __forceinline__ void lds_fft1024(C *buf, int nb, const FftTw<INV, C> &pt, int s0, const Sink &last)
{
    constexpr int nq = N8 / 4;
    const int total = nb * nq;
    if (s0 == 0) {
        C v[4][4];
        int dst[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int bq = threadIdx.x + q * NT;
            dst[q] = -1;
            if (bq < total) {
                const int b = bq >> 8, j = bq & (nq - 1);
                const C *src = buf + b * N8;
#pragma unroll
                for (int r = 0; r < 4; ++r) v[q][r] = src[j + r * nq];
                dft4<INV>(v[q][0], v[q][1], v[q][2], v[q][3]);
                dst[q] = b * N8 + (j << 2);
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (dst[q] >= 0) {
#pragma unroll
                for (int r = 0; r < 4; ++r) buf[dst[q] + r] = v[q][r];
            }
        __syncthreads();
    }
    stage8_1024<INV, 4, 0>(buf, nb, pt);
    stage8_1024<INV, 32, 7>(buf, nb, pt);
    // last stage: sub-transforms of 256, k = j = threadIdx.x, outputs j + 256 m
    C v[4][4];
    int dst[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int bq = threadIdx.x + q * NT;
        dst[q] = -1;
        if (bq < total) {
            const int b = bq >> 8, j = bq & (nq - 1);
            const C *src = buf + b * N8;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[q][r] = src[j + r * nq];
            v[q][1] = cmul(v[q][1], pt.w[14]);
            v[q][2] = cmul(v[q][2], pt.w[15]);
            v[q][3] = cmul(v[q][3], pt.w[16]);
            dft4<INV>(v[q][0], v[q][1], v[q][2], v[q][3]);
            dst[q] = b * N8 + j;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (dst[q] >= 0) {
#pragma unroll
            for (int m = 0; m < 4; ++m) last(dst[q] + m * nq, v[q][m]);
        }
    __syncthreads();
}

// Place of element i of a long line (n >= 2048) in LDS.  The 16 lanes that a
// 16-byte access serves together take i = 4j, 8j, 32 (j >> 2) + (j & 3) or
// 64 (j >> 3) + (j & 7) in the stores of the first two stages, 2 to 4 of the 16
// bank groups; bits 4, 5, 6 are folded into the low four so that each of these
// (and 16 elements in a row) meets all 16.
template <bool SWZ>
__device__ __forceinline__ int swz(int i)
{
    if constexpr (!SWZ) return i;
    const int a = (i >> 4) & 7;
    return i ^ a ^ ((a & 6) << 1);
}

// One Stockham stage of radix RAD (4 or 8) on nb transforms of length 2^logn:
// sub-transforms of length Ns = 2^l combined; butterfly j of a transform takes
// elements j + r n/RAD, twiddled by W_n^(r k n/(RAD Ns)), k = j mod Ns, and
// stores output m at RAD (j - k) + k + m Ns.  Every butterfly of the thread (Q
// at most) is loaded before the barrier and stored after it, so one buffer
// suffices; the final stage's outputs go to `last`.
template <int RAD, bool INV, int Q, int NTH, bool SWZ, typename C, typename Sink>
__device__ __forceinline__ void fft_stage(C *buf, int logn, int nb, int l, const C *tw, bool fin, const Sink &last)
{
    constexpr int LR = RAD == 8 ? 3 : 2;
    const int lq = logn - LR, nq = 1 << lq, Ns = 1 << l, sh = lq - l, total = nb << lq;
    C v[Q][RAD];
    int dst[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int bq = threadIdx.x + q * NTH;
        dst[q] = -1;
        if (bq < total) {
            const int b = bq >> lq, j = bq & (nq - 1), k = j & (Ns - 1);
            const C *src = buf + swz<SWZ>((b << logn) + j);     // r << lq leaves the swizzle alone
#pragma unroll
            for (int r = 0; r < RAD; ++r) v[q][r] = src[r << lq];
            if (l > 0) {
#pragma unroll
                for (int r = 1; r < RAD; ++r) v[q][r] = cmul(v[q][r], twiddle<INV>(tw, (r * k) << sh));
            }
            if constexpr (RAD == 8) dft8<INV>(v[q]);
            else dft4<INV>(v[q][0], v[q][1], v[q][2], v[q][3]);
            dst[q] = (b << logn) + ((j - k) << LR) + k;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        if (dst[q] >= 0) {
#pragma unroll
            for (int m = 0; m < RAD; ++m) {
                if (fin) last(dst[q] + (m << l), v[q][m]);
                else buf[swz<SWZ>(dst[q] + (m << l))] = v[q][m];
            }
        }
    }
    __syncthreads();
}

// radix-4 stages a transform of length 2^logn begins with (the rest are of
// radix 8): 64 = 8 x 8, 128 = 4 x 4 x 8, 256 = 4 x 8 x 8, 512 = 8 x 8 x 8,
// 2048 = 4 x 8 x 8 x 8, 4096 = 8 x 8 x 8 x 8
__host__ __device__ __forceinline__ int fft_lead4(int logn)
{
    const int b = logn % 3;
    return b == 0 ? 0 : b == 1 ? 2 : 1;
}
// log2 of the first stage's radix (which kernels may run in registers)
__host__ __device__ __forceinline__ int fft_first(int logn) { return fft_lead4(logn) ? 2 : 3; }

// Batched in-LDS Stockham FFT of `nb` transforms of length n = 2^logn stored
// back to back in buf, at most EB * 1024 elements.  Forward uses
// exp(-2 pi i m/n), inverse the conjugate (unnormalised).  C is double2 (FP64
// path) or float2 (FP32 preconditioner of the mixed solver).  tw: the table of
// exp(-2 pi i m/n), a copy in LDS for the short lengths.  P8: n = 1024 by the
// 4 x 8 x 8 x 4 plan (pt loaded).  l0: log2 of the sub-transforms already done
// (the caller ran the first stage in registers); the last stage's outputs go
// to `last`.  The stages are a loop, not unrolled: the code of a transform
// stays a few KB (unrolled by stage and butterfly it was 25-40 KB, and a small
// grid's kernels, each on a few CUs for a few microseconds, fetched it all).
// Inlined so that buf is known to be LDS (ds_read/ds_write, not flat accesses).
// NTH: threads of the workgroup; SWZ: the elements lie at swz<true> (the
// outputs to `last` have their natural index).
template <bool INV, bool P8, int EB, int NTH = NT, bool SWZ = false, typename C, typename Sink>
__device__ __forceinline__ void lds_fft(C *buf, int logn, int nb, const C *tw, const FftTw<INV, C> &pt, int l0,
                                        const Sink &last)
{
    if constexpr (P8) {                    // n = 1024, twiddles loaded for the plan
        lds_fft1024<INV>(buf, nb, pt, l0 ? 1 : 0, last);
    } else {
        const int l4 = 2 * fft_lead4(logn);
        int l = l0;
        for (; l < l4; l += 2) fft_stage<4, INV, (EB * NT + NTH - 1) / NTH, NTH, SWZ, C>(buf, logn, nb, l, tw, l + 2 == logn, last);
        for (; l < logn; l += 3) fft_stage<8, INV, (EB * NT / 2 + NTH - 1) / NTH, NTH, SWZ, C>(buf, logn, nb, l, tw, l + 3 == logn, last);
    }
}

// the twiddle table (or, TWL, its copy in LDS at stw, written by the block;
// read only after a barrier)
template <bool TWL, typename C>
__device__ __forceinline__ const C *tw_table(const C *__restrict__ tw, C *stw, int n)
{
    if constexpr (!TWL) return tw;
    for (int m = threadIdx.x; m < n; m += NT) stw[m] = tw[m];
    return stw;
}

// Instance b of a batched context is blockIdx.y: real fields at b * N,
// spectra at b * S, GMRES state b * gstride bytes after instance 0's.
template <typename T>
struct FftArgs {
    int nx, logn, nv, rows;     // rows: v-rows per workgroup (even)
    int64_t N, S, pitch, gstride;   // pitch: elements from mode to mode of a spectrum
    const cx_t<T> *tw;
    const int32_t *done;
    const T *add;               // rfft: x-only field added to every row, gamma add (null: none), nx per instance
    T gamma;
};

__device__ __forceinline__ int32_t cycle_done(const int32_t *done, int64_t gstride)
{
    return done != nullptr ? *reinterpret_cast<const int32_t *>(reinterpret_cast<const char *>(done) + blockIdx.y * gstride)
                           : 0;
}

// The R real rows' spectra from their packed transforms in buf (complex row
// p = real rows 2p + i 2p+1), stored mode-major: S[k][j0 + r], k <= nx/2.
template <int NTH = NT, typename C>
__device__ __forceinline__ void store_real_spectrum(const C *buf, int nx, int R, int j0, int nv, int64_t pitch,
                                                    C *__restrict__ spec)
{
    using T = typename C::value_type;
    const int nk = (nx >> 1) + 1;
    const T half = T(0.5);
    const int lr = __ffs(R) - 1;
    const bool p2 = (R & (R - 1)) == 0;
    for (int idx = threadIdx.x; idx < nk * R; idx += NTH) {
        const int k = p2 ? idx >> lr : idx / R;
        const int r = idx - k * R;
        if (j0 + r >= nv) continue;
        const C *z = buf + (r >> 1) * nx;
        const C zk = z[k];
        const C zm = z[(nx - k) & (nx - 1)];
        C out;
        if ((r & 1) == 0) out = cmk<C>((zk.x + zm.x) * half, (zk.y - zm.y) * half);
        else out = cmk<C>((zk.y + zm.y) * half, (zm.x - zk.x) * half);
        spec[(size_t)k * pitch + j0 + r] = out;
    }
}

// what J u of a row block needs besides u
struct JacRows {
    const double *uscale;                       // optional device scale of u (GMRES state)
    const double *h0, *h1p, *h1h, *h2p, *h2h;   // 1D factors of H_ave
    const InstConst *inst;
    double ht_inv, factor;
};

}  // namespace
}  // namespace vv
