// In-LDS transforms of real v-rows (Stockham FFT of power-of-two lengths), the
// spectrum's mode-major store and small helpers, shared by the spectral units.
#pragma once

#include "arakawa.h"
#include "cgs_vec.h"

namespace vv {
namespace {

constexpr int NT = 256;
constexpr int MAXE = 4096;   // complex elements of one FFT workgroup (64 KiB of LDS)

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

constexpr int MAXS = 6;     // radix-4 stages of the longest transform (MAXE = 4^6)

// Twiddles of one thread's butterflies, loaded once before a transform of
// length n <= 4 NT.  There every butterfly the thread owns, in any transform
// of the block and any stage, has the index j = threadIdx.x mod n/4 (mod n/2
// in the radix-2 stage of odd logn, where n <= 2 NT), so 3 twiddles per stage
// cover them; their loads are in flight with the tile's own loads instead of
// being waited on after every barrier of the transform.
// n = 1024 runs the plan 4 x 8 x 8 x 4 (see lds_fft1024): its 17 twiddles
// take the same registers, flat index i (always a compile-time index) at
// w[i / 3][i % 3] for i < 15, then w2 and w8 (0..6 and 7..13 for the radix-8
// stages with sub-transforms of 4 and 32, 14..16 for the last radix-4 stage;
// the last row of w, used only by n = 4096, stays out of it).
constexpr int N8 = 1024;
template <bool INV, typename C>
struct FftTw {
    C w[MAXS][3];
    C w2, w8;
    // P8: the n = 1024 plan's twiddles (n must be 1024), else the radix-4 ones
    template <bool P8 = false>
    __device__ __forceinline__ void load(const C *__restrict__ tw, int n, int logn)
    {
        if (P8) {
            const int t = threadIdx.x, ka = t & 3, kb = t & 31, kc = t & 255;
#pragma unroll
            for (int r = 1; r < 8; ++r) {
                w[(r - 1) / 3][(r - 1) % 3] = twiddle<INV>(tw, r * ka * 32);
                w[(6 + r) / 3][(6 + r) % 3] = twiddle<INV>(tw, r * kb * 4);
            }
            w[4][2] = twiddle<INV>(tw, kc);
            w2 = twiddle<INV>(tw, 2 * kc);
            w8 = twiddle<INV>(tw, 3 * kc);
            return;
        }
        const int ns = logn >> 1;
        const int j = threadIdx.x & ((n >> 2) - 1);
#pragma unroll
        for (int s = 0; s < MAXS; ++s) {
            if (s < ns) {
                const int st = (j & ((1 << (2 * s)) - 1)) << (logn - 2 - 2 * s);
                w[s][0] = twiddle<INV>(tw, st);
                w[s][1] = twiddle<INV>(tw, 2 * st);
                w[s][2] = twiddle<INV>(tw, 3 * st);
            }
        }
        if (logn & 1) {
            const int jj = threadIdx.x & ((n >> 1) - 1);
            w2 = twiddle<INV>(tw, (jj & ((1 << (2 * ns)) - 1)) << (logn - 1 - 2 * ns));
        }
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
            for (int r = 1; r < 8; ++r) v[q][r] = cmul(v[q][r], pt.w[(OFF + r - 1) / 3][(OFF + r - 1) % 3]);
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
            v[q][1] = cmul(v[q][1], pt.w[4][2]);
            v[q][2] = cmul(v[q][2], pt.w2);
            v[q][3] = cmul(v[q][3], pt.w8);
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

// Batched in-LDS Stockham FFT of `nb` transforms of length n = 2^logn stored
// back to back in buf.  Forward uses exp(-2 pi i m/n), inverse the conjugate
// (unnormalised).  Each stage loads every butterfly of the thread into
// registers, synchronises, then stores, so one buffer suffices.  C is
// double2 (FP64 path) or float2 (FP32 preconditioner of the mixed solver).
// PRE: twiddles from pt (n <= 4 NT), else from the global table tw.  P8:
// n = 1024 by the 4 x 8 x 8 x 4 plan (pt loaded with load<true>).
// s0: first radix-4 stage to run (1 when the caller did stage 0 in
// registers); the last stage's outputs go to `last`.
// Inlined so that buf is known to be LDS (ds_read/ds_write, not flat
// accesses); index arithmetic by shifts (n is a power of two).
template <bool INV, bool PRE, bool P8 = false, typename C, typename Sink>
__device__ __forceinline__ void lds_fft(C *buf, int n, int logn, int nb, const C *__restrict__ tw,
                                        const FftTw<INV, C> &pt, int s0, const Sink &last)
{
    if (P8) {                              // n = 1024, twiddles loaded for the plan
        lds_fft1024<INV>(buf, nb, pt, s0, last);
        return;
    }
    const int nq = n >> 2, lq = logn - 2, ns = logn >> 1;
    const int total4 = nb * nq;
#pragma unroll
    for (int s = 0; s < MAXS; ++s) {
        if (s >= ns) break;                // uniform over the block
        if (s < s0) continue;
        const int Ns = 1 << (2 * s);
        C v[MAXE / 4 / NT][4];
        int dst[MAXE / 4 / NT];
#pragma unroll
        for (int q = 0; q < MAXE / 4 / NT; ++q) {
            const int t = threadIdx.x + q * NT;
            dst[q] = -1;
            if (t < total4) {
                const int b = t >> lq;
                const int j = t & (nq - 1);
                const int k = j & (Ns - 1);
                const C *src = buf + (b << logn);
#pragma unroll
                for (int r = 0; r < 4; ++r) v[q][r] = src[j + r * nq];
                if (PRE) {
                    v[q][1] = cmul(v[q][1], pt.w[s][0]);
                    v[q][2] = cmul(v[q][2], pt.w[s][1]);
                    v[q][3] = cmul(v[q][3], pt.w[s][2]);
                } else {
                    const int st = k << (lq - 2 * s);
                    v[q][1] = cmul(v[q][1], twiddle<INV>(tw, st));
                    v[q][2] = cmul(v[q][2], twiddle<INV>(tw, 2 * st));
                    v[q][3] = cmul(v[q][3], twiddle<INV>(tw, 3 * st));
                }
                const C a0 = cadd(v[q][0], v[q][2]);
                const C a1 = csub(v[q][0], v[q][2]);
                const C a2 = cadd(v[q][1], v[q][3]);
                const C d = csub(v[q][1], v[q][3]);
                // forward: (v1 - v3) * (-i); inverse: (v1 - v3) * (+i)
                const C a3 = INV ? cmk<C>(-d.y, d.x) : cmk<C>(d.y, -d.x);
                v[q][0] = cadd(a0, a2);
                v[q][1] = cadd(a1, a3);
                v[q][2] = csub(a0, a2);
                v[q][3] = csub(a1, a3);
                dst[q] = (b << logn) + ((j - k) << 2) + k;
            }
        }
        __syncthreads();
        const bool fin = (s == ns - 1) && !(logn & 1);
#pragma unroll
        for (int q = 0; q < MAXE / 4 / NT; ++q) {
            if (dst[q] >= 0) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (fin) last(dst[q] + r * Ns, v[q][r]);
                    else buf[dst[q] + r * Ns] = v[q][r];
                }
            }
        }
        __syncthreads();
    }
    if (logn & 1) {
        const int Ns = 1 << (2 * ns);
        const int nh = n >> 1;
        const int total = nb * nh;
        C v[MAXE / 2 / NT][2];
        int dst[MAXE / 2 / NT];
#pragma unroll
        for (int q = 0; q < MAXE / 2 / NT; ++q) {
            const int t = threadIdx.x + q * NT;
            dst[q] = -1;
            if (t < total) {
                const int b = t >> (logn - 1);
                const int j = t & (nh - 1);
                const int k = j & (Ns - 1);
                const C *src = buf + (b << logn);
                const C x0 = src[j];
                const C w = PRE ? pt.w2 : twiddle<INV>(tw, k << (logn - 1 - 2 * ns));
                const C x1 = cmul(src[j + nh], w);
                v[q][0] = cadd(x0, x1);
                v[q][1] = csub(x0, x1);
                dst[q] = (b << logn) + ((j - k) << 1) + k;
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < MAXE / 2 / NT; ++q) {
            if (dst[q] >= 0) {
                last(dst[q], v[q][0]);
                last(dst[q] + Ns, v[q][1]);
            }
        }
        __syncthreads();
    }
}

// Instance b of a batched context is blockIdx.y: real fields at b * N,
// spectra at b * S, GMRES state b * gstride bytes after instance 0's.
template <typename T>
struct FftArgs {
    int nx, logn, nv, rows;     // rows: v-rows per workgroup (even)
    int64_t N, S, gstride;
    const cx_t<T> *tw;
    const int32_t *done;
};

__device__ __forceinline__ int32_t cycle_done(const int32_t *done, int64_t gstride)
{
    return done != nullptr ? *reinterpret_cast<const int32_t *>(reinterpret_cast<const char *>(done) + blockIdx.y * gstride)
                           : 0;
}

// The R real rows' spectra from their packed transforms in buf (complex row
// p = real rows 2p + i 2p+1), stored mode-major: S[k][j0 + r], k <= nx/2.
template <typename C>
__device__ __forceinline__ void store_real_spectrum(const C *buf, int nx, int R, int j0, int nv, C *__restrict__ spec)
{
    using T = typename C::value_type;
    const int nk = (nx >> 1) + 1;
    const T half = T(0.5);
    for (int idx = threadIdx.x; idx < nk * R; idx += NT) {
        const int k = idx / R;
        const int r = idx - k * R;
        if (j0 + r >= nv) continue;
        const C *z = buf + (r >> 1) * nx;
        const C zk = z[k];
        const C zm = z[(nx - k) & (nx - 1)];
        C out;
        if ((r & 1) == 0) out = cmk<C>((zk.x + zm.x) * half, (zk.y - zm.y) * half);
        else out = cmk<C>((zk.y + zm.y) * half, (zm.x - zk.x) * half);
        spec[(size_t)k * nv + j0 + r] = out;
    }
}

}  // namespace
}  // namespace vv
