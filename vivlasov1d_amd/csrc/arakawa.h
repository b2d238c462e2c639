// The Arakawa J1 / J2 / J4 stencils on one lane's sliding register window,
// shared by the bracket kernels (bracket.hip) and the Jacobian-vector product
// fused with the forward rFFT (spectral.hip, rows.hip).
//
// Every expression keeps the reference's IEEE operation order
// (PoissonBracket.pyx:100-113, 221-234, 360-389; C left-to-right) and is
// evaluated without contraction whatever the including unit's setting (the
// pragma below), so the callbacks that return a bracket produce the
// reference's unfused double results bit for bit.  The solver's own J u and
// F(f) use the factored form (SepWin), with the products fused explicitly, so
// every kernel that forms them agrees bit for bit whatever its unit's setting.
//
// The window of a lane at column cx, output row cy of a tile (read through
// a functor of (row, column, column offset)) holds the first argument F and the second
// argument H at column 0: rows cy-2..cy+2, columns +-1: rows cy-1..cy+1,
// columns +-2: row cy; it moves one row down per output row, so a row costs
// 5 + 5 LDS reads instead of 25.
#pragma once

#include "vv1d_internal.h"

namespace vv {
namespace {

// Cell (r, cx + d) of an LDS tile of pitch P (the column offset d is a
// compile-time constant at every call, so it folds into the LDS address).
template <typename T, int P>
struct TileRd {
    const T *p;
    __device__ __forceinline__ T operator()(int r, int cx, int d) const { return p[r * P + cx + d]; }
};

template <typename T>
struct ArakawaWin {
    T f0[5], fm[3], fp[3], fm2, fp2;
    T g0[5], gm[3], gp[3], gm2, gp2;

    template <typename RF, typename RH>
    __device__ __forceinline__ void load(const RF &F, const RH &H, int cy, int cx)
    {
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            f0[k] = F(cy - 2 + k, cx, 0);
            g0[k] = H(cy - 2 + k, cx, 0);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            fm[k] = F(cy - 1 + k, cx, -1);
            fp[k] = F(cy - 1 + k, cx, 1);
            gm[k] = H(cy - 1 + k, cx, -1);
            gp[k] = H(cy - 1 + k, cx, 1);
        }
        fm2 = F(cy, cx, -2);
        fp2 = F(cy, cx, 2);
        gm2 = H(cy, cx, -2);
        gp2 = H(cy, cx, 2);
    }

    // move to output row cn (= the current row + 1)
    template <typename RF, typename RH>
    __device__ __forceinline__ void advance(const RF &F, const RH &H, int cn, int cx)
    {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            f0[k] = f0[k + 1];
            g0[k] = g0[k + 1];
        }
        f0[4] = F(cn + 2, cx, 0);
        g0[4] = H(cn + 2, cx, 0);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            fm[k] = fm[k + 1];
            fp[k] = fp[k + 1];
            gm[k] = gm[k + 1];
            gp[k] = gp[k + 1];
        }
        fm[2] = F(cn + 1, cx, -1);
        fp[2] = F(cn + 1, cx, 1);
        gm[2] = H(cn + 1, cx, -1);
        gp[2] = H(cn + 1, cx, 1);
        fm2 = F(cn, cx, -2);
        fp2 = F(cn, cx, 2);
        gm2 = H(cn, cx, -2);
        gp2 = H(cn, cx, 2);
    }
};

// base + factor {F, H} at the window's centre (the reference's
// Y += factor * bracket with Y = base).
template <int KIND, typename T>
__device__ __forceinline__ T arakawa_add(const ArakawaWin<T> &w, T base, T factor, T af1, T af2)
{
#pragma clang fp contract(off)
#define F(di, dj) ((di) == 0 ? w.f0[(dj) + 2] : (di) == -1 ? w.fm[(dj) + 1] : (di) == 1 ? w.fp[(dj) + 1] : (di) == -2 ? w.fm2 : w.fp2)
#define H(di, dj) ((di) == 0 ? w.g0[(dj) + 2] : (di) == -1 ? w.gm[(dj) + 1] : (di) == 1 ? w.gp[(dj) + 1] : (di) == -2 ? w.gm2 : w.gp2)
    if (KIND == VV_BRACKET_J1 || KIND == VV_BRACKET_J4) {
        // PoissonBracket.pyx:100-111 (J1 / second order)
        const T jpp = (F(1, 0) - F(-1, 0)) * (H(0, 1) - H(0, -1))
                    - (F(0, 1) - F(0, -1)) * (H(1, 0) - H(-1, 0));
        const T jpc = F(1, 0) * (H(1, 1) - H(1, -1))
                    - F(-1, 0) * (H(-1, 1) - H(-1, -1))
                    - F(0, 1) * (H(1, 1) - H(-1, 1))
                    + F(0, -1) * (H(1, -1) - H(-1, -1));
        const T jcp = F(1, 1) * (H(0, 1) - H(1, 0))
                    - F(-1, -1) * (H(-1, 0) - H(0, -1))
                    - F(-1, 1) * (H(0, 1) - H(-1, 0))
                    + F(1, -1) * (H(1, 0) - H(0, -1));
        if (KIND == VV_BRACKET_J1) return base + factor * (jpp + jpc + jcp) * af1;
        // PoissonBracket.pyx:373-389 (J4 = 2 J1 - J2)
        const T jcc2 = (F(1, 1) - F(-1, -1)) * (H(-1, 1) - H(1, -1))
                     - (F(-1, 1) - F(1, -1)) * (H(1, 1) - H(-1, -1));
        const T jpc2 = F(2, 0) * (H(1, 1) - H(1, -1))
                     - F(-2, 0) * (H(-1, 1) - H(-1, -1))
                     - F(0, 2) * (H(1, 1) - H(-1, 1))
                     + F(0, -2) * (H(1, -1) - H(-1, -1));
        const T jcp2 = F(1, 1) * (H(0, 2) - H(2, 0))
                     - F(-1, -1) * (H(-2, 0) - H(0, -2))
                     - F(-1, 1) * (H(0, 2) - H(-2, 0))
                     + F(1, -1) * (H(2, 0) - H(0, -2));
        const T r1 = (jpp + jpc + jcp) * af1;
        const T r2 = (jcc2 + jpc2 + jcp2) * af2;
        return base + factor * (T(2) * r1 - r2);
    } else {
        // PoissonBracket.pyx:221-234 (J2)
        const T jcc = (F(1, 1) - F(-1, -1)) * (H(-1, 1) - H(1, -1))
                    - (F(-1, 1) - F(1, -1)) * (H(1, 1) - H(-1, -1));
        const T jpc = F(2, 0) * (H(1, 1) - H(1, -1))
                    - F(-2, 0) * (H(-1, 1) - H(-1, -1))
                    - F(0, 2) * (H(1, 1) - H(-1, 1))
                    + F(0, -2) * (H(1, -1) - H(-1, -1));
        const T jcp = F(1, 1) * (H(0, 2) - H(2, 0))
                    - F(-1, -1) * (H(-2, 0) - H(0, -2))
                    - F(-1, 1) * (H(0, 2) - H(-2, 0))
                    + F(1, -1) * (H(2, 0) - H(0, -2));
        return base + factor * (jcc + jpc + jcp) * af2;
    }
#undef F
#undef H
}

// The same stencils where H = h0(v) + phi(x), as H_ave always is: every term is
// a difference of H, so with the row differences of h0 and the column
// differences of phi
//   c1 J1 + c2 J2 = A+ D+ + A0 D0 + A- D- + A2 D2 - (B+ E+ + B0 E0 + B- E- + B2 E2),
// D+, D0, D- = F(1, b) - F(-1, b) for b = 1, 0, -1, D2 = F(2, 0) - F(-2, 0);
// E+, E0, E- = F(b, 1) - F(b, -1) for b = 1, 0, -1, E2 = F(0, 2) - F(0, -2);
// A depends on the row, B on the column:
//   A+- = c1 v+- + c2 (V + v2+-), A0 = 2 c1 V, A2 = c2 V   (B alike from phi)
// v+ = h0(1) - h0(0), v- = h0(0) - h0(-1), V = h0(1) - h0(-1), v2+ = h0(2) -
// h0(0), v2- = h0(0) - h0(-2).  No H in LDS, 5 reads and 17 operations a point
// instead of 10 and ~75, and closer to exact: the unfactored stencil subtracts
// values of H rounded at |H|, which costs |H| / (hv dH/dv) ulps.  The solver's
// J u and P^-1 F use it; the callbacks that return F and J u themselves keep the
// reference's operation order above.
__device__ __forceinline__ double phi_ave(double x0, double x1, double x2, double x3)
{
#pragma clang fp contract(off)
    return ((0.5 * x0 + 0.5 * x1) + 0.5 * x2) + 0.5 * x3;
}

// c1, c2 of factor {F, H}: J1, J2 or J4 = 2 J1 - J2
__device__ __forceinline__ void sep_weights(int kind, double factor, double af1, double af2, double &c1, double &c2)
{
#pragma clang fp contract(off)
    c1 = kind == VV_BRACKET_J2 ? 0.0 : kind == VV_BRACKET_J4 ? 2.0 * (factor * af1) : factor * af1;
    c2 = kind == VV_BRACKET_J1 ? 0.0 : kind == VV_BRACKET_J4 ? -(factor * af2) : factor * af2;
}

// A (or B) from the five values of h0 (or phi) around the centre h.  J1 has no
// terms at distance 2: those values are left out, not multiplied by 0 (an
// infinity or NaN there would spread to points whose stencil does not hold it).
template <typename T>
__device__ __forceinline__ void sep_coef(double hmm, double hm, double h, double hp, double hpp, double c1, double c2,
                                         T (&k)[4])
{
#pragma clang fp contract(off)
    const double W = hp - hm;
    const bool far = c2 != 0.0;
    k[0] = (T)(c1 * (hp - h) + (far ? c2 * (W + (hpp - h)) : 0.0));
    k[1] = (T)(2.0 * (c1 * W));
    k[2] = (T)(c1 * (h - hm) + (far ? c2 * (W + (h - hmm)) : 0.0));
    k[3] = (T)(c2 * W);
}

// row j's coefficients from h0 itself (rows past the grid read as 0: they only
// meet rows whose result is not formed)
template <typename T>
__device__ __forceinline__ void sep_row(const double *__restrict__ h0, int j, int nv, double c1, double c2, T *k)
{
    double h[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        const int r = j - 2 + q;
        h[q] = r >= 0 && r < nv ? h0[r] : 0.0;
    }
    T a[4];
    sep_coef(h[0], h[1], h[2], h[3], h[4], c1, c2, a);
#pragma unroll
    for (int q = 0; q < 4; ++q) k[q] = a[q];
}

// the points of a kind's stencil besides the diagonal ones: the nearest
// neighbours, and those at distance 2
constexpr bool sep_near(int kind) { return kind != VV_BRACKET_J2; }
constexpr bool sep_far(int kind) { return kind != VV_BRACKET_J1; }

// The first argument's window alone.
template <typename T>
struct SepWin {
    T f0[5], fm[3], fp[3], fm2, fp2;

    template <typename RF>
    __device__ __forceinline__ void load(const RF &F, int cy, int cx)
    {
#pragma unroll
        for (int k = 0; k < 5; ++k) f0[k] = F(cy - 2 + k, cx, 0);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            fm[k] = F(cy - 1 + k, cx, -1);
            fp[k] = F(cy - 1 + k, cx, 1);
        }
        fm2 = F(cy, cx, -2);
        fp2 = F(cy, cx, 2);
    }

    template <typename RF>
    __device__ __forceinline__ void advance(const RF &F, int cn, int cx)
    {
#pragma unroll
        for (int k = 0; k < 4; ++k) f0[k] = f0[k + 1];
        f0[4] = F(cn + 2, cx, 0);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            fm[k] = fm[k + 1];
            fp[k] = fp[k + 1];
        }
        fm[2] = F(cn + 1, cx, -1);
        fp[2] = F(cn + 1, cx, 1);
        fm2 = F(cn, cx, -2);
        fp2 = F(cn, cx, 2);
    }

    // the weighted bracket at the centre, of the points that the kind's stencil
    // holds: J1 none at distance 2, J2 no nearest neighbours (coefficients that
    // are 0, but an infinity or NaN would come through them)
    __device__ __forceinline__ T bracket(const T *A, const T (&B)[4], bool near, bool far) const
    {
#pragma clang fp contract(off)
        T s = A[0] * (fp[2] - fm[2]), t = B[0] * (fp[2] - fp[0]);
        if (near) {
            s = fma_t(A[1], fp[1] - fm[1], s);
            t = fma_t(B[1], f0[3] - f0[1], t);
        }
        s = fma_t(A[2], fp[0] - fm[0], s);
        t = fma_t(B[2], fm[2] - fm[0], t);
        if (far) {
            s = fma_t(A[3], fp2 - fm2, s);
            t = fma_t(B[3], f0[4] - f0[0], t);
        }
        return s - t;
    }

    static __device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }
    static __device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
};

// H_ave at (i, j) from its 1D factors: ((((h0_j + .5 h1p_i) + .5 h1h_i) +
// .5 h2p_i) + .5 h2h_i), exactly the value the reference's 2D Have vector
// holds (PETScVlasovSolver.pyx:145-149).
__device__ __forceinline__ double compose_have(double h0, double x0, double x1, double x2, double x3)
{
#pragma clang fp contract(off)
    return (((h0 + 0.5 * x0) + 0.5 * x1) + 0.5 * x2) + 0.5 * x3;
}

// The Jacobian's Y = 0; Y += u/dt (PETScNLVlasovMP.pyx:35-36).
template <typename T>
__device__ __forceinline__ T jacobian_base(T ht_inv, T u)
{
#pragma clang fp contract(off)
    return T(0) + ht_inv * u;
}

// the result times the Krylov vector's scale, rounded on its own
template <typename T>
__device__ __forceinline__ T scaled(T f, T s)
{
#pragma clang fp contract(off)
    return f * s;
}

}  // namespace
}  // namespace vv
