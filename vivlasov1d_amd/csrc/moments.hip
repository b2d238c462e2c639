// Moments, the periodic Poisson solve and the invariants.
//
//  column_kernel     column sums over v-rows of f (n_i = hv * sum_j f_ij,
//                    Toolbox.pyx:79-98) or of v f and v^2 f (u_i, e_i, the
//                    output moments, Toolbox.pyx:103-148); one chunk of rows
//                    per block row.
//  poisson_kernel    one workgroup per instance: finishes n, forms
//                    b = -(n - mean n) q (PETScPoissonSolver.pyx:58-74),
//                    solves A phi = b by the mean-free inverse of the periodic
//                    (circulant) CFD4/CFD2 matrix, then h1 = phi - mean phi
//                    (Toolbox.pyx:38-74) and the Poisson residual norm
//                    ||A phi + (n - mean n) q|| of run_base.py:631-637.
//  poisson_prep / conv / post_kernel
//                    the same in three launches, the convolution spread over
//                    the chip, for x-grids of more than 256 points that are no
//                    power of two.
//  invariants_kernel mass, L2, kinetic / potential energy over f, plus the
//                    field energy over phi (distribution_function.pyx:130-199,
//                    hamiltonian.pyx:67-100, potential.pyx:48-59).
//
// In a batched context instance b is blockIdx.y (blockIdx.z for the column
// sums); its fields start at b * N, its x-vectors at b * nx.
#include "fft_lds.h"
#include "vv1d_internal.h"

namespace vv {
namespace {

constexpr int PT = 1024;     // threads of the single-workgroup Poisson kernel
constexpr int DCH = kDensityChunks;   // row chunks of the density reduction

// Column sums over v-rows.  A workgroup owns 64 columns (one per lane, 512-byte
// row segments) and a chunk of the rows, dealt to its 16 wavefronts in turn;
// eight loads per lane are in flight.  MOM 0: sum_j f into out0; MOM 1:
// sum_j v_j f into out0 and sum_j v_j^2 f into out1.  Partial sums go to
// out[chunk][i]; with one chunk they are the sums, and scale (hv, else 1) is
// applied here.  HBM-bound for large grids, one memory latency for small ones.
// One thread per column (four workgroups at nx = 1000) took 429 us for both
// velocity moments of 1000 x 2001; density took 10.3 us at 1024 x 2048 with
// one wavefront per 64 columns and 32 rows.
constexpr int CW = 16;
template <int MOM>
__global__ __launch_bounds__(64 * CW) void column_kernel(const double *__restrict__ f, const double *__restrict__ v,
                                                         int nx, int nv, int rows, int64_t ostride, double scale,
                                                         double *__restrict__ out0, double *__restrict__ out1)
{
    __shared__ double red[MOM + 1][CW][64];
    f += (size_t)blockIdx.z * nx * nv;
    out0 += blockIdx.z * ostride + (size_t)blockIdx.y * nx;
    if (MOM) out1 += blockIdx.z * ostride + (size_t)blockIdx.y * nx;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    const int j0 = blockIdx.y * rows, j1 = min(nv, j0 + rows);
    double s = 0.0, t = 0.0;
    if (i < nx) {
        const double *fp = f + i;
        for (int j = j0 + w; j < j1; j += 8 * CW) {
            double x[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int r = j + q * CW;
                const double y = fp[(size_t)(r < j1 ? r : j0) * nx];
                x[q] = r < j1 ? y : 0.0;
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                if (MOM) {
                    const int r = j + q * CW;
                    const double vv = v[r < j1 ? r : j0];
                    s += vv * x[q];
                    t += (vv * vv) * x[q];          // v2 = v**2 (Grid), then v2_j * f_ij
                } else {
                    s += x[q];
                }
            }
        }
    }
    red[0][w][lane] = s;
    if (MOM) red[MOM][w][lane] = t;
    __syncthreads();
    if (w <= MOM && i < nx) {
        double a = red[w][0][lane];
#pragma unroll
        for (int q = 1; q < CW; ++q) a += red[w][q][lane];
        (w == 0 ? out0 : out1)[i] = a * scale;
    }
}

// the chunks' partial sums of x-vectors part0 (and part1, when out1), times scale
__global__ __launch_bounds__(NT) void column_finish_kernel(const double *__restrict__ part0,
                                                           const double *__restrict__ part1, int nch, int nx,
                                                           int64_t pstride, double scale, double *__restrict__ out0,
                                                           double *__restrict__ out1)
{
    const int i = blockIdx.x * NT + threadIdx.x;
    if (i >= nx) return;
    const double *p = blockIdx.z ? part1 : part0;
    double *out = (blockIdx.z ? out1 : out0) + (size_t)blockIdx.y * nx;
    p += blockIdx.y * pstride;
    double s = 0.0;
    for (int ch = 0; ch < nch; ++ch) s += p[(size_t)ch * nx + i];
    out[i] = s * scale;
}

// Chunks of rows of the column sums (<= kDensityChunks / 2, so the two velocity
// moments fit the density's scratch; a function of nv alone, so that a batched
// instance sums as it would alone): 128 rows a chunk, one round of eight loads
// a lane and 256 workgroups at 1024 x 2048.
int column_chunks(int nv)
{
    const int n = (nv + 127) / 128;
    return n < kDensityChunks / 2 ? n : kDensityChunks / 2;
}
// Where the sums themselves are wanted, up to 512 rows go in one chunk: 32 rows
// a wavefront, and no finish launch (velocity moments of 100 x 200: 43.5 us
// before).
int sum_chunks(int nv) { return nv <= 512 ? 1 : column_chunks(nv); }

__device__ __forceinline__ double block_sum_big(double v, double *red)
{
    const double ws = wave_sum(v);
    __syncthreads();                   // the sum before is read
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ws;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < PT / 64; ++w) s += red[w];
    return s;                          // valid in every thread
}

struct PoiArgs {
    int nx, laplace, from_part;
    int nch, logn;         // density partials per column; log2 nx (FFT form)
    int64_t npstride;      // instance stride of npart
    double hv, charge;
    const InstConst *inst;
    const double *npart;   // density partials (from_part = 1)
    const double *n_in;    // density (from_part = 0)
    const double *pinv;    // first row of the mean-free circulant inverse
    const double *plam;    // FFT form: inverse symbol over nx, 0 for the mean
    const double2 *tw;     // FFT form: exp(-2 pi i m / nx)
    double *work;          // 3*nx + 1 scratch: b | phi | n | mean n
    double *n_out, *phi, *h1, *pres;
    int pres_stride;       // doubles between the instances' residual norms in pres
};

// A x for the periodic CFD4 / CFD2 stencils, in the reference's order
// (PETScPoissonCFD4.pyx:78, PETScPoissonCFD2.pyx:78).
template <typename X>
__device__ __forceinline__ double lap(const X &x, int i, int nx, int laplace, double hx2_inv)
{
    const int im2 = i >= 2 ? i - 2 : i - 2 + nx, im1 = i >= 1 ? i - 1 : i - 1 + nx;
    const int ip1 = i + 1 < nx ? i + 1 : i + 1 - nx, ip2 = i + 2 < nx ? i + 2 : i + 2 - nx;
    const double xm2 = x[im2], xm1 = x[im1], x0 = x[i], xp1 = x[ip1], xp2 = x[ip2];
    if (laplace == VV_LAPLACE_CFD4)
        return (5. * xm2 - 32. * xm1 + 54. * x0 - 32. * xp1 + 5. * xp2) * hx2_inv / 12.;
    return (2. * x0 - xm1 - xp1) * hx2_inv;
}

// per-instance views of the Poisson buffers (pres: 16 doubles per instance)
__device__ __forceinline__ void poi_instance(PoiArgs &a)
{
    const size_t b = blockIdx.y, nx = a.nx;
    if (a.npart) a.npart += b * a.npstride;
    if (a.n_in) a.n_in += b * nx;
    if (a.pinv) a.pinv += b * nx;
    if (a.plam) a.plam += b * nx;
    a.work += b * (3 * nx + 1);
    if (a.n_out) a.n_out += b * nx;
    if (a.phi) a.phi += b * nx;
    if (a.h1) a.h1 += b * nx;
    if (a.pres) a.pres += b * a.pres_stride;
}

// n_i of the thread's columns i = t + q PT from the density partials, or as
// given; `on` marks the columns that exist.  Grids of up to PT/2 columns
// deal the chunks to PT / span threads a column (span: the columns padded to
// a power of two), whose sums are added in order.
__device__ __forceinline__ void poi_density(const PoiArgs &a, double (&n)[kMaxNx / PT], double *red)
{
    const int nx = a.nx, t = threadIdx.x;
#pragma unroll
    for (int q = 0; q < kMaxNx / PT; ++q) n[q] = 0.0;        // columns past nx count as 0
    if (a.from_part && a.nch > 1 && 2 * nx <= PT) {
        int span = 64;
        while (span < nx) span <<= 1;
        const int g = t / span, i = t & (span - 1), G = PT / span;
        double s = 0.0;
        if (i < nx) {
            for (int c0 = g; c0 < a.nch; c0 += 8 * G) {      // eight loads in flight
                double v[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) v[c] = c0 + c * G < a.nch ? a.npart[(size_t)(c0 + c * G) * nx + i] : 0.0;
#pragma unroll
                for (int c = 0; c < 8; ++c) s += v[c];
            }
        }
        red[t] = s;
        __syncthreads();
        if (t < nx) {
            double v = red[t];
            for (int q = 1; q < G; ++q) v += red[q * span + t];
            n[0] = v * a.hv;
        }
        __syncthreads();
        return;
    }
#pragma unroll
    for (int q = 0; q < kMaxNx / PT; ++q) {
        const int i = t + q * PT;
        if (i >= nx) continue;
        if (!a.from_part) {
            n[q] = a.n_in[i];
            continue;
        }
        double s = 0.0;
        for (int c0 = 0; c0 < a.nch; c0 += 8) {
            double v[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) v[c] = c0 + c < a.nch ? a.npart[(size_t)(c0 + c) * nx + i] : 0.0;
#pragma unroll
            for (int c = 0; c < 8; ++c) s += v[c];
        }
        n[q] = s * a.hv;
    }
}

struct ReX {                             // real parts of a complex line
    const double2 *p;
    __device__ __forceinline__ double operator[](int i) const { return p[i].x; }
};

// The whole Poisson pipeline of an instance in one workgroup.  FFT: nx a power
// of two whose twiddles the context holds; phi = F^-1 (b^ / lambda), two
// in-LDS transforms.  Otherwise (nx <= kPoissonOne): the convolution with the
// first row of the circulant inverse, dealt to PT / span threads an output.
// Latency-bound (barriers, LDS passes); what it saves is two dependent
// launches and the pass over `work`: prep + conv + post took 13.0 + 11.2 +
// 4.3 us at nx = 1024 and 6.1 + 2.7 + 3.3 us at nx = 64.  The convolution up to 256
// points, four threads an output; with two (257 .. 512) its chain of sums takes
// longer than the three launches: 12.9 us at 260 and 13.9 at 300, where they take
// 10.3 and 10.5.
constexpr int kPoissonOne = 256;
constexpr int kPoissonTw = 2048;
template <bool FFT>
__global__ __launch_bounds__(PT) void poisson_kernel(PoiArgs a)
{
    extern __shared__ double2 pline[];
    __shared__ double red[PT];
    __shared__ double rs[PT / 64 + 1];
    poi_instance(a);
    const double hx2_inv = a.inst[blockIdx.y].hx2_inv;
    const int nx = a.nx, t = threadIdx.x;
    constexpr int Q = kMaxNx / PT;
    // the symbol and (up to 2048 points) the twiddles' LDS copy, in flight with n
    double lam[Q];
    const double2 *tw = a.tw;
    if (FFT) {
#pragma unroll
        for (int q = 0; q < Q; ++q) lam[q] = t + q * PT < nx ? a.plam[t + q * PT] : 0.0;
        if (nx <= kPoissonTw) {
            double2 *stw = pline + nx;
            for (int m = t; m < nx; m += PT) stw[m] = a.tw[m];
            tw = stw;
        }
    }
    double n[Q];
    poi_density(a, n, red);
    double part = 0.0;
#pragma unroll
    for (int q = 0; q < Q; ++q) part += n[q];            // columns past nx hold 0
    const double nmean = block_sum_big(part, rs) / nx;
    double *sb = reinterpret_cast<double *>(pline), *sc = sb + nx;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = t + q * PT;
        if (i >= nx) continue;
        if (a.n_out) a.n_out[i] = n[q];
        const double b = -(n[q] - nmean) * a.charge;
        if (FFT) {
            pline[i] = double2{b, 0.0};
        } else {
            sb[i] = b;
            sc[i] = a.pinv[i];
        }
    }
    __syncthreads();
    if (FFT) {
        // at most one butterfly a thread: nx / 4 <= PT
        lds_fft<false, false, 1>(pline, a.logn, 1, tw, FftTw<false, double2>{}, 0, LdsSink<double2>{pline});
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int i = t + q * PT;
            if (i < nx) pline[i] = double2{pline[i].x * lam[q], pline[i].y * lam[q]};
        }
        __syncthreads();
        lds_fft<true, false, 1>(pline, a.logn, 1, tw, FftTw<true, double2>{}, 0, LdsSink<double2>{pline});
    } else {
        int span = 64;
        while (span < nx) span <<= 1;
        const int G = PT / span, g = t / span, i = t & (span - 1);
        const int len = (nx + G - 1) / G, m0 = g * len, m1 = m0 + len < nx ? m0 + len : nx;
        double s0 = 0.0, s1 = 0.0;
        if (i < nx) {
            int d = i - m0;                              // (i - m) mod nx, kept in [0, nx)
            d = d < 0 ? d + nx : d;
            for (int m = m0; m < m1; m += 2) {
                s0 += sc[m] * sb[d];
                d = d == 0 ? nx - 1 : d - 1;
                if (m + 1 < m1) s1 += sc[m + 1] * sb[d];
                d = d == 0 ? nx - 1 : d - 1;
            }
        }
        red[t] = s0 + s1;
        __syncthreads();
        if (t < nx) {
            double s = red[t];
            for (int q = 1; q < G; ++q) s += red[q * span + t];
            sb[t] = s;                                   // phi takes b's place
        }
        __syncthreads();
    }
    part = 0.0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = t + q * PT;
        if (i < nx) part += FFT ? pline[i].x : sb[i];
    }
    const double phiave = block_sum_big(part, rs) / nx;
    part = 0.0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = t + q * PT;
        if (i >= nx) continue;
        const double p = FFT ? pline[i].x : sb[i];
        if (a.phi) a.phi[i] = p;
        if (a.h1) a.h1[i] = p - phiave;
        const double l = FFT ? lap(ReX{pline}, i, nx, a.laplace, hx2_inv) : lap(sb, i, nx, a.laplace, hx2_inv);
        const double r = l + (n[q] - nmean) * a.charge;
        part += r * r;
    }
    if (a.pres == nullptr) return;                       // uniform over the block
    const double rr = block_sum_big(part, rs);
    if (t == 0) *a.pres = sqrt(rr);
}

// one workgroup: n (from the density partials), mean n, b = -(n - mean n) q
__global__ __launch_bounds__(PT) void poisson_prep_kernel(PoiArgs a)
{
    __shared__ double red[PT];
    __shared__ double rs[PT / 64 + 1];
    poi_instance(a);
    const int nx = a.nx;
    double *b = a.work, *wn = a.work + 2 * nx;
    constexpr int Q = kMaxNx / PT;
    double n[Q];
    poi_density(a, n, red);
    double part = 0.0;
#pragma unroll
    for (int q = 0; q < Q; ++q) part += n[q];
    const double nmean = block_sum_big(part, rs) / nx;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int i = threadIdx.x + q * PT;
        if (i >= nx) continue;
        wn[i] = n[q];
        if (a.n_out) a.n_out[i] = n[q];
        b[i] = -(n[q] - nmean) * a.charge;
    }
    if (threadIdx.x == 0) a.work[3 * nx] = nmean;
}

// phi_i = sum_m c_m b_{i-m}: C the mean-free circulant inverse of A.  A
// workgroup forms 64 outputs (one per lane); its 4 wavefronts take a quarter
// of the m range each, with 4 interleaved accumulators per lane, and the
// quarters are added in order: fixed summation order, chains of nx/16 terms.
constexpr int CONV_OUT = 64;
__global__ __launch_bounds__(NT) void poisson_conv_kernel(PoiArgs a)
{
    extern __shared__ double sm[];
    __shared__ double part[NT / 64][CONV_OUT];
    poi_instance(a);
    const int nx = a.nx;
    double *sb = sm, *sc = sm + nx;
    for (int i = threadIdx.x; i < nx; i += NT) {
        sb[i] = a.work[i];
        sc[i] = a.pinv[i];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = blockIdx.x * CONV_OUT + lane;
    const int q = (nx + NT / 64 - 1) / (NT / 64);
    const int m0 = wave * q, m1 = m0 + q < nx ? m0 + q : nx;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    if (i < nx) {
        int m = m0;
        int d = i - m0;                          // (i - m) mod nx, kept in [0, nx)
        d = d < 0 ? d + nx : d;
        for (; m + 4 <= m1; m += 4) {
            const int d1 = d - 1 < 0 ? d - 1 + nx : d - 1;
            const int d2 = d1 - 1 < 0 ? d1 - 1 + nx : d1 - 1;
            const int d3 = d2 - 1 < 0 ? d2 - 1 + nx : d2 - 1;
            s0 += sc[m] * sb[d];
            s1 += sc[m + 1] * sb[d1];
            s2 += sc[m + 2] * sb[d2];
            s3 += sc[m + 3] * sb[d3];
            d = d3 - 1 < 0 ? d3 - 1 + nx : d3 - 1;
        }
        for (; m < m1; ++m) {
            s0 += sc[m] * sb[d];
            d = d - 1 < 0 ? d - 1 + nx : d - 1;
        }
    }
    part[wave][lane] = (s0 + s1) + (s2 + s3);
    __syncthreads();
    if (wave == 0 && i < nx) {
        double s = part[0][lane];
        for (int w = 1; w < NT / 64; ++w) s += part[w][lane];
        a.work[nx + i] = s;
    }
}

// one workgroup: h1 = phi - mean phi and ||A phi + (n - mean n) q||
__global__ __launch_bounds__(PT) void poisson_post_kernel(PoiArgs a)
{
    extern __shared__ double sm[];
    __shared__ double red[PT / 64 + 1];
    poi_instance(a);
    const double hx2_inv = a.inst[blockIdx.y].hx2_inv;
    const int nx = a.nx;
    const double *wphi = a.work + nx, *wn = a.work + 2 * nx;
    const double nmean = a.work[3 * nx];
    double part = 0.0;
    for (int i = threadIdx.x; i < nx; i += PT) {
        sm[i] = wphi[i];
        part += wphi[i];
    }
    const double phiave = block_sum_big(part, red) / nx;
    part = 0.0;
    for (int i = threadIdx.x; i < nx; i += PT) {
        if (a.phi) a.phi[i] = sm[i];
        if (a.h1) a.h1[i] = sm[i] - phiave;
        const double r = lap(sm, i, nx, a.laplace, hx2_inv) + (wn[i] - nmean) * a.charge;
        part += r * r;
    }
    const double rr = block_sum_big(part, red);
    if (threadIdx.x == 0 && a.pres) *a.pres = sqrt(rr);
}

// y = A x (+ (n - mean n) q when n != null)
__global__ __launch_bounds__(PT) void poisson_mult_kernel(const double *x, const double *n, double *y, int nx,
                                                          int laplace, const InstConst *inst, double charge)
{
    extern __shared__ double sm[];
    __shared__ double red[PT / 64 + 1];
    const double hx2_inv = inst[blockIdx.y].hx2_inv;
    x += (size_t)blockIdx.y * nx;
    y += (size_t)blockIdx.y * nx;
    if (n) n += (size_t)blockIdx.y * nx;
    double part = 0.0;
    for (int i = threadIdx.x; i < nx; i += PT) {
        sm[i] = x[i];
        if (n) part += n[i];
    }
    const double nmean = block_sum_big(part, red) / nx;
    for (int i = threadIdx.x; i < nx; i += PT) {
        double v = lap(sm, i, nx, laplace, hx2_inv);
        if (n) v = v + (n[i] - nmean) * charge;
        y[i] = v;
    }
}

__global__ __launch_bounds__(PT) void pot_to_ham_kernel(const double *phi, double *h1, int nx)
{
    __shared__ double red[PT / 64 + 1];
    phi += (size_t)blockIdx.y * nx;
    h1 += (size_t)blockIdx.y * nx;
    double part = 0.0;
    for (int i = threadIdx.x; i < nx; i += PT) part += phi[i];
    const double ave = block_sum_big(part, red) / nx;
    for (int i = threadIdx.x; i < nx; i += PT) h1[i] = phi[i] - ave;
}

struct InvArgs {
    const double *f, *h0, *h1, *h2, *phi;
    int nx, nv;
    double hv, charge;
    const InstConst *inst;
    double *partial;      // [gridDim.x][5] per instance, pstride apart
    int64_t pstride;
    double *out;          // 6 doubles per instance
};

__device__ __forceinline__ void inv_instance(InvArgs &a)
{
    const size_t b = blockIdx.y;
    a.f += b * a.nx * a.nv;
    a.h1 += b * a.nx;
    a.h2 += b * a.nx;
    a.phi += b * a.nx;
    a.partial += b * a.pstride;
    a.out += b * 6;
}

// Partial sums per workgroup.  On the periodic x-axis each cell average of
// the mass, (f_ij + f_i+1,j + f_i,j+1 + f_i+1,j+1) over rows j < nv - 1, counts
// every f of rows 0..nv-2 twice and of rows 1..nv-1 twice, so one read of f
// serves all five sums (HBM-bound: 8 N bytes).  Column and row advance with the
// grid stride instead of being divided out.  16.1 us at 1000 x 2001 with the
// four neighbours read and a 64-bit division a point.
__global__ __launch_bounds__(NT) void invariants_kernel(InvArgs a)
{
    inv_instance(a);
    __shared__ double red[5][NT / 64];
    double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
    const unsigned nx = a.nx, nv = a.nv, N = nx * nv;
    const unsigned stride = gridDim.x * NT, dj = stride / nx, di = stride - dj * nx;
    unsigned e = blockIdx.x * NT + threadIdx.x;
    unsigned j = e / nx, i = e - j * nx;
    for (; e < N; e += stride) {
        const double fv = a.f[e];
        const double w = (j < nv - 1 ? 2.0 : 0.0) + (j > 0 ? 2.0 : 0.0);
        s[0] += w * fv;
        s[1] += j < nv - 1 ? fv * fv : 0.0;
        s[2] += fv * a.h0[j];
        s[3] += fv * a.h1[i];
        s[4] += fv * a.h2[i];
        j += dj;
        i += di;
        if (i >= nx) {
            i -= nx;
            ++j;
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int q = 0; q < 5; ++q) {
        const double v = wave_sum(s[q]);
        if (lane == 0) red[q][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x < 5) {
        double v = 0.0;
        for (int w = 0; w < NT / 64; ++w) v += red[threadIdx.x][w];
        a.partial[(size_t)blockIdx.x * 5 + threadIdx.x] = v;
    }
}

// one workgroup: sums the per-block partials and the field energy, thread
// shares first, then over the wavefronts (fixed order).  The sums by one thread
// (256 partials and nx potential differences in a row) took 68 us at nx = 1000.
__global__ __launch_bounds__(NT) void invariants_finish_kernel(InvArgs a, int nb)
{
    __shared__ double red[6][NT / 64];
    inv_instance(a);
    const double hx = a.inst[blockIdx.y].hx;
    double t6[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int b = threadIdx.x; b < nb; b += NT)
        for (int q = 0; q < 5; ++q) t6[q] += a.partial[(size_t)b * 5 + q];
    for (int i = threadIdx.x; i < a.nx; i += NT) {
        const double d = a.phi[i + 1 < a.nx ? i + 1 : 0] - a.phi[i];
        t6[5] += d * d;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int q = 0; q < 6; ++q) {
        const double v = wave_sum(t6[q]);
        if (lane == 0) red[q][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    double t[6];
    for (int q = 0; q < 6; ++q) {
        t[q] = red[q][0];
        for (int w = 1; w < NT / 64; ++w) t[q] += red[q][w];
    }
    const double hxhv = hx * a.hv;
    const double mass = t[0] * 0.25 * hx * a.hv;
    const double l2 = hxhv * t[1];
    const double ekin = t[2] * hx * a.hv;
    const double epot = (t[3] + t[4]) * hx * a.hv;
    a.out[0] = mass;
    a.out[1] = l2;
    a.out[2] = ekin + 0.5 * epot;
    a.out[3] = ekin;
    a.out[4] = epot;
    a.out[5] = 0.5 * a.charge * t[5] / hx;
}

}  // namespace

namespace {

template <int MOM>
void column_launch(vv_ctx *c, const double *f, int nch, int64_t ostride, double scale, double *out0, double *out1)
{
    const int nx = c->p.nx, nv = c->p.nv;
    const int rows = (nv + nch - 1) / nch;
    hipLaunchKernelGGL(column_kernel<MOM>, dim3((nx + 63) / 64, nch, c->B), dim3(64 * CW), 0, c->stream, f, c->vgrid,
                       nx, nv, rows, ostride, scale, out0, out1);
}

void column_finish(vv_ctx *c, const double *part1, double *out0, double *out1)
{
    const int nx = c->p.nx;
    hipLaunchKernelGGL(column_finish_kernel, dim3((nx + NT - 1) / NT, c->B, out1 != nullptr ? 2 : 1), dim3(NT), 0,
                       c->stream, c->npart, part1, column_chunks(c->p.nv), nx, (int64_t)DCH * nx, c->p.hv, out0,
                       out1);
}

}  // namespace

hipError_t launch_density_partial(vv_ctx *c, const double *f, double *npart)
{
    column_launch<0>(c, f, column_chunks(c->p.nv), (int64_t)DCH * c->p.nx, 1.0, npart != nullptr ? npart : c->npart, nullptr);
    return hipGetLastError();
}

hipError_t launch_density(vv_ctx *c, const double *f, double *n)
{
    if (sum_chunks(c->p.nv) == 1) {
        column_launch<0>(c, f, 1, c->p.nx, c->p.hv, n, nullptr);
        return hipGetLastError();
    }
    const hipError_t e = launch_density_partial(c, f, nullptr);
    if (e != hipSuccess) return e;
    column_finish(c, nullptr, n, nullptr);
    return hipGetLastError();
}

hipError_t launch_velocity_moments(vv_ctx *c, const double *f, double *u, double *e)
{
    if (sum_chunks(c->p.nv) == 1) {
        column_launch<1>(c, f, 1, c->p.nx, c->p.hv, u, e);
        return hipGetLastError();
    }
    double *part1 = c->npart + (size_t)(DCH / 2) * c->p.nx;
    column_launch<1>(c, f, column_chunks(c->p.nv), (int64_t)DCH * c->p.nx, 1.0, c->npart, part1);
    column_finish(c, part1, u, e);
    return hipGetLastError();
}

hipError_t launch_poisson(vv_ctx *c, const double *n_in, double *n_out, double *phi, double *h1, double *pres,
                          int from_part, const double *npart, double *work, int pres_stride, int nch,
                          int64_t npstride)
{
    const int nx = c->p.nx;
    PoiArgs a{nx, c->p.laplace, from_part, nch > 0 ? nch : column_chunks(c->p.nv), 0,
              nch > 0 ? npstride : (int64_t)DCH * nx, c->p.hv, c->p.charge, c->inst,
              from_part ? (npart != nullptr ? npart : c->npart) : nullptr, n_in, c->pinv, c->plam, c->twiddle,
              work != nullptr ? work : c->pwork, n_out, phi, h1, pres, pres_stride};
    if (c->plam != nullptr) {
        while ((1 << a.logn) < nx) ++a.logn;
        hipLaunchKernelGGL(poisson_kernel<true>, dim3(1, c->B), dim3(PT),
                           (nx <= kPoissonTw ? 2 : 1) * nx * sizeof(double2), c->stream, a);
        return hipGetLastError();
    }
    if (nx <= kPoissonOne) {
        hipLaunchKernelGGL(poisson_kernel<false>, dim3(1, c->B), dim3(PT), 2 * nx * sizeof(double), c->stream, a);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(poisson_prep_kernel, dim3(1, c->B), dim3(PT), 0, c->stream, a);
    hipLaunchKernelGGL(poisson_conv_kernel, dim3((nx + CONV_OUT - 1) / CONV_OUT, c->B), dim3(NT),
                       2 * nx * sizeof(double), c->stream, a);
    hipLaunchKernelGGL(poisson_post_kernel, dim3(1, c->B), dim3(PT), nx * sizeof(double), c->stream, a);
    return hipGetLastError();
}

hipError_t launch_poisson_mult(vv_ctx *c, const double *x, const double *n, double *y)
{
    const size_t lds = (size_t)c->p.nx * sizeof(double);
    hipLaunchKernelGGL(poisson_mult_kernel, dim3(1, c->B), dim3(PT), lds, c->stream, x, n, y, c->p.nx, c->p.laplace,
                       c->inst, c->p.charge);
    return hipGetLastError();
}

hipError_t launch_pot_to_ham(vv_ctx *c, const double *phi, double *h1)
{
    hipLaunchKernelGGL(pot_to_ham_kernel, dim3(1, c->B), dim3(PT), 0, c->stream, phi, h1, c->p.nx);
    return hipGetLastError();
}

hipError_t launch_invariants(vv_ctx *c, const double *f, const double *h0, const double *h1, const double *h2,
                             const double *phi, double *out_dev)
{
    InvArgs a{f, h0, h1, h2, phi, c->p.nx, c->p.nv, c->p.hv, c->p.charge, c->inst, c->partial, c->part_stride,
              out_dev};
    hipLaunchKernelGGL(invariants_kernel, dim3(kReduceBlocks, c->B), dim3(NT), 0, c->stream, a);
    hipLaunchKernelGGL(invariants_finish_kernel, dim3(1, c->B), dim3(NT), 0, c->stream, a, kReduceBlocks);
    return hipGetLastError();
}

}  // namespace vv
