// Internal declarations shared by the HIP translation units of libvv1d.so.
#pragma once

#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/vv1d.h"
#include "tile_index.h"

namespace vv {

constexpr int kMaxRestart = 64;     // GMRES restart limit (basis of restart+1 vectors)
constexpr int kGraphSteps = 6;      // Arnoldi steps of a part of the captured cycle
constexpr int kGraphParts = (kMaxRestart + kGraphSteps - 1) / kGraphSteps;
constexpr int kMaxNx = 4096;        // largest x size
constexpr int kMaxNv = 4096;
constexpr int kReduceBlocks = 512;  // fixed block count of N-sized reductions
constexpr int kDensityChunks = 64;  // rows of nx partial sums kept per instance for the column sums

// Host-visible part of the GMRES state; copied to pinned host memory at the end
// of a cycle.
struct GmresStatus {
    int32_t it;        // iterations in the current cycle
    int32_t its;       // total iterations
    int32_t reason;    // KSP converged reason (0 = iterating)
    int32_t done;      // current cycle finished: every Krylov kernel returns at once
    int32_t active;    // instance takes part in this solve (batched contexts)
    int32_t pad;
    double res;        // current residual estimate
    double rnorm0;     // norm of the right-hand side
};

// Per-instance grid constants (a batched context holds instances that share
// nx, nv, v-grid and dt but not the x-period, so hx differs).
struct InstConst {
    double hx, hx_inv, hx2_inv;
    double af1, af2;   // Arakawa factors hx^-1 hv^-1 / 12, / 24
    double afpc;       // preconditioner band factor 0.5 hx^-1 hv^-1 / 12
};

// Device-resident GMRES state, read by every Krylov kernel.  Written by one
// workgroup a launch and instance: the Hessenberg update or cycle start
// (gmres_dev.h; in a launch of its own or the first workgroup of the launch that
// carries it), the CGS update (its column of hh) and the solution update (a
// singular triangle's reason, over).
struct GmresState {
    GmresStatus st;
    double hh[(kMaxRestart + 1) * kMaxRestart];  // rotated Hessenberg, column it at hh[it*(kMaxRestart+1)]
    double cc[kMaxRestart];
    double ss[kMaxRestart];
    double grs[kMaxRestart + 1];
    double scale[kMaxRestart + 1];   // v_j = scale[j] * V_j (V_j stored unnormalised)
    double ttol, rtol, atol, dtol, haptol;
    int32_t max_it;
    int32_t max_k;
    int32_t skip[2];                 // done as of update it - 1, at it & 1: for the launch that carries update it
    int32_t over;                    // the solve has ended, as of the last solution update: for a restart's launch
    int32_t pad;
};

// Tolerances and limits a solve starts with, and which instances take part
// (null: all).
struct SolveStart {
    const int32_t *active;
    double rtol, atol, dtol;
    int32_t max_it, max_k;
};

// The Hessenberg update of Arnoldi step `it` (gmres_dev.h), or, with start, the
// start of a cycle on V_0 (1: a restart; 2: the first of a solve, whose state
// `init` fills): its norm partials
// (instance b at part + b pstride, nb of them; nb = 0: no update is due), the
// states, and where the host polls for the report (one word per instance;
// null: nobody does) and its number.
struct HessArgs {
    const double *part;
    int64_t pstride;
    int nb, it;
    GmresState *g;
    uint32_t *hout;
    uint32_t seq;
    int start;
    SolveStart init;
};

// Plan of the mixed-radix line transform (rows.hip): stage s has radix r[s]
// after sub-transforms of length ns[s]; nr = n / r, step = n / (ns r); mn, mnr,
// mns: reciprocals of n, nr, ns for division by multiplication.
constexpr int kDftStages = 11;
struct DftPlan {
    int n, stages;
    int r[kDftStages], ns[kDftStages], nr[kDftStages], step[kDftStages];
    uint32_t mn, mnr[kDftStages], mns[kDftStages];
};

// The collision operator a Jacobian-vector product adds (dissipation.hip).
struct CollTerm {
    const double *n, *U, *a;   // x-vectors
    double drag_fac, diff_fac;
    int e;                     // collE
};

constexpr int kRowsNx = 2048;   // longest x of the row-block kernels (rows.hip)

}  // namespace vv

struct vv_ctx {
    vv_params p;
    hipStream_t stream;
    int B;              // instances (1 unless created batched); instance b of every
                        // per-instance buffer lives at base + b * stride
    vv::InstConst *inst;        // device, B entries
    std::vector<vv::InstConst> inst_host;
    int32_t *active;            // device, B flags: instance takes part in the next solve
    int64_t N;          // nx * nv (per instance)
    int64_t vs;         // element stride of the Krylov basis vectors: B N rounded up to a multiple of 4
    // transform geometry of the tensor-product preconditioner: the real FFT
    // has length fft_n over fft_rows rows and nmodes = fft_n/2 + 1 modes, each
    // mode a tridiagonal system of length fft_rows.  kinetic: FFT along x
    // (fft_n = nx, fft_rows = nv); potential: along v on the transposed field
    // (fft_n = nv, fft_rows = nx)
    int nmodes;         // fft_n/2 + 1
    int logn;           // log2(fft_n) when fft_n is a power of two (FFT kernels); else a direct DFT
    int fft_n, fft_rows;
    vv::DftPlan dft;    // fft_n no power of two and <= kRowsNx: the line transform's plan (else n = 0); see dft_rows
    int64_t coef_stride;        // instance stride of gm/g0/gp (0: shared)
    double cf_lo, cf_mid, cf_hi;  // band constants: kinetic 0.5/1.0/0.5, potential 1.0/2.0/1.0
    double *tb;                 // potential: the transposed field (B N doubles)
    // grid-derived constants (x-dependent ones per instance in inst)
    double ht_inv, hv_inv;
    // Hamiltonian factors (device, ctx-owned copies): h0 shared, h1*/h2* per instance
    double *h0, *h1p, *h1h, *h2p, *h2h;
    // preconditioner data (device)
    double2 *eigen;     // nmodes used (mode k = 0..fft_n/2)
    double *lu_gm, *lu_gp;  // kinetic gm (0 at row 0) and gp (0 from row nv-1 on) in the pivots' order
    double *gm, *g0, *gp;   // per-row real factors of the bands (kinetic: of v; potential: phi differences per instance)
    double *vgrid;          // v_j (velocity moments)
    double2 *twiddle;   // exp(-2 pi i m / fft_n), m = 0..fft_n-1
    float2 *twiddle32;  // the same, rounded to float (FP32 preconditioner)
    double2 *spec;      // complex spectrum per instance, nmodes rows of fft_rows, spec_pitch apart
    // kinetic preconditioner: reciprocal LU pivots 1/u_j of every T_k, same
    // layout as the spectrum (FP64 at creation; FP32 on first FP32 use);
    // null for the potential preconditioner (its bands change every step)
    double2 *lu64;
    float2 *lu32;
    // Poisson
    double *pinv;       // first row of the mean-free circulant inverse (nx per instance); null with plam
    double *plam;       // nx a power of two: the inverse symbol over nx (nx per instance), for the FFT form
    double *pwork;      // Poisson scratch (3*nx + 1 per instance)
    // work vectors (N)
    double *X;          // bracket / residual output before P^-1
    double *rhs;        // SNES right-hand side P^-1 F
    double *D;          // Newton update
    double *basis;      // (restart+1) vectors of B*N: V_j of instance b at basis + (j*B + b)*N
    // mixed precision (allocated on first use)
    float *basis32;     // FP32 basis, same layout
    double *R;          // FP64 true residual of the refinement loop
    double *w64, *d64;  // FP32 cycle with a dissipation term: the Krylov vector widened, the term in FP64
    // reductions
    double *partial;    // per instance: part_stride doubles
    int64_t part_stride;
    double *dscalar;    // device scalars, 16 per instance
    double *npart;      // density partial sums, 64 nx per instance
    vv::GmresState *gs;             // B states
    vv::GmresStatus *host_status;   // pinned, B statuses
    vv::GmresStatus *host_status_dev;   // the same memory as the device addresses it
    uint32_t *host_poll;            // pinned, 2 slots of B words: reports of the Hessenberg updates
    uint32_t *host_poll_dev;        // the same memory as the device addresses it
    uint32_t *report_out;           // set for one launch: where the Hessenberg update reports
    uint32_t report_seq;            // number of the last report asked for (below kGraphSeq)
    int pend_it, pend_nb;           // Arnoldi step whose Hessenberg update is due (-1: none), its norm partials
    int pend_start;                 // a cycle start is due instead (HessArgs::start; 0: none)
    vv::SolveStart start;           // what a first cycle starts with
    double *host_scalars;           // pinned staging of device scalars
    double *host_scalars_dev;       // the same memory as the device addresses it
    int32_t *host_active;           // pinned staging of the instance mask
    int32_t *host_active_dev;       // the same memory as the device addresses it
    // profiling (per-kernel HIP event pairs)
    int prof;           // bit k set: time kernel kind k
    void *prof_state;
    hipEvent_t prof_a, prof_b;   // events of the next main-kernel launch (null: none)
    // linearised / adjoint operators (scratch allocated on first use):
    // operator of the GMRES cycle (0: P^-1 J of the Picard step; 1: P^-T A^T,
    // the transposed full linearisation), the midpoint state f_bar of its
    // field coupling (null: no coupling)
    int op_mode;
    const double *op_fbar;
    double *T2;         // B*N
    double *xs;         // 4 regions of B*nx: n | phi | h1 | spare
    // launch-shape tuning (0: built-in heuristic): v-rows per FFT workgroup,
    // 16-byte vectors per thread of the CGS kernels
    int tune_fft_rows, tune_cgs_ept;
    // kernel fusion (default on): the Arnoldi step's irFFT and CGS dots in
    // one launch where the geometry allows; results are bit-identical
    bool fuse;
    // captured first GMRES cycle of SNESSolve_KSPONLY (graph replay mode), in
    // parts of kGraphSteps Arnoldi steps; the norm partials of a step
    bool use_graph, capturing;
    hipGraphExec_t graph_exec[vv::kGraphParts];
    int graph_nb;
    const double *graph_f, *graph_fh;
    double graph_kp[4];
    // dissipation term (VV_DISSIPATION_*) and its parameters; moment vectors
    // are caller-owned device x-vectors: N, U, E, A current then history
    int diss_kind;
    double coll_freq, coll_diff, coll_drag, hv2_inv;
    const double *mom[8];
    double *fave;       // .5 fh + .5 f of the last residual (double brackets)
    double *db1;        // {fave, H_ave}, valid while db1_valid
    double *db2;        // scratch bracket of the Jacobian
    bool db1_valid;
    double *ex;         // explicit steppers: H | t1 | t2 | t3 | t4 | stage (6 N)
    int64_t dev_bytes;  // device memory the context has allocated so far
    double *static_scratch;   // device address of this device's copy of the allocation-free
                              // entry point's file-scope scratch array
    std::string err;
};

namespace vv {

// ---- launchers -------------------------------------------------------------
// bracket.hip
// part: per-workgroup sums of y^2 (residual_blocks of them, instances part_stride apart) when not null
hipError_t launch_residual(vv_ctx *c, const double *f, const double *fh, double *y, double *part = nullptr);
int residual_blocks(const vv_ctx *c);
hipError_t launch_jacobian_plain(vv_ctx *c, const double *u, double *y);
// the solver's own F(f) and J u (H split into row and column coefficients; the
// two above keep the reference's operation order)
hipError_t launch_residual_sep(vv_ctx *c, const double *f, const double *fh, double *y);
hipError_t launch_jacobian(vv_ctx *c, const double *u, const double *uscale, double *y);
hipError_t launch_bracket_add(vv_ctx *c, const double *x, double *y, double factor);
hipError_t launch_jacobian32(vv_ctx *c, const float *u, const double *uscale, float *y);
hipError_t launch_widen(vv_ctx *c, const float *x, double *y);                  // y = (double) x
hipError_t launch_narrow_add(vv_ctx *c, float *y, const double *d);           // y = (float)(y + d)
// y = alpha u + factor {u~, H} on all rows (u~: u on rows 2..nv-3, else 0);
// H = h2d (2D) or hxv (x only) when given, else H_ave
hipError_t launch_bracket_t(vv_ctx *c, const double *u, const double *uscale, const double *h2d, const double *hxv,
                            double *y, double alpha, double factor);
// y = alpha u + factor {u~, H_ave} on all rows and the column sums of {u~, g} over
// band_rows(nv) bands of rows; takes the due Hessenberg update when uscale is given
int band_rows(int nv);
hipError_t launch_bracket_pair(vv_ctx *c, const double *u, const double *uscale, const double *g, double *y,
                               double alpha, double factor, double *csum, int64_t cstride);
// y += factor {x, H} on rows 2..nv-3, H = h2d / hxv / H_ave as above
hipError_t launch_bracket_gen(vv_ctx *c, const double *x, const double *h2d, const double *hxv, double *y,
                              double factor);
// y (+)= factor {s x, H} on rows 2..nv-3 (store: y = 0 + ..., other rows 0),
// s = *xscale when given, H = h2d or H_ave
hipError_t launch_bracket_acc(vv_ctx *c, const double *x, const double *xscale, const double *h2d, double *y,
                              double factor, bool store, const int32_t *done);
// dissipation.hip: y += C(s f) of the context's collision operator; a = n n / (n e - u u)
hipError_t launch_collision(vv_ctx *c, const double *f, const double *fscale, double *y, const double *n,
                            const double *U, const double *a, double factor, const int32_t *done);
hipError_t launch_collision_factor(vv_ctx *c, const double *n, const double *u, const double *e, double *a);
hipError_t launch_average(vv_ctx *c, const double *f, const double *fh, double *out);   // .5 fh + .5 f
// explicit.hip: H = h0 | h1 + h2 | (h0 + h1) + h2 as a 2D field; stage combinations
hipError_t launch_compose_h(vv_ctx *c, const double *h0, const double *h1, const double *h2, double *H);
hipError_t launch_stage(vv_ctx *c, const double *x, const double *t, double s, double *out);   // x + s t
hipError_t launch_rk18_stage3(vv_ctx *c, const double *x, const double *t1, const double *t2, double cc, double s,
                              double *out);
hipError_t launch_rk18_stage4(vv_ctx *c, const double *x, const double *t1, const double *t2, const double *t3,
                              double s, double *out);
hipError_t launch_rk4_end(vv_ctx *c, bool three_eighths, double *x, const double *t1, const double *t2,
                          const double *t3, const double *t4, double s);
bool collision_term(vv_ctx *c, const double *n, const double *U, const double *a, double factor, CollTerm *t);
// rows.hip: row blocks of the kinetic form (where: rows_apply);
// J u (with the previous step's Hessenberg update, and the collision term when
// given) or F(f) formed and transformed in one launch, and the irFFT into
// basis[col+1] with its CGS dots in row_inv_blocks partial rows
DftPlan make_dft_plan(int n);
// whether rows of an fft_n that is no power of two can gain by the plan: more than
// one stage (of one the direct real DFT takes half the arithmetic: P^-1 at 1999 x
// 2048 4.4 ms with the stage, 3.1 without; 211 x 2048 67.6 us, 59.2)
inline bool dft_rows(const vv_ctx *c) { return c->dft.stages > 1; }
bool rows_apply(const vv_ctx *c);
int row_inv_blocks(const vv_ctx *c);
hipError_t launch_row_jac(vv_ctx *c, const double *u, const double *uscale, const CollTerm *coll, double2 *spec,
                          const int32_t *done);
hipError_t launch_row_jac32(vv_ctx *c, const float *u, const double *uscale, float2 *spec, const int32_t *done);
hipError_t launch_row_res(vv_ctx *c, const double *f, const double *fh, double2 *spec);
hipError_t launch_row_rfft(vv_ctx *c, const double *x, double2 *spec, const int32_t *done, const double *add,
                           double gamma);
hipError_t launch_row_rfft32(vv_ctx *c, const float *x, float2 *spec, const int32_t *done);
hipError_t launch_row_irfft(vv_ctx *c, const double2 *spec, double *y, const int32_t *done);
hipError_t launch_row_irfft32(vv_ctx *c, const float2 *spec, float *y, const int32_t *done);
// the irFFT into V_0 with its norm partials (row_inv_blocks of them)
hipError_t launch_row_inv_start(vv_ctx *c, const double2 *spec);
hipError_t launch_row_inv(vv_ctx *c, const double2 *spec, int col, const int32_t *done);
hipError_t launch_row_inv32(vv_ctx *c, const float2 *spec, int col, const int32_t *done);
// spectral.hip
int fft_blocks(vv_ctx *c);
int fft_rows_of(const vv_ctx *c);
// (rows x + gamma add with an x-only field `add`, B nx)
hipError_t launch_rfft(vv_ctx *c, const double *x, double2 *spec, const int32_t *done, const double *add = nullptr,
                       double gamma = 0.0);
// J u (u times its optional device scale) and its rFFT in one launch, the
// Jacobian never stored; jac_rfft_rows: the rows per workgroup where the
// fused kernel applies to the context (the kinetic form with a power-of-two
// nx in [256, 1024]), else 0.  No dissipation terms (the caller checks).
int jac_rfft_rows(const vv_ctx *c);
hipError_t launch_jac_rfft(vv_ctx *c, const double *u, const double *uscale, double2 *spec, const int32_t *done);
hipError_t launch_jac_rfft32(vv_ctx *c, const float *u, const double *uscale, float2 *spec, const int32_t *done);
hipError_t launch_tridiag_k(vv_ctx *c, double2 *spec, const int32_t *done);
hipError_t launch_irfft(vv_ctx *c, const double2 *spec, double *y, const int32_t *done);
hipError_t launch_tridiag_t(vv_ctx *c, double2 *spec, const int32_t *done);   // T_k^-H (transposed P)
hipError_t launch_rfft32(vv_ctx *c, const float *x, float2 *spec, const int32_t *done);
hipError_t launch_tridiag32(vv_ctx *c, float2 *spec, const int32_t *done);
hipError_t launch_irfft32(vv_ctx *c, const float2 *spec, float *y, const int32_t *done);
// irFFT into basis[col+1] fused with its CGS dots against basis[0..col]
// (per-slice partials, as launch_mdot); irfft_mdot_rows: the partial rows it
// writes (its grid), 0 where the fused kernel does not apply
int irfft_mdot_rows(const vv_ctx *c, bool fp32);
// rows per thread of the LU tridiagonal solve, and the pivots it stores per
// mode (chunk-interleaved, >= nv)
int lu_threads(int nv);
int lu_rows(int nv);
int lu_pivots_per_mode(int nv);
hipError_t launch_irfft_mdot(vv_ctx *c, const double2 *spec, int col, const int32_t *done);
hipError_t launch_irfft_start(vv_ctx *c, const double2 *spec);   // into V_0, with its norm partials per slice
hipError_t launch_irfft_mdot32(vv_ctx *c, const float2 *spec, int col, const int32_t *done);
// potential preconditioner: field (nv rows of nx) <-> transposed (nx rows of nv)
// reciprocal LU pivots of the kinetic T_k into rp64 (FP64) and / or rp32 (rounded)
hipError_t launch_tridiag_factor(vv_ctx *c, double2 *rp64, float2 *rp32);
hipError_t launch_transpose(vv_ctx *c, const double *in, double *out, bool back, const int32_t *done);
hipError_t launch_transpose32(vv_ctx *c, const float *in, float *out, bool back, const int32_t *done);
// the potential form's transforms straight on the field's columns, where they
// apply to the field f (its alignment; an even nx, nv a power of two)
bool potential_cols(const vv_ctx *c, const double *f);
bool potential_cols32(const vv_ctx *c, const float *f);
hipError_t launch_rfft_cols(vv_ctx *c, const double *x, double2 *spec, const int32_t *done);
hipError_t launch_irfft_cols(vv_ctx *c, const double2 *spec, double *y, const int32_t *done);
hipError_t launch_rfft_cols32(vv_ctx *c, const float *x, float2 *spec, const int32_t *done);
hipError_t launch_irfft_cols32(vv_ctx *c, const float2 *spec, float *y, const int32_t *done);
hipError_t launch_potential_bands(vv_ctx *c, const double *phi);
// krylov.hip
hipError_t launch_gmres_init(vv_ctx *c, double rtol, double atol, double dtol, int max_it);
// V_0 for a cycle start, with its norm partials: copied from b, rounded from r,
// or in place; the start is then due as a Hessenberg update is (take_update).
// A first cycle starts with c->start.
double *norm_partials(vv_ctx *c);                         // where they go (instances part_stride apart)
hipError_t launch_start(vv_ctx *c, const double *b, bool first);        // V_0 = b
hipError_t launch_start32(vv_ctx *c, const double *r, bool first);      // V_0 = (float) r
hipError_t launch_restart(vv_ctx *c, const double *b);    // V_0 = b - V_0
int cgs_blocks_max(int64_t N);                            // partial rows the CGS kernels may use
int cgs_ept(const vv_ctx *c, int64_t nvv);              // 16-byte vectors per thread of a CGS launch
hipError_t launch_mdot(vv_ctx *c, int col);               // CGS dots of basis[col+1] vs 0..col
// CGS update of basis[it+1]; dot_rows: partial rows of the dots launch before
// it (0: launch_mdot's grid).  The step's Hessenberg update is then due: the
// next step's fused first kernel takes it along (take_update), anything else
// runs it first (launch_update; nothing when none is due)
hipError_t launch_maxpy_norm(vv_ctx *c, int it, int dot_rows = 0);
HessArgs take_update(vv_ctx *c);
hipError_t launch_update(vv_ctx *c);
// x (FP64) = V y (store) or x += V y, y from the triangular system; with f:
// f -= V y instead of the store where the solve converged; hout: the statuses
// to host memory
hipError_t launch_build_solution(vv_ctx *c, double *x, double *f, bool store, GmresStatus *hout);
hipError_t launch_mdot32(vv_ctx *c, int col);
hipError_t launch_maxpy_norm32(vv_ctx *c, int it, int dot_rows = 0);
hipError_t launch_build_solution32(vv_ctx *c, double *x, double *f, bool store, GmresStatus *hout);
hipError_t launch_rsub(vv_ctx *c, const double *b, double *y);   // y = b - y (B fields)
// ||x_b|| of the B fields (x null: from nb partials already in c->partial) to
// host[b], and pres[16 b] to host[B + b] when pres is given
hipError_t launch_norms(vv_ctx *c, const double *x, int nb, const double *pres, double *host);
hipError_t launch_norm2(vv_ctx *c, const double *x, int64_t n, double *out_dev);
hipError_t launch_dot(vv_ctx *c, const double *x, const double *y, int64_t n, double *out_dev);
hipError_t launch_axpy(vv_ctx *c, double alpha, const double *x, double *y, int64_t n);
hipError_t launch_axpy_cond(vv_ctx *c, double alpha, const double *x, double *y);  // per instance, if reason > 0
hipError_t launch_copy(vv_ctx *c, const double *x, double *y, int64_t n);
hipError_t launch_zero(vv_ctx *c, double *y, int64_t n);
hipError_t launch_xadd(vv_ctx *c, double *y, const double *w, double alpha);  // y[b][j][i] += alpha w[b][i]
// moments.hip
// density partials (DCH x nx per instance) into npart, or the context's own
// buffer when npart is null
hipError_t launch_density_partial(vv_ctx *c, const double *f, double *npart);
hipError_t launch_density(vv_ctx *c, const double *f, double *n);
hipError_t launch_velocity_moments(vv_ctx *c, const double *f, double *u, double *e);
// Poisson pipeline; npart / work (3 nx + 1 per instance) default to the
// context's buffers when null (nch partials a column, npstride apart per
// instance, when given); the residual norm of instance b goes to
// pres[b * pres_stride]
hipError_t launch_poisson(vv_ctx *c, const double *n_in, double *n_out, double *phi, double *h1, double *pres,
                          int from_part, const double *npart = nullptr, double *work = nullptr,
                          int pres_stride = 16, int nch = 0, int64_t npstride = 0);
hipError_t launch_poisson_mult(vv_ctx *c, const double *x, const double *n, double *y);
hipError_t launch_pot_to_ham(vv_ctx *c, const double *phi, double *h1);
hipError_t launch_invariants(vv_ctx *c, const double *f, const double *h0, const double *h1,
                             const double *h2, const double *phi, double *out_dev);

// Launch a timed kernel: when the profiler armed c->prof_a / c->prof_b, the
// events are attached to this kernel's own dispatch packet (start / end
// timestamps of the kernel, as a kernel trace reports them).
template <typename K, typename... Args>
inline void launch_timed(vv_ctx *c, K kernel, dim3 grid, dim3 block, uint32_t shmem, Args... args)
{
    if (c->prof_a != nullptr) {
        hipExtLaunchKernelGGL(kernel, grid, block, shmem, c->stream, c->prof_a, c->prof_b, 0u, args...);
        c->prof_a = c->prof_b = nullptr;
    } else {
        hipLaunchKernelGGL(kernel, grid, block, shmem, c->stream, args...);
    }
}

// elements from mode to mode of a spectrum: an odd multiple of 256 bytes (FP64).
// A row block stores (loads) a short segment of every mode; with the modes a power of two
// apart they fall on few L2 channels and memory stacks.  rFFT 2048 x 4096 44.6 ->
// 41.6 us, 2048 x 1024 12.2 -> 11.6; J u + rFFT 1024 x 2048 17.5 -> 17.2; the row
// blocks of 201 x 401 10.4 -> 10.0 and 9.1 -> 8.8.
inline int64_t spec_pitch(const vv_ctx *c) { return (int64_t)(((c->fft_rows + 15) / 16) | 1) * 16; }

// element stride between the spectra of consecutive instances
inline int64_t spec_stride(const vv_ctx *c) { return (int64_t)c->nmodes * spec_pitch(c); }

}  // namespace vv
