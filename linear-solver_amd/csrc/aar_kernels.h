// aar_kernels.h -- kernel argument blocks and launchers of libaar_hip.
#pragma once

#include "aar_common.h"

namespace aar {

enum class SMode : int {
    MATVEC = 0,    // y = a*Lap(x) + sigma*x                      (system.c:189-205)
    AAR_TRUE = 1,  // r = b - A x; g = r/diag (T or FP32 out); ||r||^2 (AAR.c:80-82,119-123)
    RESID = 2,     // r = b - A x (+ optional fp32 copy), ||r||^2
    PGR_STEP = 3,  // Ax = A x; x_next = x + omega (b - Ax)/diag; ||b - Ax||^2 (PGR.c:92-103)
    CG_Q = 4,      // q = A d; d.q                                (CG.c:94-100)
    CG_RESID = 5,  // r = b - A x; r.s, r.r                        (CG.c:65-84,112-137)
    AAR_REC = 7,   // g' = g - (omega/diag) A g: the residual of x + omega g (AAR.c:134-139)
};

template <typename T>
struct SArgs {
    int nx = 0, ny = 0, nz = 0, nxy = 0;
    int lz = 0;                       // z-chunk length (planes per block)
    int ntx = 0, nty = 0, nzc = 0, nitems = 0;
    double w[R + 1] = {};             // a * coeff_lap[o]
    double cf[R + 1] = {};            // AAR_REC: g' = cf[0] g + sum_o cf[o] S_o (S_o: the 6 neighbours at o)
    double sigma = 0.0;               // screened term
    double diag = 1.0;                // Jacobi diagonal a*(3*coeff[0]) + sigma
    double omega = 0.0;
    int precond = 1;
    int trace = 0;
    const T *in0 = nullptr;           // stencil operand
    const T *bvec = nullptr;          // right-hand side for the epilogue
    // variable-coefficient operator A = a*Lap + c(x) (the VC sweeps only):
    // the sweeps read c(x); AAR_REC reads h(x) = omega/(diag + c(x))
    // with a Jacobi preconditioner, else c(x)
    const T *vf = nullptr;
    T *out0 = nullptr, *out1 = nullptr;
    float *out32 = nullptr;
    double *partials = nullptr;       // [nitems * NACC]
    Ctrl *ctrl = nullptr;
    FinArgs fin = {};
};

// Launch shape of the sweeps: tile = 0: the z-march (stencil_body.h), a block
// owning a 64 x (wy*py) column over lz planes; tile > 0: the one-shot boxes of
// stencil_tile.h, `tile` (1, 2 or 4) planes deep.  w < 64: columns w wide and
// narrow_rows() * 64/w high, whatever wy and py.
struct Shape {
    int lz = 0, wy = 8, py = 4;
    int tile = 0;
    int w = TX;               // width of the march's columns (march_width)
    double us = 0.0;          // measured time of one recurrence sweep (tuned shapes)
};

// (a plane beyond the sweeps' 32-bit offsets always marches 64 x WIDE_ROWS columns)
constexpr int WIDE_ROWS = 32;
template <typename T> constexpr int narrow_rows() { return sizeof(T) == 8 ? 32 : 16; }
// width of the march's columns on this grid
template <typename T>
int march_width(int nx, int ny);
template <typename T>
hipError_t launch_stencil(SMode m, const SArgs<T> &a, const Shape &sh, hipStream_t st);
// blocks (= partials per sum) of the sweep
template <typename T>
int stencil_items(const SArgs<T> &a, const Shape &sh);
// fills the tile geometry of `a` (nxy, ntx, nty, nzc, nitems; lz clamped)
template <typename T>
void stencil_geometry(SArgs<T> &a, const Shape &sh);
// planes of the one-shot boxes on this grid, or 0 where the march is faster
template <typename T>
int stencil_tile_planes(int nx, int ny, int nz);
// the variable-coefficient sweeps (a.vf set)
template <typename T>
hipError_t launch_stencil_vc(SMode m, const SArgs<T> &a, const Shape &sh, hipStream_t st);
// h = omega/(diag + c) (precond) or c, rounded to Tg
template <typename Tg>
hipError_t launch_vc_field(long n, const double *c, double diag, double omega, int precond, Tg *h,
                           hipStream_t st);
// r /= (diag + c), pointwise
hipError_t launch_div_vc(double *r, double diag, const double *c, long n, hipStream_t st);
// ---------------------------------------------------------------------------
// history sweeps
// ---------------------------------------------------------------------------

// History columns are indexed by AGE: the ring slot of age k holds the
// iterate (or residual) k steps before the newest, and the difference
// column of age k is slot(k) - slot(k+1) -- the reference's
// DX = x - x_old, DF = f - f_old (AAR.c:96-102, PGR.c:105-109).  Columns
// of age < nvalid exist (a prefix; the rest are the reference's never
// written zero columns, AAR.c:64-65).  The reference stores column of age
// k at index (it - 2 - k) mod m (AAR.c:97; PGR.c:105 with it = t), which
// is how results are laid out for the m x m solve.  In DIRECT mode (the
// stand-alone Anderson/Galerkin/L2 entry points) slot k holds column k
// itself and the layout is the identity.
template <typename T>
struct GramArgs {
    long n = 0;
    int m = 0;
    int kind = 0;             // 0 AAR (DF^T DF), 1 PGR (DX^T DF), 2 PL2R (DF^T DF of A x)
    int direct = 0;
    const T *F = nullptr;     // kind 0: residual ring; kinds 1/2: iterate ring
    const T *Y = nullptr;     // kinds 1/2: ring of A x
    const T *b = nullptr;     // kinds 1/2: rhs, f = b - Y[fslot]
    long ld = 0;
    int slot[MAXM + 1] = {};  // ring slot of age k
    int fslot = 0;            // slot of f (kind 0) or of A x (kinds 1/2)
    int nvalid = 0;
    int it = 0;
    long chunk = CHUNK_V;     // vectors a block walks at a time (m <= 8)
    int nblocks = 0;
    double *partials = nullptr;
    unsigned *counter = nullptr;
    Ctrl *ctrl = nullptr;
};

// The Gram's products: per-block partials, or with a.counter (and m <= 16)
// their sums in ctrl->G by the last block.  launch_gram_solve, next on the
// stream, sums the partials into ctrl->G and solves the m x m system (flags
// as launch_ls).
template <typename T>
hipError_t launch_gram_solve(const GramArgs<T> &a, int flags, hipStream_t st);
template <typename T>
hipError_t launch_gram(const GramArgs<T> &a, hipStream_t st);

// m x m pseudo-inverse solve on device, one wavefront: s = V W+ V^T g with
// the Golub-Reinsch SVD of tools.c:52-352 (bit-faithful).  Reads ctrl->G
// (allredvec layout), writes ctrl->s, ctrl->w.  flags: LS_TEXTBOOK -- the
// textbook left reflector (the complex solver's 2m x 2m real embedding);
// LS_GELSD -- LAPACK dgelsd's rcond = -1 cutoff of the PETSc variant
// (s_j <= 2^-53 s_max dropped) instead of tools.c's (s_j < m s_max eps).
constexpr int LS_TEXTBOOK = 1, LS_GELSD = 2;
hipError_t launch_ls(Ctrl *ctrl, int m, int flags, hipStream_t st);

// AAR.c:225-231 + 116-117:  x_new = (x_k + beta f_k) - sum_k (DX_k + beta DF_k) s_col(k)
template <typename T>
struct UpdArgs {
    long n = 0;
    int m = 0;
    int direct = 0;
    double beta = 0.0;
    const T *X = nullptr, *F = nullptr;
    long ld = 0;
    int slot[MAXM + 1] = {};
    int nvalid = 0;
    int it = 0;
    int xslot = 0, fslot = 0, oslot = 0;
    const Ctrl *ctrl = nullptr;
};
template <typename T>
hipError_t launch_aar_update(const UpdArgs<T> &a, hipStream_t st);

// Anderson step of the residual-recurrence AAR (solver.hip).  The iterate
// is held as an anchor x (updated in place) plus Richardson increments
// omega*g_j of the stored preconditioned residuals g_j; a term i of the
// update is ring slot gslot[i] (g_{jlo+i}), a correction term c is
// cslot[c] of the correction ring (x_{q+1} - x_q of an earlier Anderson
// step q).  With gamma = ctrl->s (reference column order) and difference
// column t, j = it - t: dg = g_j - g_{j-1}, dx = omega g_{j-1} or a
// correction,
//   corr  = beta g_it - sum_t gamma_t (dx_t + beta dg_t)   (g_it: term ng-1)
//   x_new = x + omega sum_{xlo <= i < xhi} g_i + corr,   written back to x;
//   C[cout] = corr when cout >= 0.
// With ncol = 0 and with_beta = 0 the same kernel folds x += omega sum g_i.
constexpr int NGMAX = MAXM + 2;
constexpr int NCMAX = MAXM + 1;
template <typename Tx, typename Tg>
struct AncArgs {
    long n = 0;
    Tx *x = nullptr;
    const Tg *G = nullptr;
    Tg *C = nullptr;
    long ld = 0;
    int ng = 0, nc = 0, ncol = 0;
    int gslot[NGMAX] = {};
    int xlo = 0, xhi = 0;     // terms of the Richardson increments since the anchor
    int with_beta = 0;        // beta g_it term (Anderson step)
    int cslot[NCMAX] = {};
    int col_ref[MAXM] = {};   // reference column of difference column t
    int col_j[MAXM] = {};     // term of g_j
    int col_c[MAXM] = {};     // correction of dx_t, or -1 for omega g_{j-1} (term col_j - 1)
    double omega = 0.0, beta = 0.0;
    int cout = -1;
    const Ctrl *ctrl = nullptr;
};
template <typename Tx, typename Tg>
hipError_t launch_anchor_update(const AncArgs<Tx, Tg> &a, hipStream_t st);

// PGR.c:117-130: x += sum DX s; Ax += sum DF s (in place at the age-0 slot),
// ||b - Ax||^2 -> FIN_PGR_RES, and the Richardson step from there
// (PGR.c:92-98): slot `next` of X = x + omega (b - Ax)/diag.
template <typename T>
struct PUpdArgs {
    long n = 0;
    int m = 0;
    T *X = nullptr, *Y = nullptr;
    const T *b = nullptr;
    long ld = 0;
    int slot[MAXM + 1] = {};
    int next = -1;            // X slot of the next iterate, or -1
    double omega = 0.0, diag = 1.0;
    const T *c = nullptr;     // variable coefficient: divisor diag + c(x)
    int precond = 1;
    int nvalid = 0;
    int it = 0;
    int nblocks = 0;
    double *partials = nullptr;
    unsigned *counter = nullptr;
    Ctrl *ctrl = nullptr;
    FinArgs fin = {};
};
template <typename T>
hipError_t launch_pgr_update(const PUpdArgs<T> &a, hipStream_t st);
// grid (= partial count) of the PGR update on n points with history m, given
// the streaming kernels' block count nb
int pgr_update_blocks(long n, int m, int nb);

// ||v||^2 (or v.w) with a finaliser, accumulated in FP64
template <typename T>
struct DotArgs {
    long n = 0;
    const T *v = nullptr, *w = nullptr;
    int nblocks = 0;
    double *partials = nullptr;
    unsigned *counter = nullptr;
    Ctrl *ctrl = nullptr;
    FinArgs fin = {};
};
template <typename T>
hipError_t launch_dot(const DotArgs<T> &a, hipStream_t st);

// The pointwise steps of CG (CG.c:106-150); the divisor of the Jacobi step
// is diag, or diag + c(x).
enum class CgStep : int {
    DIR = 0,     // s = r/diag; d = s + beta d, and first, when x is given, the
                 // x += alpha d that the previous iteration left pending
    RES = 1,     // r -= alpha q; partials r.(r/diag), r.r
    X = 2,       // x += alpha d
    X_PENDING = 3,   // the same if ctrl says an iteration left it pending
};
struct CgArgs {
    long n = 0;
    double *x = nullptr, *r = nullptr, *d = nullptr;
    const double *q = nullptr;
    double diag = 1.0;
    const double *c = nullptr;
    int precond = 1;
    int nblocks = 0;
    double *partials = nullptr;
    unsigned *counter = nullptr;
    Ctrl *ctrl = nullptr;
    FinArgs fin = {};
};
hipError_t launch_cg(CgStep step, const CgArgs &a, hipStream_t st);
// grid (= number of partial pairs) of the CG steps on n points
int cg_blocks(long n);

// ---------------------------------------------------------------------------
// complex Helmholtz (no MPI_REAL counterpart): A u = a*Lap(u) + (c(x) + i eta) u,
// complex128 interleaved (double2 = re, im), Jacobi D = (a*3*coeff[0] + c) + i eta
// ---------------------------------------------------------------------------
enum class HMode : int {
    MATVEC = 0,    // y = A u
    TRUE_RES = 1,  // f = b - A u; g = f / D; ||f||^2
    REC = 2,       // g' = g - omega (A g) / D; ||D g'||^2 for the history
};

struct HArgs {
    int nx = 0, ny = 0, nz = 0, nxy = 0;
    int lz = 0, box = 0;              // box: planes of a one-shot box, 0 the march
    int ntx = 0, nty = 0, nzc = 0, nitems = 0;
    double w[R + 1] = {};
    double dlap = 0.0;                // a * 3 * coeff[0]
    const double *c = nullptr;        // c(x) (N) or null: c0 everywhere
    double c0 = 0.0, eta = 0.0, omega = 0.0;
    int trace = 0;
    const double2 *in0 = nullptr, *bvec = nullptr;
    double2 *out0 = nullptr;
    double *partials = nullptr;       // [nitems]
    Ctrl *ctrl = nullptr;
    FinArgs fin = {};
};
hipError_t launch_hstencil(HMode m, const HArgs &a, hipStream_t st);
int hstencil_items(const HArgs &a);

// Hermitian Gram of the complex g ring (ages as in GramArgs): G_ij = <DF_i, DF_j>,
// g_i = <DF_i, f> with <u, v> = sum conj(u) v, laid out as the real 2m x 2m
// system [Gr -Gi; Gi Gr] [s_re; s_im] = [g_re; g_im] for the m x m solve.
struct HGramArgs {
    long n = 0;
    int m = 0;
    const double2 *F = nullptr;
    long ld = 0;
    int slot[MAXM + 1] = {};
    int nvalid = 0;
    int it = 0;
    int nblocks = 0;
    int flags = 0;            // launch_ls's
    double *partials = nullptr;
    Ctrl *ctrl = nullptr;
};
// per-block partials; then their sums as the real 2m x 2m system in ctrl->G
// and its solution
hipError_t launch_hgram(const HGramArgs &a, hipStream_t st);
hipError_t launch_hgram_solve(const HGramArgs &a, hipStream_t st);

// complex anchor update: AncArgs with complex gamma = s[t] + i s[m + t]
struct HAncArgs {
    long n = 0;
    double2 *x = nullptr;
    const double2 *G = nullptr;
    double2 *C = nullptr;
    long ld = 0;
    int m = 0;
    int ng = 0, nc = 0, ncol = 0;
    int gslot[NGMAX] = {};
    int xlo = 0, xhi = 0;
    int with_beta = 0;
    int cslot[NCMAX] = {};
    int col_ref[MAXM] = {};
    int col_j[MAXM] = {};
    int col_c[MAXM] = {};
    double omega = 0.0, beta = 0.0;
    int cout = -1;
    const Ctrl *ctrl = nullptr;
};
hipError_t launch_hanchor_update(const HAncArgs &a, hipStream_t st);

// dL/dc = -Re(conj(lambda) u) for a diagonal coefficient field c
hipError_t launch_helm_grad_c(long n, const double2 *lambda, const double2 *u, double *dc, hipStream_t st);

// Reducing kernels run the finaliser in their last block when given a
// counter, or only write per-block partials when counter == nullptr; then
// launch_finish runs a one-block second pass.  The Gram's second pass is
// launch_gram_solve (ctrl->G holds nothing before it), the complex Gram's
// launch_hgram_solve.
//
// A residual norm that is only recorded needs no finish of its own: the sweeps
// between two checks leave their partials in consecutive sets, and the finish
// of the next check sums them too, one more block each: hist[it0-1+j] =
// sqrt(sum of set j), j < count.  partials == nullptr: the record alone.
struct TraceFin {
    const double *partials = nullptr;
    int nitems = 0, count = 0, it0 = 0;
    double *hist = nullptr;
    int hist_cap = 0;
};
hipError_t launch_finish(const double *partials, int nitems, int nacc, const FinArgs &fin, Ctrl *ctrl,
                         hipStream_t st, const TraceFin &trace = TraceFin());

// small pointwise helpers
hipError_t launch_copy_f64(double *dst, const double *src, long n, const Ctrl *ctrl, hipStream_t st);
hipError_t launch_fill_f64(double *dst, double v, long n, hipStream_t st);
hipError_t launch_fill_f32(float *dst, float v, long n, hipStream_t st);
// x64 += e32 (mixed-precision correction)
hipError_t launch_axpy_f64_f32(double *x, const float *e, long n, hipStream_t st);
hipError_t launch_div_f64(double *r, double diag, long n, hipStream_t st);
hipError_t launch_zero_ctrl(Ctrl *c, hipStream_t st);

}  // namespace aar
