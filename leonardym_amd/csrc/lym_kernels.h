// lym_kernels.h -- kernel parameter blocks and host-side launchers.
#pragma once

#include "lym_common.h"

namespace lym {

typedef cplx<double> zd;

// Fused steps of the FP64 solvers on a stencil launch (DslashParams::fmode)
enum { F64_STORE = 0, F64_NORM = 1, F64_CG = 2, F64_DOT = 3 };

// Parameters of one stencil launch.  Field pointers are per parity; the
// storage element type follows `prec` (0 FP64, 1 FP32, 2 FP16 + per-site
// scales); multi-RHS fields hold `nr` right-hand sides, rhs fastest.
struct DslashParams {
    Geom g;
    int prec;              // storage precision of spinors, links and clover blocks
    int nr;                // FP32/FP16: right-hand sides per field, interleaved (rhs fastest)
    int spb;               // sites per workgroup (set by the launcher)
    const void* in[2];     // per parity: the field read at neighbours is in[1 - p]
    const float* in_sc[2];
    const void* diag_in[2];  // per parity: the field under the site-diagonal term
    const float* diag_sc[2];
    void* out[2];
    float* out_sc[2];
    const void* v2[2];     // optional axpy operand
    const float* v2_sc[2];
    const void* links;
    const void* A;         // clover blocks of D, 4 planes
    const float* A_sc;     // [2][stride] (FP16)
    const void* Ainv;      // inverse blocks (even sites), 2 planes
    const float* Ainv_sc;  // [stride] (FP16)
    double kappa;
    const double* kappa_dev;  // when set, kappa is read from device memory instead
    double hop_sign;
    zd alpha;
    int gamma5;
    int parity;            // 0 or 1: that parity only; -1: both
    int nblocks_per_parity;
    const int* skip;       // optional device flag: nonzero -> the launch does nothing (solver done)
    const int* lane_flags; // optional per-RHS (FP64: per-lane) device flags: lane r does nothing when
    int lane_skip_value;   //   lane_flags[r] == lane_skip_value (an RHS that is done or needs no update)
    int threads;           // workgroup size (0: LYM_DSLASH_THREADS); a workgroup holds threads / nr sites
    int xslice_blocks;     // set by the launcher: site blocks per x-slice and parity when an x-slice
                           // is a whole number of blocks, else 0
    int allow_split;       // the caller allows the two-threads-per-site form (low precision)
    int mfma;              // the caller allows the matrix-core form (FP16 SU(3) multi-RHS, nr 2, 4 or 8)
    int split;             // set by the launcher: threads per half of that form, or 0
    double inv_ext[3];     // set by the launcher (the one-wave-per-direction form): 1 / Ly, 1 / Lz, 1 / Lth
    double* norm_partials; // optional (FP32/FP16 only): workgroup b writes the sum of |out|^2 over
    int norm_max;          //   its sites to norm_partials[b], when the launch has at most norm_max workgroups
    // Per-lane operators (multi-RHS launches of the serving engine): lane r uses
    // kappa_dev[r] and the clover blocks at A + r * A_lane_bytes (scales at
    // A_sc + r * Asc_lane), Ainv + r * Ainv_lane_bytes (Ainv_sc + r * Ainvsc_lane)
    int lane_ops;
    long A_lane_bytes, Ainv_lane_bytes, Asc_lane, Ainvsc_lane;
    const int* lane_set;  // lane_ops: lane r reads the block set lane_set[r] (NULL: set r)
    // Fused update of the mixed-precision CG (single RHS, FP32/FP16 storage; the
    // last launch of A p): instead of storing its output v = (A p)_x, the
    // launch updates x_s += alpha p and r_s -= alpha v at every site, with
    // alpha = rr_s / (the sum of the upd_ndot <p, Ap> partials at upd_dot) and
    // rr_s from the solver state upd_state (an MCGState); workgroup b writes the
    // sum of |r_s|^2 over its sites to upd_rpart[b], workgroup 0 stores alpha
    // and rr_prev = rr_s in the state.  p: storage precision; x_s, r_s: complex
    // float [12][stride] per parity.
    void* upd_state;
    const double* upd_dot;
    int upd_ndot;
    const void* upd_p[2];
    const float* upd_p_sc[2];
    void* upd_xs[2];
    void* upd_rs[2];
    double* upd_rpart;
    // The same two steps for a batch, one value per (site, RHS) so that every
    // RHS sums its terms over the batched solver's fixed site chunks:
    // bmode 1 (the launch that writes Q p): also bsite[p][site * nr + r] =
    // |(Q p)_site|^2 of lane r; bmode 2 (the last launch of Q^2 p): no output
    // store; x_s += alpha_r p and r_s -= alpha_r v (alpha from balpha[r]; p,
    // x_s, r_s as upd_p / upd_xs / upd_rs, multi-RHS fields) and bsite = the
    // site's |r_s|^2 of lane r.
    int bmode;
    double* bsite[2];
    const double* balpha;
    // A fused step of the FP64 solvers (single RHS), from the output v before it
    // is stored: F64_NORM |v|^2; F64_CG x += alpha p, r -= alpha v and |r|^2, as
    // the fused update above (upd_state a CGState, upd_p / upd_xs / upd_rs the FP64
    // p, x, r; v is not stored); F64_DOT <w, v> (dotw) and |v|^2.  Workgroup b
    // writes its sum k to upd_rpart[k * part_stride + b].
    int fmode;
    const void* dotw[2];
    int part_stride;
    // FP64: right-hand sides as fields of their own ("lanes"), lane l of a field at
    // pointer + l * stride below (in complex elements); 0 or 1: one field.  The
    // workgroups of the lanes of a site block follow one another on one XCD.
    int lanes;
    long in_lane, diag_lane, out_lane;
    int grid1;             // set by the launcher: workgroups of one lane
};
// The arguments of such a step for vectors of one parity (an odd half) or two
struct Fuse64 {
    int mode;
    double* part;     // sums: part[k * part_stride + workgroup]
    int part_stride;  // most workgroups it holds
    const zd* w;      // F64_DOT
    void* state;      // F64_CG: CGState, the <p, Ap> partials, p, x, r
    const double* dot;
    int ndot;
    const zd* p;
    zd* x;
    zd* r;
};

// Arguments of the fused mixed-CG update (DslashParams::upd_*) for one vector
// of nparity parities: p in storage precision with its scales, x_s and r_s
// complex float [nparity][12][stride]; dot: the <p, Ap> partials (count set by
// the caller once known); rpart: NORM_FOLD_MAX doubles for the |r_s|^2 partials
struct UpdArgs {
    void* state;
    const double* dot;
    int ndot;
    const void* p;
    const float* p_sc;
    void* xs;
    void* rs;
    double* rpart;
};

// link_kind: 0 complex 18, 1 complex 12, 2 real 9, 3 real 6; diag: 0 none, 1 identity, 2 clover.
// Returns the number of output-norm partials written (0: none were asked for or they did not fit).
int launch_dslash(DslashParams a, int link_kind, int diag, bool inv, hipStream_t st);
// the one-wave-per-direction form (dslash_hop.hip) of a launch whose spb, blocks per
// parity and inv_ext launch_dslash has set
void launch_dslash_hop(const DslashParams& a, int link_kind, int diag, bool inv, int nblocks, hipStream_t st);

// ---------------------------------------------------------------- layout (layout.hip)
void launch_spinor_to_eo(const Geom& g, const zd* aos, zd* eo, hipStream_t st);
void launch_spinor_from_eo(const Geom& g, const zd* eo, zd* aos, hipStream_t st);
// links_aos: complex [V][4][3x3 col-major] (real_links = 0) or real (real_links = 1)
void launch_links_to_eo(const Geom& g, const void* links_aos, int real_links, int ncomp, int unfold_bc, void* eo,
                        hipStream_t st);

// ---------------------------------------------------------------- clover (clover.hip)
void launch_clover_B(const Geom& g, const void* links, int link_kind, zd* B, hipStream_t st);
// real_links: the block kinds of real links
void launch_clover_A(const Geom& g, const zd* B, double kc, zd* A, bool real_links, hipStream_t st);
// Ainv on parity 0 from A; returns via *flag (device int) nonzero when a block is singular
void launch_clover_inv(const Geom& g, const zd* A, zd* Ainv, bool real_links, int* flag,
                       hipStream_t st);  // pivoted; flag: singular count
void launch_clover_inv_ldl(const Geom& g, const zd* A, zd* Ainv, bool real_links, int* fallback,
                           hipStream_t st);  // unpivoted
// inverse blocks (lane_set null: set 0 for every lane; else set lane_set[l] at stride
// set_elems) applied to the even half of lane fields (mask: as for launch_lane_copy)
void launch_inv_apply(const Geom& g, const zd* blocks, bool real_links, long set_elems, const int* lane_set,
                      const int* mask, const zd* in, long in_lane, zd* out, long out_lane, int lanes, hipStream_t st);

// ---------------------------------------------------------------- BLAS-1 (blas.hip)
constexpr int RED_BLOCKS = 512;

// reductions over n complex elements; results land in `result` (device) as doubles
void launch_norm2(const zd* a, long n, double* partials, double* result, hipStream_t st);
void launch_dot(const zd* a, const zd* b, long n, double* partials, double* result, hipStream_t st);
void launch_gamma5dot(const zd* a, const zd* b, long half_stride_n, int nparity, int stride, double* partials,
                      double* result, hipStream_t st);
void launch_diffnorm(const zd* a, const zd* b, long n, double* partials, double* result, hipStream_t st);

void launch_axpy(zd* y, zd a, const zd* x, long n, hipStream_t st);         // y += a x
void launch_xpay(zd* y, const zd* x, zd a, long n, hipStream_t st);         // y = x + a y
void launch_scale_g5(zd* y, int nparity, int stride, hipStream_t st);       // lower spins negated
void launch_copy(zd* y, const zd* x, long n, hipStream_t st);
void launch_set_double(double* p, double v, hipStream_t st);                // *p = v, ordered on st
void launch_sub(zd* out, const zd* a, const zd* b, long n, hipStream_t st); // out = a - b

// ---------------------------------------------------------------- solver state machines
struct CGState {
    int done, converged, step, max_steps;
    double rr, rr_new, alpha_re, alpha_im, beta, eps;
    double rr_prev;  // rr at the start of the iteration (set by the update, read by the p update)
};

enum { BICG_FOLD = 0, BICG_CHECKED = 1, BICG_FIRST = 2 };
struct BiCGState {
    int done, converged, step, max_steps, breakdown, copy_b;
    int phase;  // what the next p update finds: BICG_FOLD the last update's partials, BICG_CHECKED
                // those already folded by launch_bicg_check, BICG_FIRST the start's <rh, r> only
    double rho_re, rho_im, rhon_re, rhon_im;
    double alpha_re, alpha_im, omega_re, omega_im, beta_re, beta_im;
    double norm, precision;
};

void launch_cg_init(CGState* s, const zd* r, long n, double* partials, double eps, int max_steps, hipStream_t st);
// The steps of an iteration that are not fused into the stencil fold npart
// partial sums of the step before (sum k of workgroup b at part[k * stride + b]).
// launch_fold folds more than FOLD_MAX of them into one; npart and part then
// describe the result.  A stencil launch that does not take its fused step leaves
// none, and the caller runs the step by itself: launch_bicg_dot, or launch_cg_alpha and
// launch_cg_update.
constexpr int FOLD_MAX = 2048;
void launch_fold(int nv, const double*& part, int stride, int& npart, double* out, const int* skip, hipStream_t st);
// one CG iteration after Ap = A p, where it is not fused into the stencil: <p, Ap>
// partials (slots 0, 1 of partials), the update folding them into alpha (|r|^2
// partials into slot 2)
void launch_cg_alpha(CGState* s, const zd* p, const zd* Ap, long n, double* partials, hipStream_t st);
void launch_cg_update(CGState* s, zd* x, zd* r, const zd* p, const zd* Ap, long n, double* partials,
                      hipStream_t st);
// the p update, folding the |r|^2 partials into beta and the stopping rule
void launch_cg_p(CGState* s, zd* p, const zd* r, long n, const double* part, int npart, hipStream_t st);

void launch_bicg_init(BiCGState* s, double precision, int max_steps, hipStream_t st);
// r = b - Ax, rh = b + Ax, p = nu = 0, and <rh, r> into the partials of launch_bicg_update
void launch_bicg_setup(zd* r, zd* rh, zd* p, zd* nu, const zd* b, const zd* Ax, long n, double* partials, int stride,
                       hipStream_t st);
// One iteration: the p update (folding the last update's <rh, r> and |r|^2: the
// stopping rule and beta), the stencil of nu with <rh, nu> fused (npart partials),
// the s update, the stencil of t with <s, t> and |t|^2 fused, the x and r update
// (leaving <rh, r> and |r|^2 partials at partials[k * stride + workgroup]).
void launch_bicg_p(BiCGState* s, zd* p, const zd* r, const zd* nu, long n, const double* partials, int stride,
                   hipStream_t st);
void launch_bicg_s(BiCGState* s, zd* sv, const zd* r, const zd* nu, long n, const double* part, int stride, int npart,
                   hipStream_t st);
void launch_bicg_update(BiCGState* s, zd* x, zd* r, const zd* rh, const zd* p, const zd* sv, const zd* t, const zd* b,
                        long n, const double* part, int stride, int npart, double* partials, hipStream_t st);
// <w, v> and |v|^2 into RED_BLOCKS partials, for a stencil launch that did not
void launch_bicg_dot(const BiCGState* s, const zd* w, const zd* v, long n, double* partials, int stride,
                     hipStream_t st);
// the stopping rule of the last update, before the host reads the state
void launch_bicg_check(BiCGState* s, const double* partials, int stride, hipStream_t st);

}  // namespace lym

namespace lym {
struct MCGState {
    int done, converged, step, max_steps, rel, skip_rel, nrel, pad;
    double rr_s, rr_true, maxrr, alpha, beta, eps, delta2;
    double rr_prev;  // rr_s at the start of the iteration (set by the update, read by the p update)
};

// low-precision copies of operator data (mixed.hip); prec 1 FP32, 2 FP16
void launch_convert_blocks(int prec, const zd* src, void* dst, float* sc, int kind, int stride, hipStream_t st);
// two rows of FP64 links [2][4][nc][stride] into the packed low-precision layout of
// link kinds 1 / 3 (row 2 rebuilt in the stencil), or three (nc = 9) into that of 0 / 2
void launch_pack_links(int prec, const void* src, int nc, int rows, int real_links, void* dst, int stride,
                       hipStream_t st);
// per-workgroup maxima (RED_BLOCKS of them) of the deviation of row 2 of
// 18-real / 9-real FP64 links from the row rebuilt out of rows 0 and 1
void launch_link_row2_err(const void* src, int real_links, int stride, double* partials, hipStream_t st);
// FP64 spinor field <-> sloppy field of storage precision prec (FP16: with its
// per-site scales), nsites = nparity * stride sites
void launch_spinor_to_sloppy(int prec, const zd* src, void* dst, float* dst_sc, long nsites, int stride,
                             hipStream_t st);
void launch_spinor_from_sloppy(int prec, const void* src, const float* src_sc, zd* dst, long nsites, int stride,
                               hipStream_t st);
// mixed-precision CG with reliable updates; vectors span nsites = nparity * stride sites
void launch_mcg_init(int prec, MCGState* s, const zd* r, cplx<float>* rs, cplx<float>* xs, void* p, float* p_sc,
                     long nsites, int stride, double* partials, double eps, double delta, int max_steps, hipStream_t st);
// <p, Ap> partials into partials[0, RED_BLOCKS); launch_mcg_update folds ndot
// partials of <p, Ap> (those, or the stencil's output-norm partials: for
// A = Q^2 with Q hermitian, <p, Ap> = |Q p|^2) into alpha and writes |r_s|^2
// partials to partials[RED_BLOCKS, 2 RED_BLOCKS)
constexpr int NORM_FOLD_MAX = 2048;  // most partials the update folds
void launch_mcg_alpha(int prec, MCGState* s, void* p, float* p_sc, void* Ap, float* Ap_sc, long nsites, int stride,
                      double* partials, hipStream_t st);
void launch_mcg_update(int prec, MCGState* s, cplx<float>* xs, cplx<float>* rs, void* p, float* p_sc, void* Ap,
                       float* Ap_sc, long nsites, int stride, double* partials, const double* dot_partials, int ndot,
                       hipStream_t st);
void launch_rel_accum(MCGState* s, zd* x, cplx<float>* xs, long nsites, int stride, hipStream_t st);
void launch_accum_xs(zd* x, const cplx<float>* xs, long nsites, int stride, hipStream_t st);
void launch_rel_resid(MCGState* s, zd* r, cplx<float>* rs, const zd* b, const zd* Ax, long nsites, int stride,
                      double* partials, hipStream_t st);
// p = r_s + beta p after launch_mcg_update, with beta and the state step taken
// from the update's |r_s|^2 partials (nupd > 0: the nupd partials at upd_part
// of an update fused into the stencil)
void launch_mcg_p(int prec, MCGState* s, void* p, float* p_sc, const cplx<float>* rs, long nsites, int stride,
                  const double* partials, hipStream_t st, const double* upd_part = nullptr, int nupd = 0);

// ---------------------------------------------------------------- multi-RHS mixed CG (batch.hip)
constexpr int BMAX = 16;
struct BState {
    int all_done, any_rel, skip_rel, max_steps;
    int done[BMAX], conv[BMAX], step[BMAX], rel[BMAX], nrel[BMAX];
    double delta2;
    double eps[BMAX], rr_s[BMAX], rr_true[BMAX], maxrr[BMAX], alpha[BMAX], beta[BMAX];
};
constexpr int BATCH_CHUNK = 64;  // sites per fixed summation chunk of the batched solver
struct BcgArgs {
    zd* x;
    zd* r;
    const zd* b;
    const zd* Ax;
    cplx<float>* xs;
    cplx<float>* rs;
    void* p;
    float* p_sc;
    void* Ap;
    float* Ap_sc;
    long nsites;  // x, r, b, Ax: FP64 lane fields of 12 * nsites elements per lane
    int stride;
    int max_steps;
    double* partials;  // BMAX * ceil(nsites / BATCH_CHUNK) doubles
    const int* mask = nullptr;  // steps 0 (init) and 6 (final accumulate): only lanes with mask[q] != 0
    const double* bsite = nullptr;  // steps 7, 8: one value per (site, RHS), site-major
    int vh = 0;                     // steps 7, 8: the real sites of each parity (of stride)
};
// the fused batch steps on one stencil launch (DslashParams::bmode)
struct BFuse {
    int mode;
    double* bsite;
    const double* balpha;
    const void* p;
    const float* p_sc;
    void* xs;
    void* rs;
};
// which: 0 init, 1 alpha, 2 update, 3 reliable accumulate, 4 reliable residual, 5 p update, 6 final accumulate,
// 7 alpha and 8 the update's sums from the per-(site, RHS) values at bsite (a stencil's bmode 1 / 2)
bool launch_bcg_step(int which, int prec, int nr, BState* s, const BcgArgs& a, hipStream_t st);
bool batch_nr_supported(int nr);
// FP64 lane fields: lane l of a field at l * its lane stride (elements), n
// elements per lane; lanes with mask[l] == 0 (mask may be null) are left alone.
// copy and difference; from and to single fields (a null pointer leaves its lane alone)
void launch_lane_copy(zd* dst, long dst_lane, const zd* src, long src_lane, long n, int lanes, const int* mask,
                      hipStream_t st);
void launch_lane_sub(zd* out, const zd* a, const zd* b, long lane, long n, int lanes, const int* mask, hipStream_t st);
void launch_lane_gather(const zd* const* srcs_dev, zd* dst, long n, int lanes, hipStream_t st);
void launch_lane_scatter(const zd* src, zd* const* dsts_dev, long n, int lanes, hipStream_t st);
// single full fields <-> an interleaved FP64 field (rhs fastest)
void launch_pack(const zd* const* srcs_dev, int nr, zd* multi, long n, hipStream_t st);
void launch_unpack(const zd* multi, int nr, zd* const* dsts_dev, long n, hipStream_t st);
// an interleaved field (rows x nr elements of esize bytes, lane fastest) to
// another width (a lane keeps its index; new lanes are zero)
void launch_relayout(int esize, const void* in, void* out, long rows, int w_old, int w_new, hipStream_t st);
// zero the padding slots (sites vh..stride-1) of an nr-field of `groups` groups
// of stride * nr elements of esize (16, 8 or 4) bytes.  No launch writes them,
// and a buffer reused at another width would otherwise hold, there, values of
// real sites of the old layout, which per-RHS sums and copies read.
void launch_zero_padding(int esize, void* buf, long groups, int stride, int vh, int nr, hipStream_t st);
// x = uniform [0,1) complex on real sites, zero on padding (BiCGStab start for a zero source)
void launch_fill_uniform(zd* x, int nparity, int stride, int Vh, uint64_t seed, hipStream_t st);
}  // namespace lym
