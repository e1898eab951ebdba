// lym_stencil.h -- the hop arithmetic and the workgroup -> site-block mapping shared
// by the stencil kernels (dslash.hip: one or two threads per site; dslash_hop.hip:
// one wave per direction).  The forms that launches of one kind choose between by size
// run the same operations in the same order on a site, so that an FP64 apply and a
// right-hand side of a batch have the same bits in any of them: k_dslash_stg,
// k_dslash_lanes and k_dslash_hop in FP64; k_dslash (its batch steps included) and
// k_dslash_hop in FP32 and FP16.  Others differ by rounding: k_dslash_split adds the
// x and y hops and the z and t hops apart, k_dslash_mfma sums in the matrix cores, and
// the fused update and the norms of single low-precision launches are formed and summed
// as each form does it, so a single mixed-precision solve depends on the form.
#pragma once

#include "lym_device.h"

// 1: each XCD works through its own contiguous range of site blocks;
// 0: all XCDs advance together through the lattice in block order
#ifndef LYM_XCD_MAP
#define LYM_XCD_MAP 1
#endif
// 1: within its block range an XCD takes the x-slices as the fastest index of
// its sweep (block j of every x-slice of the range, then block j + 1, ...), so
// the workgroups in flight together hold x-adjacent planes and the neighbour
// spinors and backward links of the x hops are read while still in L2;
// 0: plain block order within the range (one whole x-slice after the other).
// Measured on the 16^3x32 FP64 clover apply: L2 misses 277 -> 236-250 MB per
// apply, 49.5 -> 47.2 us; even-odd applies and solves gain alike.
#ifndef LYM_XSWEEP
#define LYM_XSWEEP 1
#endif
// 1: XCDs 2i and 2i+1 share the x-slices of both their ranges, each taking half
// of every slice's site blocks, so an XCD's domain is 4 x-slices by half the
// (y, z) blocks instead of 2 whole x-slices: 3/4 of the halo spinors and
// links.  Measured on the 16^3x32 FP64 clover apply: 252 -> 221 MB read,
// 47.1 -> 44.6 us; even-odd launches 68.4 -> 65.8 us.
#ifndef LYM_XCD_PAIRS
#define LYM_XCD_PAIRS 1
#endif

namespace lym {

template <int MU>
struct Dir;
// (1 - gamma_mu) keeps h_a = psi_a + c_a psi_{P_a} for a = 0, 1; c = i^C.
template <>
struct Dir<0> { static constexpr int P0 = 3, C0 = 1, P1 = 2, C1 = 1; };
template <>
struct Dir<1> { static constexpr int P0 = 3, C0 = 0, P1 = 2, C1 = 2; };
template <>
struct Dir<2> { static constexpr int P0 = 2, C0 = 1, P1 = 3, C1 = 3; };
template <>
struct Dir<3> { static constexpr int P0 = 2, C0 = 2, P1 = 3, C1 = 2; };

// forward:  h_a = psi_a + c_a psi_P, acc_a += U h_a, acc_P += conj(c_a) U h_a
// backward: h_a = psi_a - c_a psi_P, acc_a += U^+ h_a, acc_P -= conj(c_a) U^+ h_a
// hop_mul: the link times the two projected colour vectors (r0, r1).  SCALED:
// psi is an unscaled FP16 spinor, whose site scale hop_acc applies, with the
// boundary sign; else flip applies the sign, to the projected vectors: it is then
// out of the way while the link is still on its way.  On the products, between the
// multiply and the sum, every wave waited for its branch: Wilson applies 14^4 11.4
// against 11.1 us, 15^4 13.2 and 13.0, 16^3x28 25.9 and 25.5 (12-real links 23.0 and
// 22.6), 20^3x32 on 12-real links 60.4 and 58.3.
template <int MU, bool FWD, int LK, class T, bool SCALED = false>
__device__ __forceinline__ void hop_mul(const cplx<T> psi[12], const LinkMat<LK, T>& L, bool flip, cplx<T> r0[3],
                                        cplx<T> r1[3]) {
    using D = Dir<MU>;
    constexpr int PH0 = FWD ? D::C0 : D::C0 + 2;
    constexpr int PH1 = FWD ? D::C1 : D::C1 + 2;
    cplx<T> h0[3], h1[3];
    if constexpr (SCALED) {
        // FP16 operands: each component of h = psi_a + c psi_P as a fused
        // multiply-add by a unit the compiler cannot see through, so that the
        // conversions of both FP16 operands fold into one mixed-precision
        // instruction instead of two conversions and an add.  The value is
        // the same: the product by one is exact and the sum rounds once.
        T one = (T)1;
        asm volatile("" : "+v"(one));
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const cplx<T> m0 = mulph<PH0>(psi[3 * D::P0 + c]), m1 = mulph<PH1>(psi[3 * D::P1 + c]);
            h0[c] = mk(fmadd(m0.re, one, psi[c].re), fmadd(m0.im, one, psi[c].im));
            h1[c] = mk(fmadd(m1.re, one, psi[3 + c].re), fmadd(m1.im, one, psi[3 + c].im));
        }
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            h0[c] = psi[c] + mulph<PH0>(psi[3 * D::P0 + c]);
            h1[c] = psi[3 + c] + mulph<PH1>(psi[3 * D::P1 + c]);
            if (MU == 3 && flip) {
                h0[c] = -h0[c];
                h1[c] = -h1[c];
            }
        }
    }
    if constexpr (FWD) {
        matvec<LK, T>(L, h0, r0);
        matvec<LK, T>(L, h1, r1);
    } else {
        matvec_dag<LK, T>(L, h0, r0);
        matvec_dag<LK, T>(L, h1, r1);
    }
}

// a += r, or with SCALED a += f r as one fused multiply-add per component
template <bool SCALED, class T>
__device__ __forceinline__ void hop_acc(cplx<T>& a, cplx<T> r, T f) {
    if constexpr (SCALED) a = mk(fmadd(f, r.re, a.re), fmadd(f, r.im, a.im));
    else a = a + r;
}

// phases of the reconstruction: spin P_a receives i^Q_a r_a
template <int MU, bool FWD>
struct HopPhase {
    static constexpr int Q0 = FWD ? 4 - Dir<MU>::C0 : 6 - Dir<MU>::C0;
    static constexpr int Q1 = FWD ? 4 - Dir<MU>::C1 : 6 - Dir<MU>::C1;
};

// acc += the hop's 12 components from r0, r1; sc is the FP16 site scale
// (SCALED), flip the boundary sign
template <int MU, bool FWD, int LK, class T, bool SCALED = false>
__device__ __forceinline__ void hop_dir(cplx<T> acc[12], const cplx<T> psi[12], const LinkMat<LK, T>& L, bool flip,
                                        T sc = (T)1) {
    using D = Dir<MU>;
    using H = HopPhase<MU, FWD>;
    cplx<T> r0[3], r1[3];
    hop_mul<MU, FWD, LK, T, SCALED>(psi, L, flip, r0, r1);
    const T f = flip ? -sc : sc;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        hop_acc<SCALED, T>(acc[c], r0[c], f);
        hop_acc<SCALED, T>(acc[3 + c], r1[c], f);
        hop_acc<SCALED, T>(acc[3 * D::P0 + c], mulph<H::Q0>(r0[c]), f);
        hop_acc<SCALED, T>(acc[3 * D::P1 + c], mulph<H::Q1>(r1[c]), f);
    }
}

// ---------------------------------------------------------------- right-hand sides of a field
// FP32/FP16 fields interleave their right-hand sides (rhs fastest: the lanes of a
// site share its link loads); FP64 lanes are fields of their own, so that a lane
// with nothing to do costs no bytes (interleaved, a cache line holds a component
// of eight lanes, and the reliable updates of a batch, due in some lanes at a
// time, moved them all).
template <int PR>
__device__ __forceinline__ const typename Prec<PR>::S* lane_base(const void* f, long lane_elems, int r) {
    const typename Prec<PR>::S* b = reinterpret_cast<const typename Prec<PR>::S*>(f);
    if constexpr (PR == 0) b += r * lane_elems;
    return b;
}
// The right-hand sides one field holds are a.nr for every precision: 1 for FP64,
// read from the parameters on purpose.  As a constant it lets the compiler merge
// the spinors' address arithmetic with the links' and spread the loads of a hop
// between its products (175 waits instead of 116, the clover apply 2.4 % slower on
// 16^3x32 and on 32^3x64).
template <int PR>
__device__ __forceinline__ int field_rhs(int r) {
    return PR == 0 ? 0 : r;
}

// ---------------------------------------------------------------- fused steps of the FP64 solvers
// On small lattices an FP64 Krylov iteration is bound by its launches (a launch
// that does nothing takes 1.7 us in a replayed graph, a dot or a vector update of
// a few thousand elements 3 to 4 us): with the dots and the CG update on the
// launches that write Q p, A p, nu and t, a CG iteration on Q^2 is 5 launches
// (even-odd; 3 on the full lattice) instead of 7 (5) and a BiCGStab one 3 and its
// stencils instead of 8.  8^4 Wilson CG 3.35 -> 2.80 ms, BiCGStab of the 8^3x16
// fermion force 28.7 -> 23.2 ms; on 16^3x32 the dot costs the stencil 4.3 us of
// the 5.9 us it took alone and a solve gains 0.5 %.
__device__ __forceinline__ double state_rr(const MCGState* s) { return s->rr_s; }
__device__ __forceinline__ double state_rr(const CGState* s) { return s->rr; }
__device__ __forceinline__ void set_alpha(MCGState* s, double alpha, double rr) {
    s->alpha = alpha;
    s->rr_prev = rr;
}
__device__ __forceinline__ void set_alpha(CGState* s, double alpha, double rr) {
    s->alpha_re = alpha;
    s->alpha_im = 0;
    s->rr_prev = rr;
}

// The step's work on component k of a site, from its output v (in registers):
//   F64_NORM  sums[0] += |v|^2
//   F64_CG    x += al p, r -= al v, sums[0] += |r|^2 (the output is not stored)
//   F64_DOT   sums[0], [1] += conj(w) v, sums[2] += |v|^2
template <int FM>
__device__ __forceinline__ void f64_step(const DslashParams& a, int p, int k, unsigned site, double al, zd v,
                                         double* sums) {
    const size_t o = (size_t)k * a.g.stride;
    if constexpr (FM == F64_NORM) {
        sums[0] = norm_acc(v, sums[0]);
    } else if constexpr (FM == F64_CG) {
        const zd pv = fld<zd>(reinterpret_cast<const zd*>(a.upd_p[p]) + o, site);
        zd* xp = reinterpret_cast<zd*>(a.upd_xs[p]) + o;
        zd* rp = reinterpret_cast<zd*>(a.upd_rs[p]) + o;
        const zd rn = axpy1(-al, v, fld<zd>(rp, site));
        fst<zd, false>(xp, site, axpy1(al, pv, fld<zd>(xp, site)));
        fst<zd, false>(rp, site, rn);
        sums[0] = norm_acc(rn, sums[0]);
    } else if constexpr (FM == F64_DOT) {
        const zd w = fld<zd>(reinterpret_cast<const zd*>(a.dotw[p]) + o, site);
        sums[0] = fmadd(w.im, v.im, fmadd(w.re, v.re, sums[0]));
        sums[1] = fmadd(-w.im, v.re, fmadd(w.re, v.im, sums[1]));
        sums[2] = norm_acc(v, sums[2]);
    }
}

// Grid: gridDim.x workgroups dealt round-robin over the 8 XCDs.  XCD x owns a
// contiguous range of logical site blocks (x-major lattice order, the two
// parities of a block range interleaved) and its workgroups sweep that range
// in order, so at any time an XCD works on one compact slab and the
// neighbour spinors and links of that slab are reused from its L2.  A
// workgroup holds `spb` sites x `nr` right-hand sides, rhs fastest.
// (The mapping functions take the workgroup index and grid size as arguments so
// that the host can evaluate the same mapping: lym_launch_form.)
struct BlockSweep {
    int lo, hi, k, nphys;
};
__host__ __device__ __forceinline__ BlockSweep block_sweep_at(const DslashParams& a, int bx, int gdim) {
    const int nbt = a.nblocks_per_parity * (a.parity >= 0 ? 1 : 2);
    BlockSweep b;
#if LYM_XCD_MAP
    const int nx = 8;
    const int xcd = bx % nx;
    b.k = bx / nx;
    b.nphys = (gdim - xcd + nx - 1) / nx;  // workgroups on this XCD
    const int q = nbt / nx, rr = nbt % nx;
    b.lo = xcd < rr ? xcd * (q + 1) : rr * (q + 1) + (xcd - rr) * q;
    b.hi = b.lo + (xcd < rr ? q + 1 : q);
#else
    // plain order: consecutive workgroups (dealt round-robin over the XCDs) take
    // consecutive site blocks, so all XCDs advance one front through the lattice
    // and the neighbour slices they re-read are recent in the shared Infinity Cache
    b.k = bx;
    b.nphys = gdim;
    b.lo = 0;
    b.hi = nbt;
#endif
    return b;
}

// Which renumbering block_of_at applied (reported by lym_launch_form)
enum { MAP_PLAIN = 0, MAP_XSLICE = 1, MAP_XCD_PAIRS = 2 };

// logical block lb of the sweep of workgroup bx -> parity p and site block bi
// of that parity; returns the MAP_* branch taken
__host__ __device__ __forceinline__ int block_of_at(const DslashParams& a, const BlockSweep& b, int lb, int bx, int& p,
                                                    int& bi) {
    (void)bx;
    if (a.parity >= 0) {
        p = a.parity;
        bi = lb;
    } else {
        p = lb & 1;
        bi = lb >> 1;
    }
#if LYM_XSWEEP && LYM_XCD_MAP
    {
        // the range holds whole x-slices: renumber its blocks x-slice fastest
        const int W = a.xslice_blocks;
        const int b0 = a.parity >= 0 ? b.lo : b.lo >> 1;
        const int D = a.parity >= 0 ? b.hi - b.lo : (b.hi - b.lo) >> 1;
        const bool whole = a.parity >= 0 || ((b.lo | b.hi) & 1) == 0;
#if LYM_XCD_PAIRS
        // XCDs 2i and 2i+1 share the x-slices of both their ranges, each taking
        // half of every slice's blocks (a 2-D domain: shorter x halo)
        const int nbt = a.nblocks_per_parity * (a.parity >= 0 ? 1 : 2);
        if (W > 0 && whole && W % 2 == 0 && nbt % 16 == 0 && b0 % W == 0 && D % W == 0) {
            const int x1 = (bx % 8) & 1;
            const int b0p = b0 - x1 * D, nxs2 = 2 * D / W, Wh = W / 2;
            const int u = bi - b0, j = u / nxs2;
            bi = b0p + (u - j * nxs2) * W + x1 * Wh + j;
            return MAP_XCD_PAIRS;
        }
#endif
        if (W > 0 && whole && b0 % W == 0 && D % W == 0 && D > W) {
            const int u = bi - b0, nxs = D / W;
            const int j = u / nxs;
            bi = b0 + (u - j * nxs) * W + j;
            return MAP_XSLICE;
        }
    }
#endif
    return MAP_PLAIN;
}

// Workgroups of an FP64 launch over lanes, nw of them to a workgroup (a wave each): the
// lanes of one site block follow one another on its XCD (links and blocks that one
// lane reads are then in the L2 for the next).  Launcher: the grid; lane_of_block_at:
// the site block's workgroup bx of gd and the lane of wave w, from the launch's
// workgroup bx of gd; false when there is none; lane_of_block: also false when the
// lane has nothing to do.
static inline int lane_grid(const DslashParams& a, int nblocks, int nw) {
    return a.lanes > nw ? (nblocks + 7) / 8 * 8 * (a.lanes / nw) : nblocks;
}
__host__ __device__ __forceinline__ bool lane_of_block_at(const DslashParams& a, int nw, int w, int& bx, int& gd,
                                                          int& lane) {
    lane = w;
    if (a.lanes > nw) {
        const int t = bx >> 3, ng = a.lanes / nw, u = t / ng;
        lane += (t - u * ng) * nw;
        bx = u * 8 + (bx & 7);
        gd = a.grid1;
        if (bx >= gd) return false;
    }
    return true;
}
__device__ __forceinline__ bool lane_of_block(const DslashParams& a, int nw, int w, int& bx, int& gd, int& lane) {
    bx = (int)blockIdx.x;
    gd = (int)gridDim.x;
    if (!lane_of_block_at(a, nw, w, bx, gd, lane)) return false;
    return !(a.lane_flags && a.lane_flags[lane] == a.lane_skip_value);
}

// the one-wave-per-direction form (dslash_hop.hip): up to HOP_LANES (site, RHS) lanes,
// HOP_WAVES direction waves over them and two chirality waves
constexpr int HOP_LANES = 64;
constexpr int HOP_WAVES = 4;
constexpr int HOP_THREADS = HOP_LANES * (HOP_WAVES + 2);

__device__ __forceinline__ BlockSweep block_sweep(const DslashParams& a) {
    return block_sweep_at(a, (int)blockIdx.x, (int)gridDim.x);
}
__device__ __forceinline__ void block_of(const DslashParams& a, const BlockSweep& b, int lb, int& p, int& bi) {
    (void)block_of_at(a, b, lb, (int)blockIdx.x, p, bi);
}

}  // namespace lym
