// lym_plan.h -- what one stencil launch runs: its form, the sites of a workgroup, the
// workgroups and the block order, chosen on the host from the lattice, the precision,
// the right-hand sides and the steps asked for.  launch_dslash (dslash.hip) and
// lym_launch_form (plan.cpp) make the same choice.
#pragma once

#include "../../include/lym.h"
#include "lym_stencil.h"

// Launch shape of the stencil (swept on the device; defaults are the measured best)
#ifndef LYM_DSLASH_THREADS
#define LYM_DSLASH_THREADS 256
#endif
// both parities of a block range run on the same XCD (links and spinors of a
// region are then fetched into one L2 for the even and the odd sites)
// -1: automatic -- one sweeping workgroup per CU for FP64 launches and FP32 ones of
// two threads per site of at most LYM_SWEEP_MAX_BLOCKS workgroups (small lattices:
// 16^3x32 FP64 clover 38.1 us, 42.1 with all workgroups at once; FP32 21.5, 22.7),
// all workgroups at once above that (large lattices, where sweeping was slower) and
// for the others, whose waves are smaller and wait longer for what they load: one
// workgroup per CU leaves them one wave per SIMD (16^3x32 FP16 two threads per
// site 17.1 us swept, 14.8 at once; Schur complement of 3 and 4 right-hand sides
// 69.5 and 73.4, 44.7 and 45.3 at once; FP32 78.9, 72.3 at once)
#ifndef LYM_GRID_PER_CU
#define LYM_GRID_PER_CU -1
#endif
#ifndef LYM_SWEEP_MAX_BLOCKS
#define LYM_SWEEP_MAX_BLOCKS 1024
#endif
// 1: single-RHS FP32/FP16 applies of at most LYM_SPLIT_MAX_SITES sites per
// parity run two threads per site (k_dslash_split).  Measured: mixed CG on
// 16^3x32 (65536 sites) 5 % faster, on 24^3x48 (331776) 4 % slower
#ifndef LYM_SPLIT_LOWP
#define LYM_SPLIT_LOWP 1
#endif
#ifndef LYM_SPLIT_MAX_SITES
#define LYM_SPLIT_MAX_SITES 131072
#endif

namespace lym {

// FP64 waves of a workgroup of LYM_FORM_LANES at most (k_dslash_lanes)
constexpr int LANE_WAVES = 4;

// FP64 launches over lanes: their waves to a workgroup, a divisor of the lanes (the
// batch widths are 1, 2, 3, 4, 6, 8, 12 and 16)
inline bool over_lanes(const DslashParams& a) { return a.prec == 0 && (a.lanes > 1 || a.lane_flags || a.lane_ops); }
inline int lane_waves(const DslashParams& a) {
    for (int w = LANE_WAVES; w > 1; --w)
        if (a.lanes % w == 0) return a.lanes > 1 ? w : 1;
    return 1;
}

// The matrix-core form: FP16 SU(3) batches of 2, 4 or 8 RHS in whole waves, on lattices
// whose links its lanes reach
inline bool takes_mfma(const DslashParams& a) {
    return a.mfma && !a.bmode && mfma_reach(a.g.stride, a.nr) && (a.nr == 2 || a.nr == 4 || a.nr == 8) &&
           (a.spb * a.nr) % 64 == 0;
}

// Launch geometry: sites per workgroup, the split form, site blocks per parity
// and per x-slice; returns the number of workgroups.
inline int plan_dslash(DslashParams& a) {
    if (a.nr < 1) a.nr = 1;
    const int threads = (a.threads > 0 && a.threads <= LYM_DSLASH_THREADS) ? a.threads : LYM_DSLASH_THREADS;
    a.spb = threads / a.nr;
    if (a.spb < 1) a.spb = 1;
    // two threads per site: low-precision single-RHS applies that allow it
    a.split = (LYM_SPLIT_LOWP && a.allow_split && !a.lane_ops && !a.bmode && a.prec >= 1 && threads % 64 == 0 &&
               (long)a.g.Vh * a.nr <= LYM_SPLIT_MAX_SITES)
                  ? threads
                  : 0;
    a.nblocks_per_parity = (a.g.Vh + a.spb - 1) / a.spb;
    {
        const int xs = a.g.Vh / a.g.L[0];  // sites of one parity per x-slice
        a.xslice_blocks = (xs % a.spb == 0) ? xs / a.spb : 0;
    }
    int nblocks = a.nblocks_per_parity * (a.parity >= 0 ? 1 : 2);
    // workgroups in flight: LYM_GRID_PER_CU per CU of the 256 CUs, sweeping
    const bool sweep = (a.prec == 0 || (a.prec == 1 && a.split)) && nblocks <= LYM_SWEEP_MAX_BLOCKS;
    const int gpc = LYM_GRID_PER_CU >= 0 ? LYM_GRID_PER_CU : (sweep ? 1 : 0);
    if (gpc > 0 && nblocks > 256 * gpc) nblocks = 256 * gpc;
    return nblocks;
}

// Launches of at most this many (site, RHS) lanes take the one-wave-per-direction
// form (dslash_hop.hip); low-precision launches of one parity, whose other form
// waits longest, more of them, and FP64 launches over several lanes fewer: their other
// form has a wave per lane for every 64 sites, which hide each other's waits.  Measured, that form against the other: FP64 even-odd
// CG iteration 83 against 91 us at 32768 lanes, Schur complement 39.0 against 38.4 at
// 40960 and 43.0 against 41.9 at 49152; full applies 10.2 against 13.6 us at 20736
// lanes (clover), 14.3 against 12.5 us at 41472 (Wilson).  Low-precision Schur
// complement at 41472 lanes of two RHS 14.2 against 21.9 us (FP16), 18.8 against 22.5
// (FP32), at 49152 lanes of one 17.7 against 19.6 and 23.3 against 25.7; FP16 mixed CG
// iteration 78 against 67 us at 65536.  FP64 over lanes, by whole batched FP16 solves of
// as many right-hand sides: four and more at 8192 lanes 3.13 against 3.24 ms (8^4, 4),
// at 16384 4.37 against 4.20 (8^3x16, 4) and 3.56 against 3.47 (8^4, 8), at 82944 7.7
// against 7.1 (12^4, 8), at 393216 21.1 against 19.1 (16^4, 12); two, whose other form
// has half the waves, at 41472 4.99 against 5.02 (12^3x24; adjoint 4.58 and 4.67), at
// 54880 6.51 against 6.37 (14^3x20), at 65536 6.74 against 6.50 (16^4).
#ifndef LYM_HOP_MAX
#define LYM_HOP_MAX 32768
#endif
#ifndef LYM_HOP_MAX_LOWP_HALF
#define LYM_HOP_MAX_LOWP_HALF 49152
#endif
#ifndef LYM_HOP_MAX_FP64_LANES
#define LYM_HOP_MAX_FP64_LANES 8192
#endif
#ifndef LYM_HOP_MAX_FP64_PAIR
#define LYM_HOP_MAX_FP64_PAIR 49152
#endif

// The launch geometry of that form: sites per workgroup and site blocks per
// parity; returns the number of workgroups, or 0 when the launch takes another.
inline int plan_hop(DslashParams& a) {
    const int par = a.parity >= 0 ? 1 : 2;
    const int rhs = a.prec == 0 && a.lanes > 1 ? a.lanes : a.nr;
    const long lanes = (long)a.g.Vh * par * rhs;
    const long most = a.prec ? (par == 1 ? LYM_HOP_MAX_LOWP_HALF : LYM_HOP_MAX)
                             : (rhs > 2 ? LYM_HOP_MAX_FP64_LANES : rhs == 2 ? LYM_HOP_MAX_FP64_PAIR : LYM_HOP_MAX);
    if (LYM_T_SLOW || a.mfma || a.nr > 64 || lanes > most) return 0;
    a.spb = 64 / a.nr;
    // tiny launches: fewer sites per workgroup, so that more CUs share the loads
    while (a.spb > 1 && a.spb * a.nr > 16 && (a.g.Vh + a.spb - 1) / a.spb * par < 256) a.spb = (a.spb + 1) / 2;
    a.nblocks_per_parity = (a.g.Vh + a.spb - 1) / a.spb;
    a.inv_ext[0] = 1.0 / a.g.L[1];
    a.inv_ext[1] = 1.0 / a.g.L[2];
    a.inv_ext[2] = 1.0 / a.g.Lth;
    return a.nblocks_per_parity * par;
}

// FP64 launches of one field that a sweep would spread badly run one wave to a
// workgroup instead of four.  A CU's time is that of the waves it gets: with n
// workgroups of four waves, 4 ceil(n / 256), some CUs a workgroup more than others;
// with single waves ceil(4 n / 256).  Where that is at most 0.8 of the other (more
// than it costs that fewer z neighbours are in the block's own copy): SU(3) clover
// 16^3x20 31.4 -> 24.6 us, 16^3x24 33.6 -> 30.1, 14^4 16.3 -> 15.1, 17x15x13x21
// 31.7 -> 24.4, Schur complement 16x20^2x24 81.0 -> 68.6.  Above it the four waves are as
// fast or faster: at 7 against 8 (16^3x28) 35.4 and 36.4, at 4 against 4 (15^4) 18.1 and
// 18.7.  Launches over lanes always hold blocks of 64 sites, a wave each.  Returns the
// workgroups (of one lane), or 0 when the launch keeps workgroups of four.
inline int plan_waves(DslashParams& a) {
    if (a.prec != 0) return 0;
    const int par = a.parity >= 0 ? 1 : 2;
    const int n4 = a.nblocks_per_parity * par, nb = (a.g.Vh + 63) / 64, n1 = nb * par;
    if (!over_lanes(a)) {
        if (LYM_DSLASH_THREADS != 256) return 0;  // (the rule counts workgroups of four waves)
        if (n4 > LYM_SWEEP_MAX_BLOCKS || 5 * ((n1 + 255) / 256) > 16 * ((n4 + 255) / 256)) return 0;
        if (a.fmode && n1 > FOLD_MAX) return 0;  // a fold more would take what it gains
    }
    a.spb = 64;
    a.nblocks_per_parity = nb;
    const int xs = a.g.Vh / a.g.L[0];
    a.xslice_blocks = xs % 64 == 0 ? xs / 64 : 0;
    return n1;
}

// What a launch runs: its form, the workgroups of one lane, and the partial sums its
// fused step leaves (0: none asked for, or not fused).  Sets in a what the kernels
// read of it, and clears the steps the launch does not take.
struct LaunchPlan {
    int form, nblocks, partials;
};
inline LaunchPlan plan_launch(DslashParams& a, int link_kind, int diag, bool inv) {
    const int threads = (a.threads > 0 && a.threads <= LYM_DSLASH_THREADS) ? a.threads : LYM_DSLASH_THREADS;
    if (a.nr < 1) a.nr = 1;
    if (a.prec == 0) a.threads = 0;
    LaunchPlan L{LYM_FORM_SITE, plan_hop(a), 0};
    if (L.nblocks) {
        L.form = LYM_FORM_HOP;
    } else {
        L.nblocks = plan_dslash(a);
        if (const int n = plan_waves(a)) L.nblocks = n;
        if (a.prec == 0) L.form = over_lanes(a) ? LYM_FORM_LANES : a.spb == 64 ? LYM_FORM_WAVE : LYM_FORM_STAGED;
        else if (a.prec == 2 && link_kind == 0 && takes_mfma(a)) L.form = LYM_FORM_MFMA;
        else if (a.split) L.form = LYM_FORM_SPLIT;
    }
    a.grid1 = L.nblocks;
    // output norm partials: low precision only, one per workgroup, and only
    // when the caller's buffer holds one per workgroup of this launch
    // (the workgroup sum shuffles over whole 64-lane waves)
    const bool whole_waves = L.form == LYM_FORM_HOP || threads % 64 == 0;
    if (a.prec == 0 || diag == 0 || inv || a.nr != 1 || a.lane_flags || !whole_waves || L.nblocks > a.norm_max)
        a.norm_partials = nullptr;
    // the FP64 solvers' fused steps: one RHS, a diagonal and no R^-1, and room for
    // one partial per workgroup (the caller checks the return value and runs the
    // separate step when it is 0)
    if (a.prec != 0 || diag == 0 || inv || a.lanes > 1 || a.lane_flags || a.lane_ops || L.nblocks > a.part_stride)
        a.fmode = F64_STORE;
    // the fused update: FP64 F64_CG; low precision under the same conditions
    if (a.prec == 0) {
        if (a.fmode != F64_CG) a.upd_state = nullptr;
    } else if (diag == 0 || inv || a.nr != 1 || a.lane_flags || a.lane_ops || !whole_waves ||
               L.nblocks > a.norm_max || a.norm_partials) {
        a.upd_state = nullptr;
    }
    L.partials = a.norm_partials || a.upd_state || a.fmode ? L.nblocks : 0;
    return L;
}

}  // namespace lym
