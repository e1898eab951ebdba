// plan.cpp -- the stencil's launch choices, evaluated on the host for the caller to see
// (lym_launch_plan, lym_launch_form).
#include <cstring>

#include "lym_plan.h"

namespace lym_internal {
int fail(int code, const char* fmt, ...);
}

// the geometry of a context's launches on this lattice: even-odd when all extents are
// even, else one class (whose launches are parity 0)
static int plan_geometry(const int dims[4], int parity, lym::DslashParams& a) {
    using lym_internal::fail;
    for (int i = 0; i < 4; ++i)
        if (dims[i] < 2) return fail(LYM_ERR_INVALID, "lattice extent %d must be >= 2", dims[i]);
    const int tsh = (dims[0] | dims[1] | dims[2] | dims[3]) % 2 == 0 ? 1 : 0;
    if (parity < -1 || parity > 1 || (!tsh && parity != 0)) return fail(LYM_ERR_INVALID, "bad launch arguments");
    const long V = (long)dims[0] * dims[1] * dims[2] * dims[3];
    if ((V >> tsh) > (1L << 27) - 64) return fail(LYM_ERR_INVALID, "lattice too large");
    std::memset(&a, 0, sizeof(a));
    for (int i = 0; i < 4; ++i) a.g.L[i] = dims[i];
    a.g.tsh = tsh;
    a.g.Lth = dims[3] >> tsh;
    a.g.Lxh = dims[0] >> tsh;
    a.g.Vh = (int)(V >> tsh);
    a.g.stride = (int)(((V >> tsh) + 63) / 64 * 64);
    a.g.bc_t = -1;
    a.parity = parity;
    return LYM_OK;
}

extern "C" int lym_launch_plan(const int dims[4], int parity, int nr, int threads, int lowp, int* grid, int* spb,
                               int* nbpp, int* xslice_blocks, int* visits, long visits_len, int* branches) {
    using lym_internal::fail;
    if (!dims || !grid || !spb || !nbpp || !xslice_blocks) return fail(LYM_ERR_INVALID, "null argument");
    if (nr < 1 || nr > 16 || threads < 0 || threads > LYM_DSLASH_THREADS)
        return fail(LYM_ERR_INVALID, "bad launch arguments");
    lym::DslashParams a;
    if (const int rc = plan_geometry(dims, parity, a)) return rc;
    a.nr = nr;
    a.threads = threads;
    a.prec = lowp ? 2 : 0;
    a.allow_split = lowp ? 1 : 0;
    const int gdim = lym::plan_dslash(a);
    *grid = gdim;
    *spb = a.spb;
    *nbpp = a.nblocks_per_parity;
    *xslice_blocks = a.xslice_blocks;
    if (visits && visits_len < 2L * a.nblocks_per_parity) return fail(LYM_ERR_INVALID, "visits array too short");
    if (visits) std::memset(visits, 0, sizeof(int) * 2 * (size_t)a.nblocks_per_parity);
    if (branches) branches[0] = branches[1] = branches[2] = 0;
    for (int bx = 0; bx < gdim; ++bx) {
        const lym::BlockSweep b = lym::block_sweep_at(a, bx, gdim);
        for (int lb = b.lo + b.k; lb < b.hi; lb += b.nphys) {
            int p = 0, bi = 0;
            const int br = lym::block_of_at(a, b, lb, bx, p, bi);
            if (p < 0 || p > 1 || bi < 0 || bi >= a.nblocks_per_parity)
                return fail(LYM_ERR_INVALID, "workgroup %d maps block %d to (%d, %d), outside the lattice", bx, lb, p,
                            bi);
            if (visits) ++visits[p * a.nblocks_per_parity + bi];
            if (branches) ++branches[br];
        }
    }
    return LYM_OK;
}

extern "C" int lym_launch_form(const int dims[4], int parity, int prec, int nrhs, int threads, int options, int step,
                               int part_max, lym_launch_info* info, int* visits, long visits_len) {
    using lym_internal::fail;
    if (!dims || !info) return fail(LYM_ERR_INVALID, "null argument");
    if (prec < 0 || prec > 2 || nrhs < 1 || nrhs > 16 || threads < 0 || threads > LYM_DSLASH_THREADS || step < 0 ||
        step > 2 || part_max < 0 || (options & ~(LYM_LAUNCH_SINGLE | LYM_LAUNCH_MATRIX_CORES | LYM_LAUNCH_LANE_OPS)))
        return fail(LYM_ERR_INVALID, "bad launch arguments");
    lym::DslashParams a;
    if (const int rc = plan_geometry(dims, parity, a)) return rc;
    a.prec = prec;
    a.nr = prec ? nrhs : 1;
    a.lanes = prec ? 0 : nrhs;
    a.threads = threads;
    a.allow_split = prec && (options & LYM_LAUNCH_SINGLE);
    a.mfma = (options & LYM_LAUNCH_MATRIX_CORES) ? 1 : 0;
    a.lane_ops = (options & LYM_LAUNCH_LANE_OPS) ? 1 : 0;
    double part;  // (its address only: the step is asked for)
    if (step && prec == 0) a.fmode = step == 2 ? lym::F64_CG : lym::F64_NORM;
    if (step == 1 && prec) a.norm_partials = &part;
    if (step == 2) a.upd_state = &part;
    a.part_stride = a.norm_max = part_max;
    const lym::LaunchPlan L = lym::plan_launch(a, 0, 1, false);
    std::memset(info, 0, sizeof(*info));
    info->form = L.form;
    info->spb = a.spb;
    info->nbpp = a.nblocks_per_parity;
    info->partials = L.partials;
    const bool lanes = prec == 0 && (L.form == LYM_FORM_HOP || L.form == LYM_FORM_LANES);
    const int nw = L.form == LYM_FORM_LANES ? lym::lane_waves(a) : 1;
    info->grid = lanes ? lym::lane_grid(a, L.nblocks, nw) : L.nblocks;
    info->threads = L.form == LYM_FORM_HOP     ? lym::HOP_THREADS
                    : L.form == LYM_FORM_LANES ? 64 * nw
                    : L.form == LYM_FORM_SPLIT ? 2 * a.split
                                               : a.spb * a.nr;
    if (visits && visits_len < 2L * info->nbpp) return fail(LYM_ERR_INVALID, "visits array too short");
    if (visits) std::memset(visits, 0, sizeof(int) * 2 * (size_t)info->nbpp);
    auto visit = [&](int p, int bi, int br) {
        if (p < 0 || p > 1 || bi < 0 || bi >= info->nbpp) return false;
        if (visits) ++visits[p * info->nbpp + bi];
        ++info->branches[br];
        return true;
    };
    for (int b0 = 0; b0 < info->grid; ++b0)
        for (int w = 0; w < nw; ++w) {
            int bx = b0, gd = info->grid, lane = 0;
            if (lanes && (!lym::lane_of_block_at(a, nw, w, bx, gd, lane) || lane >= nrhs)) continue;
            bool ok = true;
            if (L.form == LYM_FORM_HOP) {
                const int lb = lym::xcd_block(bx, gd);
                ok = visit(parity >= 0 ? parity : lb & 1, parity >= 0 ? lb : lb >> 1, lym::MAP_PLAIN);
            } else {
                const lym::BlockSweep b = lym::block_sweep_at(a, bx, gd);
                for (int lb = b.lo + b.k; ok && lb < b.hi; lb += b.nphys) {
                    int p = 0, bi = 0;
                    const int br = lym::block_of_at(a, b, lb, bx, p, bi);
                    ok = visit(p, bi, br);
                    if (lanes) break;  // (one block a wave: the grid holds them all)
                }
            }
            if (!ok) return fail(LYM_ERR_INVALID, "workgroup %d maps to a block outside the lattice", b0);
        }
    return LYM_OK;
}
