// dslash.hip -- Wilson / clover hopping stencil for gfx950, FP64.
//
// One thread per lattice site of one parity.  For every direction mu the
// neighbour spinors x+mu and x-mu (other parity) are loaded as 12 coalesced
// complex streams, spin-projected to two colour vectors with (1 -+ gamma_mu),
// multiplied by U_mu(x) or U_mu(x-mu)^dagger and accumulated with the
// gamma_mu reconstruction, as in the reference's per-site loops
// (source/dirac_operators/DiracWilsonOperator.cpp:21-192,
//  BasicDiracWilsonOperator.cpp:16-93, EvenOddImprovedDiracWilsonOperator.cpp:204-281).
//
// The epilogue is fused: v = diag(psi_x) + hop_sign * (-kappa H psi),
// optionally v = Ainv v, gamma5, and v += alpha v2.  diag is nothing, the
// identity (Wilson) or the packed clover block A = 1 + kappa csw gamma5 B
// (ImprovedDiracWilsonOperator.cpp:200-243), so a single kernel covers
//   full-lattice Q / D and multiplyAdd        diag = A or 1, hop_sign = +1
//   EO  tmp_e = R_ee^-1 D_eo psi_o            diag = none,   INV
//   EO  out_o = R_oo psi_o - D_oe tmp_e       diag = A,      hop_sign = -1
//   EO driver source b_o - D_oe R^-1 b_e and even reconstruction
//   R_ee^-1 (b_e - D_eo x_o)                  diag = 1, hop_sign = -1 [, INV]
// (PreconditionedBiCGStab.cpp:56-86).
#include "lym_plan.h"

// Full-lattice applies: odd-parity sites take each direction's backward hop
// before its forward hop, so the two reads of a link U_mu(y) -- by y (forward)
// and by y + mu (backward), sites of opposite parity -- happen at the same
// step of the kernel instead of one step apart.
#ifndef LYM_ALT_ORDER
#define LYM_ALT_ORDER 0
#endif
// Hops whose loads may be in flight together: a register barrier (pin) after
// every hop (1), every direction pair (2) or every two directions (4).
// More hops in flight raise memory-level parallelism per wave at the cost of
// registers, which pays when the lattice gives few waves per SIMD anyway.
// FP64: 2 (about 237 VGPRs, 2 waves per SIMD) -- the single-parity launches of
// the even-odd operator ran 7 % faster than with 1 (120 VGPRs), full applies
// alike; 4 (380 registers, 1 wave per SIMD) was slower.
#ifndef LYM_PIN_HOPS
#define LYM_PIN_HOPS 2
#endif
// the same for FP32/FP16 storage, whose hops need far fewer registers
// (8: no barrier between hops at all).  4 (125-150 VGPRs for FP16): the
// mixed-precision even-odd CG ran 5-14 % faster than with 1; 8 slowed the
// FP32 stencil down.
#ifndef LYM_PIN_HOPS_LOWP
#define LYM_PIN_HOPS_LOWP 4
#endif
#ifdef LYM_WAVES_PER_EU
#define LYM_OCC __attribute__((amdgpu_waves_per_eu(LYM_WAVES_PER_EU, LYM_WAVES_PER_EU)))
#else
#define LYM_OCC
#endif

namespace lym {

// Empty asm that reads and writes the accumulator and clobbers memory: the
// hop of one direction must finish before the next direction's loads are
// issued, which bounds the live registers to one hop (without it every load of
// all eight hops is hoisted ahead of the arithmetic and the kernel spills).
template <class T>
__device__ __forceinline__ void pin(cplx<T> acc[12]) {
#pragma unroll
    for (int k = 0; k < 12; ++k) asm volatile("" : "+v"(acc[k].re), "+v"(acc[k].im));
    asm volatile("" ::: "memory");
}

// the neighbour spinor at idx: from the LDS copy of the other parity's site
// block [lbase, lbase + TH) when lds is set and idx is inside,
// else from the field
template <int MU, int PR, int TH>
__device__ __forceinline__ void load_nb(const SpinorRef<PR>& src, int stride, int nr, int idx, int r,
                                        cplx<typename Prec<PR>::T> psi[12], typename Prec<PR>::T& sc,
                                        const cplx<double>* lds, int lbase) {
    if constexpr (PR == 0 && MU >= 2) {
        if (lds) {
            const unsigned j = (unsigned)(idx - lbase);
            if (j < (unsigned)TH) {
#pragma unroll
                for (int k = 0; k < 12; ++k) psi[k] = lds[k * TH + j];
                sc = 1.0;
                return;
            }
        }
    }
    load_spinor_unscaled<PR>(src, stride, nr, idx, r, psi, sc);
}

// one hop pair (forward and backward, or backward first when BWD_FIRST) in
// direction MU for site (p, site), rhs r; lds, lbase: as for load_nb
template <int MU, int PR, int LK, bool BWD_FIRST = false, int TH = LYM_DSLASH_THREADS>
__device__ __forceinline__ void hop_pair(const DslashParams& a, int p, int site, int r, const int c[4],
                                         cplx<typename Prec<PR>::T> acc[12], const cplx<double>* lds = nullptr,
                                         int lbase = 0) {
    typedef typename Prec<PR>::T T;
    const Geom& g = a.g;
    const int q = p ^ g.tsh;
    int cu[4] = {c[0], c[1], c[2], c[3]}, cd[4] = {c[0], c[1], c[2], c[3]};
    cu[MU] = c[MU] + 1 == g.L[MU] ? 0 : c[MU] + 1;
    cd[MU] = c[MU] == 0 ? g.L[MU] - 1 : c[MU] - 1;
    const int iu = eo_index(g, cu[0], cu[1], cu[2], cu[3]);
    const int id = eo_index(g, cd[0], cd[1], cd[2], cd[3]);
    const bool anti = MU == 3 && g.bc_t < 0;
    const SpinorRef<PR> src{lane_base<PR>(a.in[q], a.in_lane, r), a.in_sc[q]};
    const int rr = field_rhs<PR>(r);
    constexpr bool SC = PR == 2;
    cplx<T> psi[12];
    T sc;
    LinkMat<LK, T> L;
    constexpr int PH = PR == 0 ? LYM_PIN_HOPS : LYM_PIN_HOPS_LOWP;
    constexpr bool pin_mid = PH == 1;
    constexpr bool pin_end = PH <= 2 || (PH == 4 && (MU & 1));
    if constexpr (!BWD_FIRST) {
        load_nb<MU, PR, TH>(src, g.stride, a.nr, iu, rr, psi, sc, lds, lbase);
        load_link<PR, LK>(a.links, g.stride, p, MU, site, L);
        hop_dir<MU, true, LK, T, SC>(acc, psi, L, anti && c[3] == g.L[3] - 1, sc);
        if constexpr (pin_mid) pin(acc);
    }
    {
        cplx<T> psi2[12];
        T sc2;
        LinkMat<LK, T> L2;
        load_nb<MU, PR, TH>(src, g.stride, a.nr, id, rr, psi2, sc2, lds, lbase);
        load_link<PR, LK>(a.links, g.stride, q, MU, id, L2);
        hop_dir<MU, false, LK, T, SC>(acc, psi2, L2, anti && c[3] == 0, sc2);
    }
    if constexpr (BWD_FIRST) {
        if constexpr (pin_mid) pin(acc);
        load_nb<MU, PR, TH>(src, g.stride, a.nr, iu, rr, psi, sc, lds, lbase);
        load_link<PR, LK>(a.links, g.stride, p, MU, site, L);
        hop_dir<MU, true, LK, T, SC>(acc, psi, L, anti && c[3] == g.L[3] - 1, sc);
    }
    if constexpr (pin_end) pin(acc);
}

template <int PR, int LK, int DIAG, bool INV, bool NORM, bool LO, bool UPD = false, int BM = 0, int FM = 0,
          bool NT = true>
__device__ __forceinline__ double dslash_epilogue(const DslashParams& a, int p, int site, int r,
                                                  const cplx<typename Prec<PR>::T> acc[12], float ual = 0.f,
                                                  double al = 0.0, double* sums = nullptr);

// NORM (low precision only): returns |v|^2 of the site's output as computed,
// before rounding to the storage precision; else 0.  A template parameter, so
// kernels without it compile as if the sum did not exist.  LO: lane r has its
// own kappa and clover blocks (a.lane_ops); also a template parameter.  UPD:
// the fused mixed-CG update with step ual (a.upd_*): returns the site's
// |r_s|^2 after it, and stores no output.
// FM: a fused step of the FP64 solvers (F64_*), with step al, its terms added to
// sums.  NT: FP64 blocks stream past the caches (no other lane reads them).
template <int PR, int LK, int DIAG, bool INV, bool NORM = false, bool LO = false, bool UPD = false, int BM = 0,
          int FM = 0, bool NT = true, int TH = LYM_DSLASH_THREADS>
__device__ __forceinline__ double dslash_site(const DslashParams& a, int p, int site, int r, float ual = 0.f,
                                              const cplx<double>* lds = nullptr, int lbase = 0, double al = 0.0,
                                              double* sums = nullptr) {
    typedef typename Prec<PR>::T T;
    int c[4];
    eo_coords(a.g, p, site, c);
    cplx<T> acc[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) acc[k] = mk((T)0, (T)0);
    if (LYM_ALT_ORDER && a.parity < 0 && p == 1) {
        hop_pair<0, PR, LK, true>(a, p, site, r, c, acc);
        hop_pair<1, PR, LK, true>(a, p, site, r, c, acc);
        hop_pair<2, PR, LK, true>(a, p, site, r, c, acc);
        hop_pair<3, PR, LK, true>(a, p, site, r, c, acc);
    } else {
        hop_pair<0, PR, LK>(a, p, site, r, c, acc);
        hop_pair<1, PR, LK>(a, p, site, r, c, acc);
        hop_pair<2, PR, LK, false, TH>(a, p, site, r, c, acc, lds, lbase);
        hop_pair<3, PR, LK, false, TH>(a, p, site, r, c, acc, lds, lbase);
    }
    return dslash_epilogue<PR, LK, DIAG, INV, NORM, LO, UPD, BM, FM, NT>(a, p, site, r, acc, ual, al, sums);
}

// The site's output from its hopping sum acc: v = diag(psi_x) + hop_sign
// (-kappa acc), then R^-1, gamma5, the axpy and the store (the value
// returned is as for dslash_site)
template <int PR, int LK, int DIAG, bool INV, bool NORM, bool LO, bool UPD, int BM, int FM, bool NT>
__device__ __forceinline__ double dslash_epilogue(const DslashParams& a, int p, int site, int r,
                                                  const cplx<typename Prec<PR>::T> acc[12], float ual, double al64,
                                                  double* sums) {
    typedef typename Prec<PR>::T T;
    typedef typename Prec<PR>::S S;
    const int ST = a.g.stride;
    const double kap = LO ? a.kappa_dev[r] : (a.kappa_dev ? *a.kappa_dev : a.kappa);
    const T hk = (T)(-kap * a.hop_sign);
    constexpr int BK_A = LK >= 2 ? BLK_A_REAL : BLK_A, BK_I = LK >= 2 ? BLK_INV_REAL : BLK_INV;
    // this lane's clover blocks
    const void* Ab_ = a.A;
    const void* Ai_ = a.Ainv;
    const float* Asc_ = a.A_sc;
    const float* Aisc_ = a.Ainv_sc;
    if constexpr (LO) {
        // lanes of one kappa share a block set
        const int bs = a.lane_set ? a.lane_set[r] : r;
        Ab_ = reinterpret_cast<const char*>(a.A) + bs * a.A_lane_bytes;
        Ai_ = reinterpret_cast<const char*>(a.Ainv) + bs * a.Ainv_lane_bytes;
        if constexpr (PR == 2) {
            Asc_ = a.A_sc + bs * a.Asc_lane;
            Aisc_ = a.Ainv_sc + bs * a.Ainvsc_lane;
        }
    }
    cplx<T> v[12];
    if constexpr (DIAG == 0) {
#pragma unroll
        for (int k = 0; k < 12; ++k) v[k] = hk * acc[k];
    } else if constexpr (DIAG == 2 && PR >= 1) {
        // the field's FP16 scale on the 12 outputs
        cplx<T> s[12], t[12];
        T scp;
        load_spinor_unscaled<PR>(SpinorRef<PR>{reinterpret_cast<const S*>(a.diag_in[p]), a.diag_sc[p]}, ST, a.nr,
                                 site, r, s, scp);
        const T sc = PR == 2 ? (T)Asc_[(size_t)p * ST + site] : (T)1;
        block_apply_at<PR, BK_A>(Ab_, 4, ST, 2 * p, site, sc, s, t);
        block_apply_at<PR, BK_A>(Ab_, 4, ST, 2 * p + 1, site, sc, s + 6, t + 6);
        if constexpr (PR == 2) {
#pragma unroll
            for (int k = 0; k < 12; ++k) t[k] = scp * t[k];
        }
#pragma unroll
        for (int k = 0; k < 12; ++k) v[k] = axpy1(hk, acc[k], t[k]);
    } else {
        cplx<T> s[12];
        load_spinor<PR>(SpinorRef<PR>{lane_base<PR>(a.diag_in[p], a.diag_lane, r), a.diag_sc[p]}, ST, a.nr,
                        site, field_rhs<PR>(r), s);
        if constexpr (DIAG == 2) {
            cplx<T> t[12];
            block_apply_at<PR, BK_A, NT>(Ab_, 4, ST, 2 * p, site, (T)1, s, t);
            block_apply_at<PR, BK_A, NT>(Ab_, 4, ST, 2 * p + 1, site, (T)1, s + 6, t + 6);
#pragma unroll
            for (int k = 0; k < 12; ++k) v[k] = axpy1(hk, acc[k], t[k]);
        } else {
#pragma unroll
            for (int k = 0; k < 12; ++k) v[k] = axpy1(hk, acc[k], s[k]);
        }
    }
    if constexpr (INV) {
        cplx<T> t[12];
        const T sc = PR == 2 ? (T)Aisc_[site] : (T)1;
        block_apply_at<PR, BK_I, NT || PR != 0>(Ai_, 2, ST, 0, site, sc, v, t);
        block_apply_at<PR, BK_I, NT || PR != 0>(Ai_, 2, ST, 1, site, sc, v + 6, t + 6);
#pragma unroll
        for (int k = 0; k < 12; ++k) v[k] = t[k];
    }
    if (a.gamma5) {
#pragma unroll
        for (int k = 6; k < 12; ++k) v[k] = -v[k];
    }
    if (a.v2[p]) {
        cplx<T> w[12];
        load_spinor<PR, true>(SpinorRef<PR>{reinterpret_cast<const S*>(a.v2[p]), a.v2_sc[p]}, ST, a.nr, site,
                              field_rhs<PR>(r), w);
        const cplx<T> al = mk((T)a.alpha.re, (T)a.alpha.im);
#pragma unroll
        for (int k = 0; k < 12; ++k) cfma(v[k], al, w[k]);
    }
    if constexpr (BM == 2) {
        // batch lane r: x_s += alpha_r p, r_s -= alpha_r v (v in FP32, never
        // rounded to storage), the site's |r_s|^2 to bsite
        static_assert(PR >= 1, "the fused update is the mixed-precision solver's");
        const float al = (float)a.balpha[r];
        cplx<T> pv[12];
        load_spinor<PR>(SpinorRef<PR>{reinterpret_cast<const S*>(a.upd_p[p]), a.upd_p_sc[p]}, ST, a.nr, site, r, pv);
        cplx<float>* xs = reinterpret_cast<cplx<float>*>(a.upd_xs[p]);
        cplx<float>* rs = reinterpret_cast<cplx<float>*>(a.upd_rs[p]);
        const size_t o = (size_t)site * a.nr + r, ks = (size_t)ST * a.nr;
        double n2[6] = {0, 0, 0, 0, 0, 0};  // per pair of components, as the one-wave-per-direction form sums them
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            const cplx<float> rr = axpy1(-al, v[k], rs[k * ks + o]);
            xs[k * ks + o] = axpy1(al, pv[k], xs[k * ks + o]);
            rs[k * ks + o] = rr;
            n2[k / 2] = norm_acc(mk((double)rr.re, (double)rr.im), n2[k / 2]);
        }
        a.bsite[p][o] = ((((n2[0] + n2[1]) + n2[2]) + n2[3]) + n2[4]) + n2[5];
        return 0;
    }
    if constexpr (UPD) {
        // x_s += alpha p, r_s -= alpha v (v in FP32, never rounded to storage)
        static_assert(PR >= 1, "the fused update is the mixed-precision solver's");
        cplx<T> pv[12];
        load_spinor<PR>(SpinorRef<PR>{reinterpret_cast<const S*>(a.upd_p[p]), a.upd_p_sc[p]}, ST, 1, site, 0, pv);
        cplx<float>* xs = reinterpret_cast<cplx<float>*>(a.upd_xs[p]);
        cplx<float>* rs = reinterpret_cast<cplx<float>*>(a.upd_rs[p]);
        double n2 = 0;
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            cplx<float> x = fld<cplx<float>>(xs + (size_t)k * ST, (unsigned)site);
            cplx<float> rr = fld<cplx<float>>(rs + (size_t)k * ST, (unsigned)site);
            x = x + ual * pv[k];
            rr = rr - ual * v[k];
            fst<cplx<float>, false>(xs + (size_t)k * ST, (unsigned)site, x);
            fst<cplx<float>, false>(rs + (size_t)k * ST, (unsigned)site, rr);
            n2 += (double)rr.re * rr.re + (double)rr.im * rr.im;
        }
        return n2;
    }
    if constexpr (FM != F64_STORE) {
        static_assert(PR == 0 && !NORM && !LO && !UPD && BM == 0, "the FP64 solvers' fused steps: one RHS");
#pragma unroll
        for (int k = 0; k < 12; ++k) f64_step<FM>(a, p, k, (unsigned)site, al64, v[k], sums);
        if constexpr (FM == F64_CG) return 0;
    }
    store_spinor<PR>(SpinorOut<PR>{const_cast<S*>(lane_base<PR>(a.out[p], a.out_lane, r)), a.out_sc[p]}, ST,
                     a.nr, site, field_rhs<PR>(r), v);
    if constexpr (BM == 1) {  // lane r's |v|^2 at this site: the 24 squares in FP32
        float n2[2] = {0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 12; ++k) n2[k / 6] = norm_acc(v[k], n2[k / 6]);
        a.bsite[p][(size_t)site * a.nr + r] = (double)(n2[0] + n2[1]);
    }
    if constexpr (NORM) {  // the site's 24 squares in FP32, the sum over sites in FP64
        float n2 = 0.f;
#pragma unroll
        for (int k = 0; k < 12; ++k) n2 += v[k].re * v[k].re + v[k].im * v[k].im;
        return (double)n2;
    }
    return 0;
}

// Sums of N values over the workgroup (blockDim.x a multiple of 64, at most
// 1024), in one fixed order; thread 0 writes total k to out[k * stride + blockIdx.x].
// Every thread of the workgroup must call it.
template <int N>
__device__ __forceinline__ void block_sums_store(const double v[N], double* out, size_t stride) {
    __shared__ double sh[N][16];
#pragma unroll
    for (int k = 0; k < N; ++k) {
        double t = v[k];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
        if ((threadIdx.x & 63) == 0) sh[k][threadIdx.x >> 6] = t;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            double t = 0;
            for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += sh[k][w];
            out[k * stride + blockIdx.x] = t;
        }
    }
}
__device__ __forceinline__ void block_sum_store(double v, double* out) { block_sums_store<1>(&v, out, 0); }

// The fused update's step: alpha = rr / (sum of the n <p, Ap> partials), folded
// by every workgroup in one fixed order (so all get the same alpha); workgroup 0
// stores alpha and rr_prev = rr in the state (ST: MCGState, or CGState for the
// FP64 CG).  Every thread of the workgroup must call it.
template <class ST>
__device__ __forceinline__ double upd_alpha(const DslashParams& a) {
    __shared__ double sh[16];
    double v = 0;
    for (int k = (int)threadIdx.x; k < a.upd_ndot; k += (int)blockDim.x) v += a.upd_dot[k];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) t += sh[w];
    ST* st = reinterpret_cast<ST*>(a.upd_state);
    const double rr = state_rr(st);
    const double alpha = rr / t;
    __syncthreads();  // every thread has read rr before workgroup 0 moves it to rr_prev
    if (blockIdx.x == 0 && threadIdx.x == 0) set_alpha(st, alpha, rr);
    return alpha;
}

// NORM: also the per-workgroup output norms (a.norm_partials); LO: per-lane
// operators; UPD: the fused mixed-CG update instead of the output store
template <int PR, int LK, int DIAG, bool INV, bool NORM = false, bool LO = false, bool UPD = false, int BM = 0>
__global__ __launch_bounds__(LYM_DSLASH_THREADS) LYM_OCC void k_dslash(DslashParams a) {
    static_assert(!NORM || PR >= 1, "output norms are the low-precision stencil's");
    static_assert(!(NORM && UPD), "one per-workgroup sum per launch");
    if (a.skip && *a.skip) return;
    const BlockSweep b = block_sweep(a);
    const int ls = (int)threadIdx.x / a.nr, r = (int)threadIdx.x - ls * a.nr;
    if constexpr (UPD) {
        // one RHS, no lane flags: every thread holds a site slot and reaches the sums
        const float ual = (float)upd_alpha<MCGState>(a);
        double n2 = 0;
        for (int lb = b.lo + b.k; lb < b.hi; lb += b.nphys) {
            int p, bi;
            block_of(a, b, lb, p, bi);
            const int site = bi * a.spb + (int)threadIdx.x;
            if (site < a.g.Vh) n2 += dslash_site<PR, LK, DIAG, INV, false, false, true>(a, p, site, 0, ual);
        }
        block_sum_store(n2, a.upd_rpart);
    } else if constexpr (!NORM) {
        if (ls >= a.spb) return;
        if (a.lane_flags && a.lane_flags[r] == a.lane_skip_value) return;
        for (int lb = b.lo + b.k; lb < b.hi; lb += b.nphys) {
            int p, bi;
            block_of(a, b, lb, p, bi);
            const int site = bi * a.spb + ls;
            if (site < a.g.Vh) dslash_site<PR, LK, DIAG, INV, false, LO, false, BM>(a, p, site, r);
        }
    } else {
        // one RHS, no lane flags (the launcher's condition for output norms):
        // every thread holds a site slot, and every thread reaches the sum
        double n2 = 0;
        for (int lb = b.lo + b.k; lb < b.hi; lb += b.nphys) {
            int p, bi;
            block_of(a, b, lb, p, bi);
            const int site = bi * a.spb + (int)threadIdx.x;
            if (site < a.g.Vh) n2 += dslash_site<PR, LK, DIAG, INV, true>(a, p, site, 0);
        }
        block_sum_store(n2, a.norm_partials);
    }
}

// FP64, one thread per site (spb == TH): each site
// block first copies the other parity's spinors of the same block index --
// with t fastest, the z and t neighbours of most of the block's sites -- into
// LDS, coalesced, once; those hops then read LDS instead of issuing four
// reads of every such spinor to L2.  Measured against reading them from L2:
// 16^3x32 full apply 3 % faster, even-odd launches 2 %, 32^3x64 full apply 5 %
// (same bits: only where the operands come from changes).  Filling the copy with
// direct global-to-LDS loads instead of through registers, and a second copy
// filled for the next block while the current one computes, were measured too:
// the first the same, the second 15 % slower on 16^3x32.
// FM: a fused step of the FP64 solvers; its terms' per-workgroup sums go to
// a.upd_rpart.  LN: over lanes; LO: per-lane operators.
template <int LK, int DIAG, bool INV, int FM = 0, int TH = LYM_DSLASH_THREADS>
__global__ __launch_bounds__(TH) LYM_OCC void k_dslash_stg(DslashParams a) {
    __shared__ cplx<double> stg[12 * TH];
    if (a.skip && *a.skip) return;
    const BlockSweep b = block_sweep(a);
    const int t = (int)threadIdx.x;
    double al = 0, sums[3] = {0, 0, 0};
    if constexpr (FM == F64_CG) al = upd_alpha<CGState>(a);
    for (int lb = b.lo + b.k; lb < b.hi; lb += b.nphys) {
        int p, bi;
        block_of(a, b, lb, p, bi);
        const int base = bi * TH;
        __syncthreads();  // the previous block's reads of stg are done
        if (base + t < a.g.Vh) {
            const zd* src = reinterpret_cast<const zd*>(a.in[p ^ a.g.tsh]);
#pragma unroll
            for (int k = 0; k < 12; ++k)
                stg[k * TH + t] = fld<zd>(src + (size_t)k * a.g.stride, (unsigned)(base + t));
        }
        __syncthreads();
        const int site = base + t;
        if (site < a.g.Vh)
            dslash_site<0, LK, DIAG, INV, false, false, false, 0, FM, true, TH>(a, p, site, 0, 0.f, stg, base, al, sums);
    }
    if constexpr (FM == F64_DOT) block_sums_store<3>(sums, a.upd_rpart, a.part_stride);
    else if constexpr (FM != F64_STORE) block_sums_store<1>(sums, a.upd_rpart, 0);
}

// The same over lanes: a workgroup holds 64 sites of LANE_WAVES (or fewer) lanes, a
// wave each, so that the waves that read a site's links and blocks do so from one
// CU's cache; a wave stages its own lane's spinors and waits for no other.  Against
// workgroups of 256 sites of one lane, whose lanes shared links in the L2 only: 32^3x64
// propagator 625 -> 597 ms (4 RHS at a time 654 -> 612), served burst 38.4 -> 37.6 ms.
// Eight waves to a workgroup: 610 and 38.9.
template <int LK, int DIAG, bool INV, bool LO>
__global__ __launch_bounds__(64 * LANE_WAVES) LYM_OCC void k_dslash_lanes(DslashParams a) {
    __shared__ cplx<double> stg_all[LANE_WAVES * 12 * 64];
    if (a.skip && *a.skip) return;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), nw = (int)blockDim.x >> 6;
    int bx, gd, lane;
    if (!lane_of_block(a, nw, w, bx, gd, lane)) return;
    cplx<double>* stg = stg_all + w * (12 * 64);
    const BlockSweep b = block_sweep_at(a, bx, gd);
    const int t = (int)threadIdx.x & 63;
    int p, bi;
    if (b.lo + b.k >= b.hi) return;
    (void)block_of_at(a, b, b.lo + b.k, bx, p, bi);
    const int base = bi * 64, site = base + t;
    if (site < a.g.Vh) {
        const zd* src = lane_base<0>(a.in[p ^ a.g.tsh], a.in_lane, lane);
#pragma unroll
        for (int k = 0; k < 12; ++k) stg[k * 64 + t] = fld<zd>(src + (size_t)k * a.g.stride, (unsigned)site);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (site < a.g.Vh)
        dslash_site<0, LK, DIAG, INV, false, LO, false, 0, F64_STORE, false, 64>(a, p, site, lane, 0.f, stg, base);
}

// ---------------------------------------------------------------- two threads per site (FP32/FP16)
// Split form of the single-RHS low-precision stencil: a workgroup holds its
// sites twice.  The waves of the first half take the x and y hops of every
// site, those of the second half the z and t hops; the halves swap, through
// LDS, the partial sums of the chirality the other half finishes, and each
// half applies the diagonal, R^-1, gamma5, the axpy and the store to one
// chirality (spins 0,1 or 2,3: the clover blocks are chiral, so the epilogue
// splits exactly).  An FP16 site's scale is the largest component of both
// halves, also swapped through LDS.  Twice the waves per site block hide the
// load latency where one thread per site leaves one wave per SIMD.
template <int PR, int LK, int DIAG, bool INV>
__device__ __forceinline__ void epilogue_half_lp(const DslashParams& a, int p, int site, int r, int h,
                                                 const cplx<float> u[6], cplx<float> v[6]) {
    typedef float T;
    typedef typename Prec<PR>::S S;
    const int ST = a.g.stride;
    const size_t ks = (size_t)ST * a.nr;
    const unsigned o = (unsigned)site * (unsigned)a.nr + (unsigned)r;
    const double kap = a.kappa_dev ? *a.kappa_dev : a.kappa;
    const T hk = (T)(-kap * a.hop_sign);
    if constexpr (DIAG == 0) {
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] = hk * u[k];
    } else {
        S e[6];
        load_half_lp<PR>(reinterpret_cast<const S*>(a.diag_in[p]), ks, o, h, e);
        const T scp = PR == 2 ? fld<float>(a.diag_sc[p], o) : (T)1;
        cplx<T> s6[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) s6[k] = to_c<PR>(e[k]);
        if constexpr (DIAG == 2) {
            const T sc = PR == 2 ? (T)a.A_sc[(size_t)p * ST + site] : (T)1;
            cplx<T> t[6];
            block_apply_at<PR, LK >= 2 ? BLK_A_REAL : BLK_A>(a.A, 4, ST, 2 * p + h, site, sc, s6, t);
#pragma unroll
            for (int k = 0; k < 6; ++k) v[k] = axpy1(hk, u[k], PR == 2 ? scp * t[k] : t[k]);
        } else {
#pragma unroll
            for (int k = 0; k < 6; ++k) v[k] = scp * s6[k] + hk * u[k];
        }
    }
    if constexpr (INV) {
        const T sc = PR == 2 ? (T)a.Ainv_sc[site] : (T)1;
        cplx<T> t[6];
        block_apply_at<PR, LK >= 2 ? BLK_INV_REAL : BLK_INV>(a.Ainv, 2, ST, h, site, sc, v, t);
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] = t[k];
    }
    if (a.gamma5 && h) {
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] = -v[k];
    }
    if (a.v2[p]) {
        S e[6];
        load_half_lp<PR, true>(reinterpret_cast<const S*>(a.v2[p]), ks, o, h, e);
        const T sc2 = PR == 2 ? fld<float>(a.v2_sc[p], o) : (T)1;
        const cplx<T> al = mk((T)a.alpha.re, (T)a.alpha.im);
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] = v[k] + al * (sc2 * to_c<PR>(e[k]));
    }
}

// blockDim.x = 2 * TH, TH a multiple of 64 (the launcher's thread count), so
// every wave lies in one half.  Every thread reaches both barriers of every
// block of the sweep (invalid lanes carry zeros and store nothing).
template <int PR, int LK, int DIAG, bool INV, bool NORM = false, bool UPD = false>
__global__ __launch_bounds__(2 * LYM_DSLASH_THREADS) LYM_OCC void k_dslash_split(DslashParams a) {
    static_assert(PR >= 1, "the split form is the low-precision stencil's");
    static_assert(!(NORM && UPD), "one per-workgroup sum per launch");
    typedef float T;
    typedef typename Prec<PR>::S S;
    __shared__ cplx<T> xch[2][6][LYM_DSLASH_THREADS];
    __shared__ float mx[2][LYM_DSLASH_THREADS];
    if (a.skip && *a.skip) return;
    const BlockSweep b = block_sweep(a);
    const int TH = (int)blockDim.x >> 1;
    const int h = __builtin_amdgcn_readfirstlane((int)threadIdx.x >= TH ? 1 : 0);
    const int tl = (int)threadIdx.x - h * TH;
    const int ls = tl / a.nr, r = tl - ls * a.nr;
    const bool lane_ok = ls < a.spb && !(a.lane_flags && a.lane_flags[r] == a.lane_skip_value);
    const size_t ks = (size_t)a.g.stride * a.nr;
    [[maybe_unused]] double n2 = 0;
    [[maybe_unused]] float ual = 0.f;
    if constexpr (UPD) ual = (float)upd_alpha<MCGState>(a);
    for (int lb = b.lo + b.k; lb < b.hi; lb += b.nphys) {
        int p, bi;
        block_of(a, b, lb, p, bi);
        const int site = bi * a.spb + ls;
        const bool ok = lane_ok && site < a.g.Vh;
        cplx<T> acc[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) acc[k] = mk((T)0, (T)0);
        if (ok) {
            int c[4];
            eo_coords(a.g, p, site, c);
            if (h == 0) {
                hop_pair<0, PR, LK>(a, p, site, r, c, acc);
                hop_pair<1, PR, LK>(a, p, site, r, c, acc);
            } else {
                hop_pair<2, PR, LK>(a, p, site, r, c, acc);
                hop_pair<3, PR, LK>(a, p, site, r, c, acc);
            }
        }
        // (constant indices only: a select between acc[k] and acc[6 + k] would
        // become a dynamic index and put the accumulator in scratch memory)
        if (h == 0) {
#pragma unroll
            for (int k = 0; k < 6; ++k) xch[0][k][tl] = acc[6 + k];
        } else {
#pragma unroll
            for (int k = 0; k < 6; ++k) xch[1][k][tl] = acc[k];
        }
        __syncthreads();
        cplx<T> u[6], v[6];
        if (h == 0) {
#pragma unroll
            for (int k = 0; k < 6; ++k) u[k] = acc[k] + xch[1][k][tl];
        } else {
#pragma unroll
            for (int k = 0; k < 6; ++k) u[k] = acc[6 + k] + xch[0][k][tl];
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] = mk((T)0, (T)0);
        if (ok) epilogue_half_lp<PR, LK, DIAG, INV>(a, p, site, r, h, u, v);
        if constexpr (NORM) {  // invalid lanes hold zeros
            float h2 = 0.f;
#pragma unroll
            for (int k = 0; k < 6; ++k) h2 += v[k].re * v[k].re + v[k].im * v[k].im;
            n2 += (double)h2;
        }
        const unsigned o = (unsigned)site * (unsigned)a.nr + (unsigned)r;
        S e[6];
        if constexpr (UPD) {
            // x_s += alpha p, r_s -= alpha v on this half's components 6 h + k
            if (ok) {
                load_half_lp<PR>(reinterpret_cast<const S*>(a.upd_p[p]), ks, o, h, e);
                const T psc = PR == 2 ? fld<float>(a.upd_p_sc[p], o) : (T)1;
                const int ST = a.g.stride;
                cplx<float>* xs = reinterpret_cast<cplx<float>*>(a.upd_xs[p]) + (size_t)(6 * h) * ST;
                cplx<float>* rs = reinterpret_cast<cplx<float>*>(a.upd_rs[p]) + (size_t)(6 * h) * ST;
#pragma unroll
                for (int k = 0; k < 6; ++k) {
                    cplx<float> x = fld<cplx<float>>(xs + (size_t)k * ST, (unsigned)site);
                    cplx<float> rr = fld<cplx<float>>(rs + (size_t)k * ST, (unsigned)site);
                    x = x + ual * (psc * to_c<PR>(e[k]));
                    rr = rr - ual * v[k];
                    fst<cplx<float>, false>(xs + (size_t)k * ST, (unsigned)site, x);
                    fst<cplx<float>, false>(rs + (size_t)k * ST, (unsigned)site, rr);
                    n2 += (double)rr.re * rr.re + (double)rr.im * rr.im;
                }
            }
            __syncthreads();  // every xch read of this block is done before the next block writes it
        } else if constexpr (PR == 2) {
            float m = 0.f;
#pragma unroll
            for (int k = 0; k < 6; ++k) m = fmaxf(m, fmaxf(fabsf(v[k].re), fabsf(v[k].im)));
            mx[h][tl] = m;
            __syncthreads();  // also: every xch read of this block is done
            m = fmaxf(mx[0][tl], mx[1][tl]);
            const float inv = fp16_site_inv(m);
#pragma unroll
            for (int k = 0; k < 6; ++k) e[k] = from_c<PR>(inv * v[k]);
            if (ok) {
                store_half_lp<PR>(reinterpret_cast<S*>(a.out[p]), ks, o, h, e);
                if (h == 0) fst<float, false>(a.out_sc[p], o, m);
            }
        } else {
            __syncthreads();  // every xch read of this block is done before the next block writes it
#pragma unroll
            for (int k = 0; k < 6; ++k) e[k] = from_c<PR>(v[k]);
            if (ok) store_half_lp<PR>(reinterpret_cast<S*>(a.out[p]), ks, o, h, e);
        }
    }
    if constexpr (NORM) block_sum_store(n2, a.norm_partials);  // every thread reaches it
    if constexpr (UPD) block_sum_store(n2, a.upd_rpart);
}

// ---------------------------------------------------------------- multi-RHS FP16 stencil on the matrix cores
// k_dslash_mfma: the hopping term of a batch of nr = 2, 4 or 8 right-hand
// sides per site (FP16 storage, SU(3) links with all three rows) with the link
// product on the matrix cores, one v_mfma_f32_16x16x16_f16 per hop and site:
//   C (16 x 16) = A (16 x 16) . B (16 x 16), FP16 inputs, FP32 products and sums
//   B column n = 2 r + h (RHS r, spin half h = 0, 1); B rows k 0-5: the
//     neighbour spinor's spin h, colour k / 2, (re, im); k 6-11: its partner
//     spin P_h of the direction (negated for h = 1 when c_1 = -c_0); 12-15 zero
//   A rows m 0-5: the direct output (spin h), colour m / 2, (re, im); m 6-11:
//     the partner output (spin P_h); 12-15 zero.  A is the real form of the
//     3x3 blocks  forward: direct [U | c U], partner [c* U | U];
//                 backward: direct [U+ | -c U+], partner [-c* U+ | U+]
//     with c = i^C0 of the direction,
// so the projection (1 -+ gamma_mu), the link multiply and the
// reconstruction all happen inside the MFMA on the stored FP16 values, with
// no rounding before the FP32 sums.  The neighbour's FP16 scale (one per site
// and RHS, i.e. per column), the boundary sign and the sign of partner rows
// for h = 1 multiply C in FP32.  Lane l holds A row l % 16 and B column
// l % 16 at k = 4 (l / 16) + 0..3, and C column l % 16, rows 4 (l / 16) +
// 0..3 (checked on the device).  A wave works through its sites one at a
// time (the site, its neighbours and the link bases are wave-uniform); the
// hopping sums go through LDS to one thread per (site, RHS), which runs the
// epilogue of the VALU stencil (diagonal, R^-1, gamma5, axpy, FP16 store).
typedef _Float16 hv4 __attribute__((ext_vector_type(4)));
typedef float fv4 __attribute__((ext_vector_type(4)));

// z i^p on FP16 values (exact: a swap and sign changes)
__device__ __forceinline__ h2_t mul_ip(h2_t z, int p) {
    const bool sw = (p & 1) != 0;
    _Float16 x = sw ? z.y : z.x, y = sw ? z.x : z.y;
    if (p == 1 || p == 2) x = -x;
    if (p >= 2) y = -y;
    h2_t o;
    o.x = x;
    o.y = y;
    return o;
}

constexpr int MFMA_LDS_STRIDE = 26;  // floats per (site, RHS) slot: 24 used, padded against bank conflicts

// lane constants of the MFMA stencil
struct MfmaLane {
    int rr, hh;         // B/C column: RHS and spin half
    bool bval;          // column rr < nr and k-group < 3: this lane loads B
    bool aval;          // A row < 12 and k-group < 3: this lane loads A
    int arow, aore;     // A row: 0 direct, 1 partner; 0 real row, 1 imaginary row
    bool partP[2];      // A/B k slot s: colour block of the partner spin (else of spin h)
    // link entry of slot s of link li: entry (li << lsh) + lofs of the packed field
    unsigned lofs_f[2], lofs_b[2], lsh_f[2], lsh_b[2];
    int kgrp;           // k-group l / 16
};

// entry k of a packed FP16 link: vectors of entries 0-3 and 4-7, then entry 8
__device__ __forceinline__ void mfma_entry(int stride, int k, unsigned& ofs, unsigned& sh) {
    ofs = k < 8 ? (unsigned)(k >> 2) * 32u * (unsigned)stride + (k & 3) : 64u * (unsigned)stride;
    sh = k < 8 ? 2 : 0;
}

template <int MU>
__device__ __forceinline__ int mfma_phase(const MfmaLane& L, int s, bool fwd) {
    constexpr int C0 = Dir<MU>::C0;
    if (L.arow == 0 && L.partP[s]) return fwd ? C0 : (C0 + 2) & 3;
    if (L.arow == 1 && !L.partP[s]) return fwd ? (4 - C0) & 3 : (6 - C0) & 3;
    return 0;
}

// Operands of one hop (direction MU, forward or backward) of the wave's
// current site: A (the link block), B (the neighbour spinor's components) and
// the neighbour's FP16 scale.  Branch-free: lanes without an operand load a
// valid address and select zero, so the loads of all eight hops of a site can
// be issued before the first MFMA waits on them.  lsite: the link's site
// index on parity lp; nb: the neighbour spinor's index on parity q
template <int MU, bool FWD>
__device__ __forceinline__ void mfma_load(const DslashParams& a, const MfmaLane& L, int lp, int lsite, int q, int nb,
                                          const unsigned sofs[2], bool use_b, hv4& Av, hv4& Bv, float& sc) {
    const int ST = a.g.stride;
    const unsigned li = (unsigned)((lp * 4 + MU) * ST + lsite);  // the packed link: entries 0-3, 4-7, 8
    const h2_t* lb = reinterpret_cast<const h2_t*>(a.links);
    const h2_t* sb = reinterpret_cast<const h2_t*>(a.in[q]) + (size_t)nb * a.nr * 4;
    constexpr bool SIGN1 = Dir<MU>::C1 != Dir<MU>::C0;  // c_1 = -c_0
    const _Float16 hz = (_Float16)0;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const unsigned lo = FWD ? L.lofs_f[s] : L.lofs_b[s], sh = FWD ? L.lsh_f[s] : L.lsh_b[s];
        h2_t z = fld<h2_t>(lb, L.aval ? (li << sh) + lo : 0u);
        if (!FWD) z.y = -z.y;
        z = mul_ip(z, mfma_phase<MU>(L, s, FWD));
        Av[2 * s] = L.aval ? (L.aore ? z.y : z.x) : hz;
        Av[2 * s + 1] = L.aval ? (L.aore ? z.x : (_Float16)(-z.y)) : hz;
        h2_t v = fld<h2_t>(sb, use_b ? sofs[s] : 0u);
        if (SIGN1 && L.hh && L.partP[s]) {
            v.x = -v.x;
            v.y = -v.y;
        }
        Bv[2 * s] = use_b ? v.x : hz;
        Bv[2 * s + 1] = use_b ? v.y : hz;
    }
    const float f = fld<float>(a.in_sc[q] + (size_t)nb * a.nr, use_b ? (unsigned)L.rr : 0u);
    sc = use_b ? f : 0.f;
}

// G += f * (A . B) for one hop: f = the neighbour's scale, with the boundary
// sign and, for partner rows of columns h = 1 where c_1 = -c_0, a minus sign
template <int MU>
__device__ __forceinline__ void mfma_acc(const MfmaLane& L, const hv4& Av, const hv4& Bv, float sc, bool flip,
                                         fv4& G) {
    constexpr bool SIGN1 = Dir<MU>::C1 != Dir<MU>::C0;
    const fv4 zero = {0.f, 0.f, 0.f, 0.f};
    const fv4 Cv = __builtin_amdgcn_mfma_f32_16x16x16f16(Av, Bv, zero, 0, 0, 0);
    const float f = flip ? -sc : sc;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        // C row 4 k + t is a partner row for k = 1, t >= 2 and for k = 2
        const bool prow = L.kgrp == 2 || (L.kgrp == 1 && t >= 2);
        G[t] += ((SIGN1 && L.hh && prow) ? -f : f) * Cv[t];
    }
}

template <int DIAG, bool INV, bool LO>
__global__ __launch_bounds__(LYM_DSLASH_THREADS) void k_dslash_mfma(DslashParams a) {
    __shared__ float accs[LYM_DSLASH_THREADS * MFMA_LDS_STRIDE];
    if (a.skip && *a.skip) return;
    const BlockSweep b = block_sweep(a);
    const int nr = a.nr, spb = a.spb;
    const int lane = (int)threadIdx.x & 63, wv = (int)threadIdx.x >> 6;
    const int spw = 64 / nr;  // sites per wave (nr divides 64)
    MfmaLane L;
    {
        const int n = lane & 15;
        L.kgrp = lane >> 4;
        L.rr = n >> 1;
        L.hh = n & 1;
        L.bval = L.rr < nr && L.kgrp < 3;
        L.arow = n < 6 ? 0 : 1;
        L.aore = n & 1;
        L.aval = n < 12 && L.kgrp < 3;
        const int ai = (n % 6) >> 1;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const int idx = 2 * L.kgrp + s;  // 0..5: (spin h, colour 0..2), then (partner, colour 0..2)
            const int j = idx % 3;
            L.partP[s] = idx >= 3;
            mfma_entry(a.g.stride, 3 * ai + j, L.lofs_f[s], L.lsh_f[s]);
            mfma_entry(a.g.stride, 3 * j + ai, L.lofs_b[s], L.lsh_b[s]);
        }
    }
    // B offsets (h2 elements from the neighbour's base) per direction and slot
    unsigned sofs[4][2];
    {
        const size_t ks = (size_t)a.g.stride * nr;
        const int P0[4] = {Dir<0>::P0, Dir<1>::P0, Dir<2>::P0, Dir<3>::P0};
        const int P1[4] = {Dir<0>::P1, Dir<1>::P1, Dir<2>::P1, Dir<3>::P1};
#pragma unroll
        for (int mu = 0; mu < 4; ++mu)
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int idx = 2 * L.kgrp + s;
                const int j = idx % 3;
                const int spin = idx < 3 ? L.hh : (L.hh ? P1[mu] : P0[mu]);
                const int comp = 3 * spin + j;  // 16-byte vector comp / 4, slot comp % 4
                sofs[mu][s] = L.kgrp < 3 ? (unsigned)(((comp >> 2) * ks + L.rr) * 4 + (comp & 3)) : 0u;
            }
    }
    const bool anti = a.g.bc_t < 0;
    const bool skip_col = L.rr < nr && a.lane_flags && a.lane_flags[L.rr] == a.lane_skip_value;
    for (int lb = b.lo + b.k; lb < b.hi; lb += b.nphys) {
        int p, bi;
        block_of(a, b, lb, p, bi);
        const int q = p ^ a.g.tsh;
        for (int sl = 0; sl < spw; ++sl) {
            const int ls = wv * spw + sl;
            const int site = __builtin_amdgcn_readfirstlane(bi * spb + ls);
            if (ls >= spb || site >= a.g.Vh) break;
            int c[4];
            eo_coords(a.g, p, site, c);
            const bool use_b = L.bval && !skip_col;
            // neighbour indices (wave-uniform) and the operands of all eight hops
            hv4 Ah[8], Bh[8];
            float sch[8];
            bool fl[8];
#define LYM_MFMA_LOAD(MU)                                                                                        \
    {                                                                                                            \
        int cu[4] = {c[0], c[1], c[2], c[3]}, cd[4] = {c[0], c[1], c[2], c[3]};                                  \
        cu[MU] = c[MU] + 1 == a.g.L[MU] ? 0 : c[MU] + 1;                                                         \
        cd[MU] = c[MU] == 0 ? a.g.L[MU] - 1 : c[MU] - 1;                                                         \
        const int iu = __builtin_amdgcn_readfirstlane(eo_index(a.g, cu[0], cu[1], cu[2], cu[3]));                \
        const int id = __builtin_amdgcn_readfirstlane(eo_index(a.g, cd[0], cd[1], cd[2], cd[3]));                \
        mfma_load<MU, true>(a, L, p, site, q, iu, sofs[MU], use_b, Ah[2 * MU], Bh[2 * MU], sch[2 * MU]);         \
        mfma_load<MU, false>(a, L, q, id, q, id, sofs[MU], use_b, Ah[2 * MU + 1], Bh[2 * MU + 1], sch[2 * MU + 1]); \
        fl[2 * MU] = MU == 3 && anti && c[3] == a.g.L[3] - 1;                                                    \
        fl[2 * MU + 1] = MU == 3 && anti && c[3] == 0;                                                           \
    }
            LYM_MFMA_LOAD(0)
            LYM_MFMA_LOAD(1)
            LYM_MFMA_LOAD(2)
            LYM_MFMA_LOAD(3)
#undef LYM_MFMA_LOAD
            fv4 G0 = {0.f, 0.f, 0.f, 0.f}, G1 = G0;
            mfma_acc<0>(L, Ah[0], Bh[0], sch[0], fl[0], G0);
            mfma_acc<0>(L, Ah[1], Bh[1], sch[1], fl[1], G0);
            mfma_acc<1>(L, Ah[2], Bh[2], sch[2], fl[2], G0);
            mfma_acc<1>(L, Ah[3], Bh[3], sch[3], fl[3], G0);
            mfma_acc<2>(L, Ah[4], Bh[4], sch[4], fl[4], G1);
            mfma_acc<2>(L, Ah[5], Bh[5], sch[5], fl[5], G1);
            mfma_acc<3>(L, Ah[6], Bh[6], sch[6], fl[6], G1);
            mfma_acc<3>(L, Ah[7], Bh[7], sch[7], fl[7], G1);
            // directions 0, 1 send the partner half of column h to spin 3 - h,
            // directions 2, 3 to spin 2 + h: the lane of column h = 0 collects
            // spin 2 (its G1, its neighbour's G0), the lane of h = 1 spin 3
            float other[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) other[t] = __shfl_xor(G0[t], 1, 64);
            if (L.bval) {
                float* slot = accs + (ls * nr + L.rr) * MFMA_LDS_STRIDE;
#pragma unroll
                for (int t = 0; t < 4; t += 2) {
                    const int m = 4 * L.kgrp + t;  // C rows m (re), m + 1 (im)
                    float re, im;
                    int comp;
                    if (m < 6) {
                        re = G0[t] + G1[t];
                        im = G0[t + 1] + G1[t + 1];
                        comp = 3 * L.hh + (m >> 1);
                    } else {
                        re = G1[t] + other[t];
                        im = G1[t + 1] + other[t + 1];
                        comp = 3 * (2 + L.hh) + ((m - 6) >> 1);
                    }
                    slot[2 * comp] = re;
                    slot[2 * comp + 1] = im;
                }
            }
        }
        __syncthreads();
        {
            const int t = (int)threadIdx.x;
            const int ls = t / nr, r = t - ls * nr;
            const int site = bi * spb + ls;
            if (ls < spb && site < a.g.Vh && !(a.lane_flags && a.lane_flags[r] == a.lane_skip_value)) {
                cplx<float> acc[12];
                const float* slot = accs + t * MFMA_LDS_STRIDE;
#pragma unroll
                for (int k = 0; k < 12; ++k) acc[k] = mk(slot[2 * k], slot[2 * k + 1]);
                (void)dslash_epilogue<2, 0, DIAG, INV, false, LO>(a, p, site, r, acc);
            }
        }
        __syncthreads();
    }
}

// one field, in workgroups of TH sites
template <int LK, int DIAG, bool INV, int TH>
static void launch_stg(const DslashParams& a, int nblocks, hipStream_t st) {
    const dim3 g(nblocks), th(TH);
    if constexpr (DIAG >= 1 && !INV) {
        switch (a.fmode) {
            case F64_NORM:
                hipLaunchKernelGGL((k_dslash_stg<LK, DIAG, INV, F64_NORM, TH>), g, th, 0, st, a);
                return;
            case F64_CG:
                hipLaunchKernelGGL((k_dslash_stg<LK, DIAG, INV, F64_CG, TH>), g, th, 0, st, a);
                return;
            case F64_DOT:
                hipLaunchKernelGGL((k_dslash_stg<LK, DIAG, INV, F64_DOT, TH>), g, th, 0, st, a);
                return;
            default: break;
        }
    }
    hipLaunchKernelGGL((k_dslash_stg<LK, DIAG, INV, F64_STORE, TH>), g, th, 0, st, a);
}
template <int LK, int DIAG, bool INV>
static void launch_f64(const DslashParams& a, int nblocks, hipStream_t st) {
    if (over_lanes(a)) {
        const int nw = lane_waves(a);
        const dim3 g(lane_grid(a, nblocks, nw)), th(64 * nw);
        if (a.lane_ops) hipLaunchKernelGGL((k_dslash_lanes<LK, DIAG, INV, true>), g, th, 0, st, a);
        else hipLaunchKernelGGL((k_dslash_lanes<LK, DIAG, INV, false>), g, th, 0, st, a);
        return;
    }
    if (a.spb == 64) launch_stg<LK, DIAG, INV, 64>(a, nblocks, st);  // plan_waves
    else launch_stg<LK, DIAG, INV, LYM_DSLASH_THREADS>(a, nblocks, st);
}

template <int PR, int LK, int DIAG, bool INV>
static void launch_lp(const DslashParams& a, int nblocks, hipStream_t st);
template <int PR, int LK, int DIAG, bool INV>
static void launch_one(const DslashParams& a, int nblocks, hipStream_t st) {
    if constexpr (PR == 0) {
        launch_f64<LK, DIAG, INV>(a, nblocks, st);
    } else {
        launch_lp<PR, LK, DIAG, INV>(a, nblocks, st);
    }
}
template <int PR, int LK, int DIAG, bool INV>
static void launch_lp(const DslashParams& a, int nblocks, hipStream_t st) {
    if constexpr (PR == 2 && LK == 0) {
        if (takes_mfma(a)) {
            if (a.lane_ops)
                hipLaunchKernelGGL((k_dslash_mfma<DIAG, INV, true>), dim3(nblocks), dim3(a.spb * a.nr), 0, st, a);
            else
                hipLaunchKernelGGL((k_dslash_mfma<DIAG, INV, false>), dim3(nblocks), dim3(a.spb * a.nr), 0, st, a);
            return;
        }
    }
    if (a.lane_ops) {  // per-lane operators: the serving engine's batches (never split, no output norms)
        if constexpr (PR >= 1 && DIAG >= 1 && !INV) {
            // with the batched solver's fused steps
            if (a.bmode == 1) {
                hipLaunchKernelGGL((k_dslash<PR, LK, DIAG, INV, false, true, false, 1>), dim3(nblocks),
                                   dim3(a.spb * a.nr), 0, st, a);
                return;
            }
            if (a.bmode == 2) {
                hipLaunchKernelGGL((k_dslash<PR, LK, DIAG, INV, false, true, false, 2>), dim3(nblocks),
                                   dim3(a.spb * a.nr), 0, st, a);
                return;
            }
        }
        hipLaunchKernelGGL((k_dslash<PR, LK, DIAG, INV, false, true>), dim3(nblocks), dim3(a.spb * a.nr), 0, st, a);
        return;
    }
    if constexpr (PR >= 1 && DIAG >= 1 && !INV) {
        // the batched solver's fused steps (one thread per (site, RHS), never split)
        if (a.bmode == 1) {
            hipLaunchKernelGGL((k_dslash<PR, LK, DIAG, INV, false, false, false, 1>), dim3(nblocks),
                               dim3(a.spb * a.nr), 0, st, a);
            return;
        }
        if (a.bmode == 2) {
            hipLaunchKernelGGL((k_dslash<PR, LK, DIAG, INV, false, false, false, 2>), dim3(nblocks),
                               dim3(a.spb * a.nr), 0, st, a);
            return;
        }
    }
    // the fused mixed-CG update and output norms: asked for only on launches
    // with a diagonal and no R^-1 (the last launch of a Schur apply, a
    // full-lattice apply)
    if constexpr (PR >= 1 && DIAG >= 1 && !INV) {
        if (a.upd_state) {
            if (a.split)
                hipLaunchKernelGGL((k_dslash_split<PR, LK, DIAG, INV, false, true>), dim3(nblocks), dim3(2 * a.split),
                                   0, st, a);
            else
                hipLaunchKernelGGL((k_dslash<PR, LK, DIAG, INV, false, false, true>), dim3(nblocks),
                                   dim3(a.spb * a.nr), 0, st, a);
            return;
        }
        if (a.norm_partials) {
            if (a.split)
                hipLaunchKernelGGL((k_dslash_split<PR, LK, DIAG, INV, true>), dim3(nblocks), dim3(2 * a.split), 0, st,
                                   a);
            else
                hipLaunchKernelGGL((k_dslash<PR, LK, DIAG, INV, true>), dim3(nblocks), dim3(a.spb * a.nr), 0, st, a);
            return;
        }
    }
    if constexpr (PR >= 1) {
        if (a.split) {
            hipLaunchKernelGGL((k_dslash_split<PR, LK, DIAG, INV>), dim3(nblocks), dim3(2 * a.split), 0, st, a);
            return;
        }
    }
    hipLaunchKernelGGL((k_dslash<PR, LK, DIAG, INV>), dim3(nblocks), dim3(a.spb * a.nr), 0, st, a);
}

template <int PR, int LK>
static void launch_lk(const DslashParams& a, int diag, bool inv, int nblocks, hipStream_t st) {
    if (diag == 0) {
        if (inv) launch_one<PR, LK, 0, true>(a, nblocks, st);
        else launch_one<PR, LK, 0, false>(a, nblocks, st);
    } else if (diag == 1) {
        if (inv) launch_one<PR, LK, 1, true>(a, nblocks, st);
        else launch_one<PR, LK, 1, false>(a, nblocks, st);
    } else {
        launch_one<PR, LK, 2, false>(a, nblocks, st);
    }
}

template <int PR>
static void launch_pr(const DslashParams& a, int link_kind, int diag, bool inv, int nblocks, hipStream_t st) {
    switch (link_kind) {
        case 0: launch_lk<PR, 0>(a, diag, inv, nblocks, st); break;
        case 1: launch_lk<PR, 1>(a, diag, inv, nblocks, st); break;
        case 2: launch_lk<PR, 2>(a, diag, inv, nblocks, st); break;
        default: launch_lk<PR, 3>(a, diag, inv, nblocks, st); break;
    }
}

int launch_dslash(DslashParams a, int link_kind, int diag, bool inv, hipStream_t st) {
    const LaunchPlan L = plan_launch(a, link_kind, diag, inv);
    if (L.form == LYM_FORM_HOP) {
        launch_dslash_hop(a, link_kind, diag, inv, L.nblocks, st);
        return L.partials;
    }
    switch (a.prec) {
        case 0: launch_pr<0>(a, link_kind, diag, inv, L.nblocks, st); break;
        case 1: launch_pr<1>(a, link_kind, diag, inv, L.nblocks, st); break;
        default: launch_pr<2>(a, link_kind, diag, inv, L.nblocks, st); break;
    }
    return L.partials;
}

}  // namespace lym
