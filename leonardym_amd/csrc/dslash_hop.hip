// dslash_hop.hip -- the stencil of dslash.hip with one wave per direction, for
// launches too small to fill the chip with one thread per site.
//
// What bounds it: with one thread per site a wave issues the loads of two hops,
// waits, and goes on to the next two, four times over, then the site diagonal;
// on a lattice that leaves one wave per SIMD or less nothing else covers those
// waits, and an 8^4 launch (9 us) is five such waits long whatever it reads.
// Here a workgroup holds up to 64 (site, RHS) lanes four times over, one wave
// per direction, plus two waves, one per chirality, that load the site's own
// operands (diagonal spinor and clover block, R^-1, the axpy operand) at the same
// time: every load of a site is in flight at once, one wait instead of five.
// The direction waves leave their two colour vectors per hop in LDS; the
// chirality waves sum the eight hops in the order of dslash.hip's accumulator and
// finish spins 0, 1 and 2, 3 (the clover blocks and R^-1 are chiral).  A site's
// operations and their order are those of the one-thread form, so outputs and a
// batch's fused steps have the same bits in both (a single launch's norms and update
// are summed in another order).  A fused update (x_s, r_s) is spread over all six waves.
//
// Measured (MI355X, against the one- or two-thread form): FP64 Wilson apply on
// 8^4 9.1 -> 5.8 us, on 8^3x16 clover 12.0 -> 6.3 us; FP64 even-odd CG iteration
// 53.7 -> 34.6 us on 8^4, 80.8 -> 67 us on 12^3x24; mixed CG iteration 47 -> 32 us
// on 8^4 and 54 -> 43 us on 12^3x24 in FP16 storage, 62 -> 48 us in FP32.  One
// wave per hop (eight and two waves) was as fast on the smallest lattices and
// 20 % slower from 12^4 on, where only one such workgroup fits a CU.
#include "lym_stencil.h"

namespace lym {

// n / d for 0 <= n < 2^27 by the reciprocal: (n + 1/2) / d lies at least
// 1 / (2 d) from an integer, far more than the rounding of the product
__device__ __forceinline__ int div_by(int n, double inv) { return (int)fma((double)n, inv, 0.5 * inv); }

__device__ __forceinline__ void eo_coords_inv(const Geom& g, const double inv[3], int p, int idx, int c[4]) {
    int r = div_by(idx, inv[2]);
    const int th = idx - r * g.Lth;
    int s = div_by(r, inv[1]);
    c[2] = r - s * g.L[2];
    c[0] = div_by(s, inv[0]);
    c[1] = s - c[0] * g.L[1];
    c[3] = (th << g.tsh) + ((c[0] + c[1] + c[2] + p) & g.tsh);
}

// One hop of a site: r[0..2], r[3..5] the link times the projected colour
// vectors; returns the factor hop_acc applies (FP16: the neighbour's scale, with
// the boundary sign; else the sign is in r and the factor unused)
template <int MU, bool FWD, int PR, int LK>
__device__ __forceinline__ typename Prec<PR>::T one_hop(const DslashParams& a, int p, int site, int r, const int c[4],
                                                        cplx<typename Prec<PR>::T> o[6]) {
    typedef typename Prec<PR>::T T;
    const Geom& g = a.g;
    const int q = p ^ g.tsh;
    int n[4] = {c[0], c[1], c[2], c[3]};
    if constexpr (FWD) n[MU] = c[MU] + 1 == g.L[MU] ? 0 : c[MU] + 1;
    else n[MU] = c[MU] == 0 ? g.L[MU] - 1 : c[MU] - 1;
    const int in = eo_index(g, n[0], n[1], n[2], n[3]);
    cplx<T> psi[12];
    T sc;
    LinkMat<LK, T> L;
    load_spinor_unscaled<PR>(SpinorRef<PR>{lane_base<PR>(a.in[q], a.in_lane, r), a.in_sc[q]}, g.stride,
                             a.nr, in, field_rhs<PR>(r), psi, sc);
    load_link<PR, LK>(a.links, g.stride, FWD ? p : q, MU, FWD ? site : in, L);
    // (the sign on the products here: one wave of four takes it, and on the projected
    // vectors it cost the fused FP64 steps 1 %)
    hop_mul<MU, FWD, LK, T, PR == 2>(psi, L, false, o, o + 3);
    const bool flip = MU == 3 && g.bc_t < 0 && c[3] == (FWD ? g.L[3] - 1 : 0);
    if constexpr (PR != 2 && MU == 3) {
        if (flip) {
#pragma unroll
            for (int k = 0; k < 6; ++k) o[k] = -o[k];
        }
    }
    return flip ? -sc : sc;
}

// what a hop contributes to chirality CH, added to u
template <int CH, int MU, bool FWD, int PR>
__device__ __forceinline__ void add_hop(cplx<typename Prec<PR>::T> u[6], const cplx<typename Prec<PR>::T>* x, int lane,
                                        typename Prec<PR>::T f) {
    typedef typename Prec<PR>::T T;
    using D = Dir<MU>;
    using H = HopPhase<MU, FWD>;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const cplx<T> r0 = x[c * HOP_LANES + lane], r1 = x[(3 + c) * HOP_LANES + lane];
        if constexpr (CH == 0) {
            hop_acc<PR == 2, T>(u[c], r0, f);
            hop_acc<PR == 2, T>(u[3 + c], r1, f);
        } else {
            hop_acc<PR == 2, T>(u[3 * (D::P0 - 2) + c], mulph<H::Q0>(r0), f);
            hop_acc<PR == 2, T>(u[3 * (D::P1 - 2) + c], mulph<H::Q1>(r1), f);
        }
    }
    // keep the LDS reads of later hops behind this one (FP32, FP16: this pair of
    // hops): all issued at once they would take the registers of another workgroup
    if constexpr (PR == 0 || !FWD) asm volatile("" ::: "memory");
}

// spins 2h, 2h + 1 of a spinor, unscaled
template <int PR, bool NT = false>
__device__ __forceinline__ void load_half(const void* base, size_t ks, unsigned o, int h,
                                          cplx<typename Prec<PR>::T> s[6]) {
    typedef typename Prec<PR>::S S;
    if constexpr (PR == 0) {
        const zd* b = reinterpret_cast<const zd*>(base) + (size_t)(6 * h) * ks;
#pragma unroll
        for (int k = 0; k < 6; ++k) s[k] = fld<zd, NT>(b + k * ks, o);
    } else {
        S e[6];
        load_half_lp<PR, NT>(reinterpret_cast<const S*>(base), ks, o, h, e);
#pragma unroll
        for (int k = 0; k < 6; ++k) s[k] = to_c<PR>(e[k]);
    }
}

// fused steps of a launch
enum { HOP_STORE = 0, HOP_NORM = 1, HOP_UPD = 2, HOP_BM1 = 3, HOP_BM2 = 4 };

// The fused update of components 2 w, 2 w + 1: x_s += alpha p, r_s -= alpha v.
// Its operands are loaded with the hops'; every wave of the workgroup takes one
// pair, so the update's streams are spread over all of them.
template <int PR>
struct UpdPair {
    cplx<float> p[2], x[2], r[2];
    __device__ __forceinline__ void load(const DslashParams& a, int par, size_t ks, unsigned o, int w) {
        typedef typename Prec<PR>::S S;
        if constexpr (PR >= 1) {
            S e[2];
            if constexpr (PR == 1) {
                const V16 v = fld<V16>(reinterpret_cast<const V16*>(a.upd_p[par]) + (size_t)w * ks, o);
                __builtin_memcpy(e, &v, 16);
            } else {
                // half of the 16-byte vector w / 2
                const V8 v = fld<V8>(reinterpret_cast<const V8*>(a.upd_p[par]) + (size_t)(w >> 1) * 2 * ks,
                                     2 * o + (unsigned)(w & 1));
                __builtin_memcpy(e, &v, 8);
            }
            const cplx<float>* xs = reinterpret_cast<const cplx<float>*>(a.upd_xs[par]) + (size_t)(2 * w) * ks;
            const cplx<float>* rs = reinterpret_cast<const cplx<float>*>(a.upd_rs[par]) + (size_t)(2 * w) * ks;
            const float sc = PR == 2 ? fld<float>(a.upd_p_sc[par], o) : 1.f;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                x[k] = fld<cplx<float>>(xs + k * ks, o);
                r[k] = fld<cplx<float>>(rs + k * ks, o);
                p[k] = to_c<PR>(e[k]);
                if constexpr (PR == 2) p[k] = sc * p[k];
            }
        }
    }
    // returns |r_s|^2 of the pair
    __device__ __forceinline__ double step(const DslashParams& a, int par, size_t ks, unsigned o, int w, float al,
                                           cplx<float> v0, cplx<float> v1) {
        cplx<float>* xs = reinterpret_cast<cplx<float>*>(a.upd_xs[par]) + (size_t)(2 * w) * ks;
        cplx<float>* rs = reinterpret_cast<cplx<float>*>(a.upd_rs[par]) + (size_t)(2 * w) * ks;
        double n2 = 0;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const cplx<float> rr = axpy1(-al, k ? v1 : v0, r[k]);
            fst<cplx<float>, false>(xs + k * ks, o, axpy1(al, p[k], x[k]));
            fst<cplx<float>, false>(rs + k * ks, o, rr);
            n2 = norm_acc(mk((double)rr.re, (double)rr.im), n2);
        }
        return n2;
    }
};

// The same for the FP64 CG (F64_CG).
struct UpdPair64 {
    zd p[2], x[2], r[2];
    __device__ __forceinline__ void load(const DslashParams& a, int par, unsigned o, int w) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const size_t c = (size_t)(2 * w + k) * a.g.stride;
            p[k] = fld<zd>(reinterpret_cast<const zd*>(a.upd_p[par]) + c, o);
            x[k] = fld<zd>(reinterpret_cast<const zd*>(a.upd_xs[par]) + c, o);
            r[k] = fld<zd>(reinterpret_cast<const zd*>(a.upd_rs[par]) + c, o);
        }
    }
    __device__ __forceinline__ double step(const DslashParams& a, int par, unsigned o, int w, double al, zd v0, zd v1) {
        double n2 = 0;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const size_t c = (size_t)(2 * w + k) * a.g.stride;
            const zd rn = axpy1(-al, k ? v1 : v0, r[k]);
            fst<zd, false>(reinterpret_cast<zd*>(a.upd_xs[par]) + c, o, axpy1(al, p[k], x[k]));
            fst<zd, false>(reinterpret_cast<zd*>(a.upd_rs[par]) + c, o, rn);
            n2 = norm_acc(rn, n2);
        }
        return n2;
    }
};

// sum over a wave, in every lane
__device__ __forceinline__ double wave_total(double v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// One workgroup: the spb sites of one block x nr right-hand sides (rhs
// fastest, spb * nr <= 64).  LO: per-lane operators.  FM: a fused step of the FP64
// solvers (F64_*).
template <int PR, int LK, int DIAG, bool INV, int MODE, bool LO, int FM = F64_STORE>
__global__ __launch_bounds__(HOP_THREADS, PR == 0 ? 3 : (PR == 1 ? 5 : 6)) void k_dslash_hop(DslashParams a) {
    typedef typename Prec<PR>::T T;
    typedef typename Prec<PR>::S S;
    static_assert(MODE == HOP_STORE || (PR >= 1 && DIAG >= 1 && !INV), "fused steps: low precision, last launch");
    static_assert(FM == F64_STORE || (PR == 0 && DIAG >= 1 && !INV && !LO), "the FP64 solvers' fused steps");
    __shared__ cplx<T> xch[8][6 * HOP_LANES];
    __shared__ float fsc[PR == 2 ? 8 : 1][HOP_LANES];
    constexpr bool UPDATE = MODE == HOP_UPD || MODE == HOP_BM2;
    __shared__ double half_sum[MODE == HOP_STORE || UPDATE ? 1 : HOP_LANES];
    __shared__ cplx<T> vout[UPDATE || FM == F64_CG ? 12 : 1][HOP_LANES];
    __shared__ double pair_sum[UPDATE ? HOP_WAVES + 2 : 1][HOP_LANES];
    __shared__ float al_sh[1];
    __shared__ double al64[1], wsum[3][HOP_WAVES + 2];
    __shared__ float half_max[PR == 2 ? 2 : 1][HOP_LANES];
    if (a.skip && *a.skip) return;
    const int lane = (int)threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    int bx = (int)blockIdx.x, gd = (int)gridDim.x, ls, r;
    if constexpr (PR == 0) {
        if (!lane_of_block(a, 1, 0, bx, gd, r)) return;
        ls = lane;
    } else {
        ls = lane / a.nr;
        r = lane - ls * a.nr;
    }
    const int lb = xcd_block(bx, gd);
    const int p = a.parity >= 0 ? a.parity : lb & 1, bi = a.parity >= 0 ? lb : lb >> 1;
    const int site = bi * a.spb + ls;
    const bool ok = ls < a.spb && site < a.g.Vh && (PR == 0 || !(a.lane_flags && a.lane_flags[r] == a.lane_skip_value));
    const int ST = a.g.stride;
    const size_t ks = (size_t)ST * a.nr;
    const unsigned o = (unsigned)site * (unsigned)a.nr + (unsigned)field_rhs<PR>(r);

    [[maybe_unused]] UpdPair<PR> up;
    if constexpr (UPDATE) {
        if (ok) up.load(a, p, ks, o, w);
    }

    if (w < HOP_WAVES) {
        if (ok) {
            int c[4];
            eo_coords_inv(a.g, a.inv_ext, p, site, c);
            cplx<T> v[2][6];
            T f[2];
            switch (w) {
#define LYM_HOP_PAIR(MU)                                       \
    f[0] = one_hop<MU, true, PR, LK>(a, p, site, r, c, v[0]);  \
    f[1] = one_hop<MU, false, PR, LK>(a, p, site, r, c, v[1]); \
    break
                case 0: LYM_HOP_PAIR(0);
                case 1: LYM_HOP_PAIR(1);
                case 2: LYM_HOP_PAIR(2);
                default: LYM_HOP_PAIR(3);
#undef LYM_HOP_PAIR
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int k = 0; k < 6; ++k) xch[2 * w + i][k * HOP_LANES + lane] = v[i][k];
                if constexpr (PR == 2) fsc[2 * w + i][lane] = f[i];
            }
        }
        if constexpr (FM == F64_CG) {
            // (its operands are on their way while the workgroup gathers)
            UpdPair64 u64;
            if (ok) u64.load(a, p, o, w);
            __syncthreads();
            __syncthreads();
            const double t =
                wave_total(ok ? u64.step(a, p, o, w, al64[0], vout[2 * w][lane], vout[2 * w + 1][lane]) : 0.0);
            if (lane == 0) wsum[0][w] = t;
            __syncthreads();
            if (threadIdx.x == 0) {
                double n2 = 0;
                for (int k = 0; k < HOP_WAVES + 2; ++k) n2 += wsum[0][k];
                a.upd_rpart[blockIdx.x] = n2;
            }
            return;
        }
        __syncthreads();
        if constexpr (FM != F64_STORE) {
            __syncthreads();
        } else if constexpr (UPDATE) {
            __syncthreads();
            pair_sum[w][lane] = ok ? up.step(a, p, ks, o, w, MODE == HOP_BM2 ? (float)a.balpha[r] : al_sh[0],
                                             vout[2 * w][lane], vout[2 * w + 1][lane])
                                   : 0.0;
            __syncthreads();
            if (w == 0) {
                // the pairs in order, as the one-thread form sums them
                double n2 = pair_sum[0][lane];
#pragma unroll
                for (int k = 1; k < HOP_WAVES + 2; ++k) n2 += pair_sum[k][lane];
                if constexpr (MODE == HOP_BM2) {
                    if (ok) a.bsite[p][o] = n2;
                } else {
                    const double t = wave_total(n2);
                    if (lane == 0) a.upd_rpart[blockIdx.x] = t;
                }
            }
        } else if constexpr (PR == 2 || MODE != HOP_STORE) {
            __syncthreads();
        }
        return;
    }

    // ------------------------------------------------ chirality h
    const int h = w - HOP_WAVES;
    constexpr int BK_A = LK >= 2 ? BLK_A_REAL : BLK_A, BK_I = LK >= 2 ? BLK_INV_REAL : BLK_INV;
    cplx<T> s[6], w2[6];  // s: the diagonal term, formed while the hops are under way
    T binv[block_reals(BK_I)];
    T isc = (T)1, hk = (T)0, wsc = (T)1;
    if (ok) {
        const void *Ab = a.A, *Ai = a.Ainv;
        const float *Asc = a.A_sc, *Aisc = a.Ainv_sc;
        if constexpr (LO) {
            const int bs = a.lane_set ? a.lane_set[r] : r;
            Ab = reinterpret_cast<const char*>(Ab) + bs * a.A_lane_bytes;
            Ai = reinterpret_cast<const char*>(Ai) + bs * a.Ainv_lane_bytes;
            if constexpr (PR == 2) {
                Asc += bs * a.Asc_lane;
                Aisc += bs * a.Ainvsc_lane;
            }
        }
        if constexpr (INV) {
            load_block<PR, BK_I>(Ai, 2, ST, h, site, binv);
            if constexpr (PR == 2) isc = Aisc[site];
        }
        if (!INV && a.v2[p]) {
            load_half<PR, true>(a.v2[p], ks, o, h, w2);
            if constexpr (PR == 2) wsc = fld<float>(a.v2_sc[p], o);
        }
        if constexpr (DIAG == 2) {
            cplx<T> t[6];
            T blk[block_reals(BK_A)];
            T sc = (T)1;
            load_half<PR>(lane_base<PR>(a.diag_in[p], a.diag_lane, r), ks, o, h, t);
            load_block<PR, BK_A>(Ab, 4, ST, 2 * p + h, site, blk);
            if constexpr (PR == 2) sc = fld<float>(a.diag_sc[p], o);
            block_apply<PR, BK_A>(blk, PR == 2 ? (T)Asc[(size_t)p * ST + site] : (T)1, t, s);
            if constexpr (PR == 2) {
#pragma unroll
                for (int k = 0; k < 6; ++k) s[k] = sc * s[k];
            }
        } else if constexpr (DIAG == 1) {
            load_half<PR>(lane_base<PR>(a.diag_in[p], a.diag_lane, r), ks, o, h, s);
            if constexpr (PR == 2) {
                const T sc = fld<float>(a.diag_sc[p], o);
#pragma unroll
                for (int k = 0; k < 6; ++k) s[k] = sc * s[k];
            }
        }
        const double kap = LO ? a.kappa_dev[r] : (a.kappa_dev ? *a.kappa_dev : a.kappa);
        hk = (T)(-kap * a.hop_sign);
    }
    [[maybe_unused]] UpdPair64 u64;
    [[maybe_unused]] cplx<T> dw[6];
    if constexpr (FM == F64_CG) {
        if (ok) u64.load(a, p, o, w);
        if (h == 0) {
            double d = 0;
            for (int k = lane; k < a.upd_ndot; k += 64) d += a.upd_dot[k];
            CGState* st = reinterpret_cast<CGState*>(a.upd_state);
            const double rr = st->rr, alpha = rr / wave_total(d);
            if (lane == 0) {
                al64[0] = alpha;
                if (blockIdx.x == 0) set_alpha(st, alpha, rr);
            }
        }
    } else if constexpr (FM == F64_DOT) {
        if (ok) load_half<PR>(a.dotw[p], ks, o, h, dw);
    }
    if constexpr (MODE == HOP_UPD) {
        // alpha = rr_s / <p, Ap>, folded by every workgroup in one order
        if (h == 0) {
            double d = 0;
            for (int k = lane; k < a.upd_ndot; k += 64) d += a.upd_dot[k];
            MCGState* st = reinterpret_cast<MCGState*>(a.upd_state);
            const double rr = st->rr_s, alpha = rr / wave_total(d);
            if (lane == 0) {
                al_sh[0] = (float)alpha;
                if (blockIdx.x == 0) {
                    st->alpha = alpha;
                    st->rr_prev = rr;
                }
            }
        }
    }
    __syncthreads();
    cplx<T> v[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) v[k] = mk((T)0, (T)0);
    if (ok) {
        cplx<T> u[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) u[k] = mk((T)0, (T)0);
#define LYM_ADD_HOPS(CH)                                                                      \
    add_hop<CH, 0, true, PR>(u, xch[0], lane, PR == 2 ? (T)fsc[PR == 2 ? 0 : 0][lane] : (T)1);  \
    add_hop<CH, 0, false, PR>(u, xch[1], lane, PR == 2 ? (T)fsc[PR == 2 ? 1 : 0][lane] : (T)1); \
    add_hop<CH, 1, true, PR>(u, xch[2], lane, PR == 2 ? (T)fsc[PR == 2 ? 2 : 0][lane] : (T)1);  \
    add_hop<CH, 1, false, PR>(u, xch[3], lane, PR == 2 ? (T)fsc[PR == 2 ? 3 : 0][lane] : (T)1); \
    add_hop<CH, 2, true, PR>(u, xch[4], lane, PR == 2 ? (T)fsc[PR == 2 ? 4 : 0][lane] : (T)1);  \
    add_hop<CH, 2, false, PR>(u, xch[5], lane, PR == 2 ? (T)fsc[PR == 2 ? 5 : 0][lane] : (T)1); \
    add_hop<CH, 3, true, PR>(u, xch[6], lane, PR == 2 ? (T)fsc[PR == 2 ? 6 : 0][lane] : (T)1);  \
    add_hop<CH, 3, false, PR>(u, xch[7], lane, PR == 2 ? (T)fsc[PR == 2 ? 7 : 0][lane] : (T)1)
        if (h == 0) {
            LYM_ADD_HOPS(0);
        } else {
            LYM_ADD_HOPS(1);
        }
#undef LYM_ADD_HOPS
        if constexpr (DIAG == 0) {
#pragma unroll
            for (int k = 0; k < 6; ++k) v[k] = hk * u[k];
        } else {
#pragma unroll
            for (int k = 0; k < 6; ++k) v[k] = axpy1(hk, u[k], s[k]);
        }
        if constexpr (INV) {
            cplx<T> t[6];
            block_apply<PR, BK_I>(binv, isc, v, t);
#pragma unroll
            for (int k = 0; k < 6; ++k) v[k] = t[k];
        }
        if (a.gamma5 && h) {
#pragma unroll
            for (int k = 0; k < 6; ++k) v[k] = -v[k];
        }
        if (a.v2[p]) {
            if constexpr (INV) {  // (R^-1 holds the registers until here)
                load_half<PR, true>(a.v2[p], ks, o, h, w2);
                if constexpr (PR == 2) wsc = fld<float>(a.v2_sc[p], o);
            }
            const cplx<T> al2 = mk((T)a.alpha.re, (T)a.alpha.im);
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                if constexpr (PR == 2) w2[k] = wsc * w2[k];
                cfma(v[k], al2, w2[k]);
            }
        }
    }
    if constexpr (FM == F64_CG) {
#pragma unroll
        for (int k = 0; k < 6; ++k) vout[6 * h + k][lane] = v[k];
        __syncthreads();
        const double t =
            wave_total(ok ? u64.step(a, p, o, w, al64[0], vout[2 * w][lane], vout[2 * w + 1][lane]) : 0.0);
        if (lane == 0) wsum[0][w] = t;
        __syncthreads();
        return;
    } else if constexpr (UPDATE) {
        // v in FP32 to every wave, never rounded to storage
#pragma unroll
        for (int k = 0; k < 6; ++k) vout[6 * h + k][lane] = v[k];
        __syncthreads();
        pair_sum[w][lane] = ok ? up.step(a, p, ks, o, w, MODE == HOP_BM2 ? (float)a.balpha[r] : al_sh[0],
                                         vout[2 * w][lane], vout[2 * w + 1][lane])
                               : 0.0;
        __syncthreads();
        return;
    } else {
        float m = 0.f;
        if constexpr (PR == 2) {
#pragma unroll
            for (int k = 0; k < 6; ++k) m = fmaxf(m, fmaxf(fabsf(v[k].re), fabsf(v[k].im)));
            half_max[h][lane] = m;
        }
        float n2 = 0.f;
        if constexpr (MODE != HOP_STORE) {
#pragma unroll
            for (int k = 0; k < 6; ++k) n2 = norm_acc(v[k], n2);
            if (h == 1) half_sum[lane] = n2;
        }
        if constexpr (PR == 2 || MODE != HOP_STORE) __syncthreads();
        S e[6];
        if constexpr (PR == 2) {
            m = fmaxf(half_max[0][lane], half_max[1][lane]);
            const float inv = fp16_site_inv(m);
#pragma unroll
            for (int k = 0; k < 6; ++k) e[k] = from_c<PR>(inv * v[k]);
        } else {
#pragma unroll
            for (int k = 0; k < 6; ++k) e[k] = from_c<PR>(v[k]);
        }
        if (ok) {
            if constexpr (PR == 0) {
                zd* b = const_cast<zd*>(lane_base<0>(a.out[p], a.out_lane, r)) + (size_t)(6 * h) * ks;
#pragma unroll
                for (int k = 0; k < 6; ++k) fst(b + k * ks, o, e[k]);
            } else {
                store_half_lp<PR>(reinterpret_cast<S*>(a.out[p]), ks, o, h, e);
                if (PR == 2 && h == 0) fst<float, false>(a.out_sc[p], o, m);
            }
        }
        if constexpr (FM != F64_STORE) {
            // (lanes without a site hold zeros in v)
            double sums[3] = {0, 0, 0};
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                if constexpr (FM == F64_DOT) {
                    const zd wv = ok ? dw[k] : mk(0.0, 0.0);
                    sums[0] = fmadd(wv.im, v[k].im, fmadd(wv.re, v[k].re, sums[0]));
                    sums[1] = fmadd(-wv.im, v[k].re, fmadd(wv.re, v[k].im, sums[1]));
                    sums[2] = norm_acc(v[k], sums[2]);
                } else {
                    sums[0] = norm_acc(v[k], sums[0]);
                }
            }
            constexpr int NS = FM == F64_DOT ? 3 : 1;
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                sums[k] = wave_total(sums[k]);
                if (h == 1 && lane == 0) wsum[k][0] = sums[k];
            }
            __syncthreads();
            if (h == 0 && lane == 0)
#pragma unroll
                for (int k = 0; k < NS; ++k)
                    a.upd_rpart[(size_t)k * a.part_stride + blockIdx.x] = sums[k] + wsum[k][0];
        }
        if constexpr (MODE != HOP_STORE) {
            if (h == 0) {
                n2 += (float)half_sum[lane];
                if constexpr (MODE == HOP_BM1) {
                    if (ok) a.bsite[p][o] = (double)n2;
                } else {
                    const double t = wave_total((double)n2);
                    if (lane == 0) a.norm_partials[blockIdx.x] = t;
                }
            }
        }
    }
}

template <int PR, int LK, int DIAG, bool INV, int MODE = HOP_STORE>
static void hop_go(const DslashParams& a, int nblocks, hipStream_t st) {
    if constexpr (MODE != HOP_NORM && MODE != HOP_UPD) {
        if (a.lane_ops) {
            hipLaunchKernelGGL((k_dslash_hop<PR, LK, DIAG, INV, MODE, true>),
                               dim3(PR == 0 ? lane_grid(a, nblocks, 1) : nblocks), dim3(HOP_THREADS), 0, st, a);
            return;
        }
    }
    hipLaunchKernelGGL((k_dslash_hop<PR, LK, DIAG, INV, MODE, false>),
                       dim3(PR == 0 ? lane_grid(a, nblocks, 1) : nblocks), dim3(HOP_THREADS), 0, st, a);
}

// the FP64 solvers' fused steps
template <int LK, int DIAG>
static void hop_f64(const DslashParams& a, int nblocks, hipStream_t st) {
    const dim3 g(nblocks), t(HOP_THREADS);
    switch (a.fmode) {
        case F64_NORM:
            hipLaunchKernelGGL((k_dslash_hop<0, LK, DIAG, false, HOP_STORE, false, F64_NORM>), g, t, 0, st, a);
            break;
        case F64_CG:
            hipLaunchKernelGGL((k_dslash_hop<0, LK, DIAG, false, HOP_STORE, false, F64_CG>), g, t, 0, st, a);
            break;
        default:
            hipLaunchKernelGGL((k_dslash_hop<0, LK, DIAG, false, HOP_STORE, false, F64_DOT>), g, t, 0, st, a);
            break;
    }
}

template <int PR, int LK>
static void hop_lk(const DslashParams& a, int diag, bool inv, int nblocks, hipStream_t st) {
    if (diag == 0) {
        if (inv) hop_go<PR, LK, 0, true>(a, nblocks, st);
        else hop_go<PR, LK, 0, false>(a, nblocks, st);
        return;
    }
    if constexpr (PR >= 1) {
        if (!inv && (a.upd_state || a.norm_partials || a.bmode)) {
            if (diag == 1) {
                if (a.bmode == 1) hop_go<PR, LK, 1, false, HOP_BM1>(a, nblocks, st);
                else if (a.bmode == 2) hop_go<PR, LK, 1, false, HOP_BM2>(a, nblocks, st);
                else if (a.upd_state) hop_go<PR, LK, 1, false, HOP_UPD>(a, nblocks, st);
                else hop_go<PR, LK, 1, false, HOP_NORM>(a, nblocks, st);
            } else {
                if (a.bmode == 1) hop_go<PR, LK, 2, false, HOP_BM1>(a, nblocks, st);
                else if (a.bmode == 2) hop_go<PR, LK, 2, false, HOP_BM2>(a, nblocks, st);
                else if (a.upd_state) hop_go<PR, LK, 2, false, HOP_UPD>(a, nblocks, st);
                else hop_go<PR, LK, 2, false, HOP_NORM>(a, nblocks, st);
            }
            return;
        }
    }
    if constexpr (PR == 0) {
        if (a.fmode) {
            if (diag == 1) hop_f64<LK, 1>(a, nblocks, st);
            else hop_f64<LK, 2>(a, nblocks, st);
            return;
        }
    }
    if (diag == 1) {
        if (inv) hop_go<PR, LK, 1, true>(a, nblocks, st);
        else hop_go<PR, LK, 1, false>(a, nblocks, st);
    } else {
        hop_go<PR, LK, 2, false>(a, nblocks, st);
    }
}

template <int PR>
static void hop_pr(const DslashParams& a, int link_kind, int diag, bool inv, int nblocks, hipStream_t st) {
    switch (link_kind) {
        case 0: hop_lk<PR, 0>(a, diag, inv, nblocks, st); break;
        case 1: hop_lk<PR, 1>(a, diag, inv, nblocks, st); break;
        case 2: hop_lk<PR, 2>(a, diag, inv, nblocks, st); break;
        default: hop_lk<PR, 3>(a, diag, inv, nblocks, st); break;
    }
}

void launch_dslash_hop(const DslashParams& a, int link_kind, int diag, bool inv, int nblocks, hipStream_t st) {
    switch (a.prec) {
        case 0: hop_pr<0>(a, link_kind, diag, inv, nblocks, st); break;
        case 1: hop_pr<1>(a, link_kind, diag, inv, nblocks, st); break;
        default: hop_pr<2>(a, link_kind, diag, inv, nblocks, st); break;
    }
}

}  // namespace lym
