// batch.hip -- multi-RHS mixed-precision CG with per-RHS reliable updates.
//
// NR right-hand sides share every operator apply (rhs-fastest fields, so one
// link load serves all NR lanes of a site) while each keeps its own CG
// recursion: alpha, beta, |r|^2, its reliable-update decisions, its tolerance
// and its stopping point.  A converged RHS is frozen.  Every per-RHS sum runs
// over the same site partition and in the same order as the single-RHS kernels
// of mixed.hip (thread per site, 512 x 256 grid-stride, fixed trees), and the
// per-site arithmetic is the same, so an RHS gives bit-identical results alone
// and in any batch.
#include "lym_device.h"

namespace lym {

// Every per-RHS sum runs over fixed chunks of BC consecutive sites: a chunk's
// sum is an LDS tree over its BC sites, and the final sum an LDS tree over
// per-thread strided sums of the chunk partials, with a fixed FT-thread
// block.  Neither tree depends on NR, so an RHS sums its terms in the same
// order in a batch of any size.
constexpr int BC = BATCH_CHUNK;  // sites per chunk
constexpr int FT = 1024;   // threads of the final-sum block

// chunk sum of v (one value per (site, lane) thread; block = BC sites x NR lanes)
template <int NR>
__device__ __forceinline__ void chunk_store(double v, double* partials, long nchunks) {
    __shared__ double red[NR * BC];
    const int t = threadIdx.x, sl = t / NR, q = t - sl * NR;
    red[q * BC + sl] = v;
    __syncthreads();
#pragma unroll
    for (int off = BC / 2; off > 0; off >>= 1) {
        if (sl < off) red[q * BC + sl] += red[q * BC + sl + off];
        __syncthreads();
    }
    if (sl == 0) partials[(long)q * nchunks + blockIdx.x] = red[q * BC];
}

// final per-RHS sums into tot (shared, valid after the call), one FT-thread block.
// Thread t sums the chunks t, t + FT, ...; the tree over the FT sums pairs t with
// t + 512, then 256, ... 1.  All lanes (in groups of FG) load at once, and wave q of
// the block runs lane q's tree, the steps down to 64 in registers and the rest by
// shuffles (one lane after the other, with a barrier a step, 8 lanes of 16384 chunks
// took 45 us and 4 lanes of small lattices 8 to 11, now 18 and 3.5 to 4).
constexpr int FG = 8;
template <int NR>
__device__ __forceinline__ void final_sums(const double* partials, long nchunks, double* tot) {
    constexpr int G = NR < FG ? NR : FG;
    __shared__ double sh[G * FT];
    const int t = threadIdx.x, w = t >> 6, l = t & 63;
#pragma unroll
    for (int q0 = 0; q0 < NR; q0 += G) {
        double v[G];
#pragma unroll
        for (int g = 0; g < G; ++g) v[g] = 0;
        for (long c = t; c < nchunks; c += FT) {
#pragma unroll
            for (int g = 0; g < G; ++g)
                if (q0 + g < NR) v[g] += partials[(long)(q0 + g) * nchunks + c];
        }
        if (q0) __syncthreads();  // the trees of the group before have read sh
#pragma unroll
        for (int g = 0; g < G; ++g) sh[g * FT + t] = v[g];
        __syncthreads();
        if (w < G && q0 + w < NR) {
            double u[FT / 64];
#pragma unroll
            for (int m = 0; m < FT / 64; ++m) u[m] = sh[w * FT + l + 64 * m];
#pragma unroll
            for (int off = FT / 128; off > 0; off >>= 1) {
#pragma unroll
                for (int m = 0; m < off; ++m) u[m] += u[m + off];
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) u[0] += __shfl_down(u[0], off);
            if (l == 0) tot[q0 + w] = u[0];
        }
    }
    __syncthreads();
}

#define BSITE_LOOP(j, n) for (long j = (long)blockIdx.x * blockDim.x + threadIdx.x; j < (n); j += (long)gridDim.x * blockDim.x)

// (site, lane) of this thread in a chunked launch; false past the field
template <int NR>
__device__ __forceinline__ bool chunk_pair(long nsites, long& j, int& q) {
    const int t = threadIdx.x, sl = t / NR;
    q = t - sl * NR;
    j = (long)blockIdx.x * BC + sl;
    return j < nsites;
}

#define PAIR_LOOP(j, q, NR, nsites)                                                                        \
    for (long t_ = (long)blockIdx.x * blockDim.x + threadIdx.x, j, q; t_ < (nsites) * (NR) &&              \
                                                                  ((j = t_ / (NR)), (q = t_ - j * (NR)), 1); \
         t_ += (long)gridDim.x * blockDim.x)

// element (parity p, component k, site i, rhs r) of an nr-field: ((p*12 + k)*stride + i)*nr + r
__device__ __forceinline__ long bidx(int stride, int nr, long j, int k, int r) {
    const long p = j / stride, i = j % stride;
    return ((p * 12 + k) * stride + i) * nr + r;
}

// parity base of a low-precision nr-field and the lane element of (site j, rhs r)
template <int PR, int NR>
__device__ __forceinline__ long bs_parity_off(int stride, long j) {
    return (j / stride) * 12L * stride * NR;
}

template <int PR, int NR>
__device__ __forceinline__ void bs_load(const typename Prec<PR>::S* d, const float* sc, int stride, long j, int r,
                                        cplx<float> s[12]) {
    typename Prec<PR>::S e[12];
    load_packed<PR>(d + bs_parity_off<PR, NR>(stride, j), (size_t)stride * NR, (unsigned)((j % stride) * NR + r), e);
#pragma unroll
    for (int k = 0; k < 12; ++k) {
        cplx<typename Prec<PR>::T> z = to_c<PR>(e[k]);
        s[k] = mk((float)z.re, (float)z.im);
    }
    if constexpr (PR == 2) {
        const float f = sc[j * NR + r];
#pragma unroll
        for (int k = 0; k < 12; ++k) s[k] = f * s[k];
    }
}

template <int PR, int NR>
__device__ __forceinline__ void bs_store(typename Prec<PR>::S* d, float* sc, int stride, long j, int r,
                                         const cplx<float> s[12]) {
    if constexpr (PR == 2) {
        float m = 0.f;
#pragma unroll
        for (int k = 0; k < 12; ++k) m = fmaxf(m, fmaxf(fabsf(s[k].re), fabsf(s[k].im)));
        const float inv = fp16_site_inv(m);
        typename Prec<PR>::S e[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) e[k] = from_c<PR>(inv * s[k]);
        store_packed<PR, false>(d + bs_parity_off<PR, NR>(stride, j), (size_t)stride * NR,
                                (unsigned)((j % stride) * NR + r), e);
        sc[j * NR + r] = m;
    } else {
        typename Prec<PR>::S e[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) e[k] = from_c<PR>(s[k]);
        store_packed<PR, false>(d + bs_parity_off<PR, NR>(stride, j), (size_t)stride * NR,
                                (unsigned)((j % stride) * NR + r), e);
    }
}

// FP64 lane fields: lane r holds [nparity][12][stride] of its own (nsites = nparity * stride)
__device__ __forceinline__ void ld_lane(const zd* d, long nsites, int stride, long j, int r, zd s[12]) {
    const long p = j / stride, i = j - p * stride;
    const zd* b = d + (r * nsites + p * stride) * 12 + i;
#pragma unroll
    for (int k = 0; k < 12; ++k) s[k] = b[(long)k * stride];
}
__device__ __forceinline__ void st_lane(zd* d, long nsites, int stride, long j, int r, const zd s[12]) {
    const long p = j / stride, i = j - p * stride;
    zd* b = d + (r * nsites + p * stride) * 12 + i;
#pragma unroll
    for (int k = 0; k < 12; ++k) b[(long)k * stride] = s[k];
}

template <class E, int NR>
__device__ __forceinline__ void bg_load(const E* d, int stride, long j, int r, E s[12]) {
#pragma unroll
    for (int k = 0; k < 12; ++k) s[k] = d[bidx(stride, NR, j, k, r)];
}
template <class E, int NR>
__device__ __forceinline__ void bg_store(E* d, int stride, long j, int r, const E s[12]) {
#pragma unroll
    for (int k = 0; k < 12; ++k) d[bidx(stride, NR, j, k, r)] = s[k];
}

// ---------------------------------------------------------------- kernels
// Sums: one thread per (site, RHS) pair, RHS fastest (coalesced like the
// fields), chunk_store / final_sums.  Element-wise kernels: PAIR_LOOP.
// mask (may be null: every lane): only the lanes with mask[q] != 0 start
template <int PR, int NR>
__global__ __launch_bounds__(BC * NR) void k_bcg_init(const zd* r, cplx<float>* rs, cplx<float>* xs,
                                                      typename Prec<PR>::S* p, float* p_sc, long nsites, int stride,
                                                      double* partials, long nchunks, const int* mask) {
    long j;
    int q;
    double v = 0;
    if (chunk_pair<NR>(nsites, j, q) && (!mask || mask[q])) {
        zd a[12];
        cplx<float> f[12], z[12];
        ld_lane(r, nsites, stride, j, q, a);
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            v += a[k].re * a[k].re + a[k].im * a[k].im;
            f[k] = mk((float)a[k].re, (float)a[k].im);
            z[k] = mk(0.f, 0.f);
        }
        bg_store<cplx<float>, NR>(rs, stride, j, q, f);
        bg_store<cplx<float>, NR>(xs, stride, j, q, z);
        bs_store<PR, NR>(p, p_sc, stride, j, q, f);
    }
    chunk_store<NR>(v, partials, nchunks);
}

template <int NR>
__global__ __launch_bounds__(FT) void k_bcg_init_final(BState* s, const double* partials, long nchunks,
                                                       int max_steps, const int* mask) {
    __shared__ double tot[NR];
    final_sums<NR>(partials, nchunks, tot);
    const int q = threadIdx.x;
    if (q >= 64) return;
    const bool on = q < NR;
    if (on && !(mask && !mask[q])) {  // else a lane that keeps its state
        s->rr_s[q] = s->rr_true[q] = s->maxrr[q] = tot[q];
        s->step[q] = 0;
        s->nrel[q] = 0;
        s->rel[q] = 0;
        s->alpha[q] = s->beta[q] = 0;
        // a zero source has the solution x = x0 = 0: nothing to iterate
        s->conv[q] = tot[q] == 0.0 ? 1 : 0;
        s->done[q] = (max_steps <= 0 || tot[q] == 0.0) ? 1 : 0;
    }
    // a lane that keeps its state may hold an update due at the next slot
    const int any = __any(on && s->rel[q] && !s->done[q]), all = __all(!on || s->done[q]);
    if (q == 0) {
        s->max_steps = max_steps;
        s->all_done = all;
        s->any_rel = any;
        s->skip_rel = any ? 0 : 1;
    }
}

template <int PR, int NR>
__global__ __launch_bounds__(BC * NR) void k_bcg_dot(const BState* s, const typename Prec<PR>::S* p,
                                                     const float* p_sc, const typename Prec<PR>::S* Ap,
                                                     const float* Ap_sc, long nsites, int stride, double* partials,
                                                     long nchunks) {
    if (s->all_done) return;
    long j;
    int q;
    double v = 0;
    if (chunk_pair<NR>(nsites, j, q) && !s->done[q]) {
        cplx<float> a[12], b[12];
        bs_load<PR, NR>(p, p_sc, stride, j, q, a);
        bs_load<PR, NR>(Ap, Ap_sc, stride, j, q, b);
#pragma unroll
        for (int k = 0; k < 12; ++k) v += (double)a[k].re * b[k].re + (double)a[k].im * b[k].im;
    }
    chunk_store<NR>(v, partials, nchunks);
}

// chunk sums of one value per (site, RHS) written by a fused stencil launch
// (bsite[j * NR + q]); lanes that are done contribute zero, as in k_bcg_dot.
// Only the vh real sites of each parity count: the stencil never writes the
// padding slots up to the stride, which may hold values a wider batch left.
// Widths of a power of two: a wave per chunk, its BC sites x NR lanes in NR registers
// a thread (value 64 m + l of the chunk in register m of lane l), the tree's steps
// (pairs of sites 32, 16, ... 1 apart) first between registers, then by shuffles, in
// the same order as chunk_store.  A block of BC x NR threads with a barrier a step
// read 1.5 TB/s (45 us for 8 lanes of 32^3x64, now 14).
constexpr int CHUNK_WAVES = 4;
template <int NR>
constexpr bool chunk_wave = (NR & (NR - 1)) == 0;
template <int NR>
__global__ __launch_bounds__(chunk_wave<NR> ? 64 * CHUNK_WAVES : BC * NR) void k_bcg_chunksum(
    const BState* s, const double* bsite, long nsites, int stride, int vh, double* partials, long nchunks) {
    if (s->all_done) return;
    if constexpr (chunk_wave<NR>) {
        const int l = threadIdx.x & 63;
        const long c = (long)blockIdx.x * CHUNK_WAVES + (threadIdx.x >> 6), j0 = c * BC;
        if (c >= nchunks) return;
        const bool on = !s->done[l % NR];
        const int i0 = (int)(j0 % stride);  // a chunk lies within one parity (the stride is a multiple of BC)
        double v[NR];
#pragma unroll
        for (int m = 0; m < NR; ++m) {
            const int sl = (64 * m + l) / NR;
            v[m] = on && j0 + sl < nsites && i0 + sl < vh ? bsite[j0 * NR + 64 * m + l] : 0.0;
        }
#pragma unroll
        for (int off = NR / 2; off > 0; off >>= 1) {
#pragma unroll
            for (int m = 0; m < off; ++m) v[m] += v[m + off];
        }
#pragma unroll
        for (int off = 32; off >= NR; off >>= 1) v[0] += __shfl_down(v[0], off);
        if (l < NR) partials[(long)l * nchunks + c] = v[0];
    } else {
        long j;
        int q;
        double v = 0;
        if (chunk_pair<NR>(nsites, j, q) && !s->done[q] && j % stride < vh) v = bsite[j * NR + q];
        chunk_store<NR>(v, partials, nchunks);
    }
}

template <int NR>
__global__ __launch_bounds__(FT) void k_bcg_alpha_final(BState* s, const double* partials, long nchunks) {
    if (s->all_done) return;
    __shared__ double tot[NR];
    const int q = threadIdx.x < NR ? threadIdx.x : 0;
    const double rr = s->rr_s[q];
    const int done = s->done[q];
    final_sums<NR>(partials, nchunks, tot);
    if (threadIdx.x < NR && !done) s->alpha[q] = rr / tot[q];
}

template <int PR, int NR>
__global__ __launch_bounds__(BC * NR) void k_bcg_update(const BState* s, cplx<float>* xs, cplx<float>* rs,
                                                        const typename Prec<PR>::S* p, const float* p_sc,
                                                        const typename Prec<PR>::S* Ap, const float* Ap_sc,
                                                        long nsites, int stride, double* partials, long nchunks) {
    if (s->all_done) return;
    long j;
    int q;
    double v = 0;
    if (chunk_pair<NR>(nsites, j, q) && !s->done[q]) {
        const float al = (float)s->alpha[q];
        cplx<float> x[12], r[12], a[12], b[12];
        bg_load<cplx<float>, NR>(xs, stride, j, q, x);
        bg_load<cplx<float>, NR>(rs, stride, j, q, r);
        bs_load<PR, NR>(p, p_sc, stride, j, q, a);
        bs_load<PR, NR>(Ap, Ap_sc, stride, j, q, b);
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            x[k] = x[k] + al * a[k];
            r[k] = r[k] - al * b[k];
            v += (double)r[k].re * r[k].re + (double)r[k].im * r[k].im;
        }
        bg_store<cplx<float>, NR>(xs, stride, j, q, x);
        bg_store<cplx<float>, NR>(rs, stride, j, q, r);
    }
    chunk_store<NR>(v, partials, nchunks);
}

template <int NR>
__global__ __launch_bounds__(FT) void k_bcg_update_final(BState* s, const double* partials, long nchunks) {
    if (s->all_done) return;
    __shared__ double tot[NR];
    const bool on = threadIdx.x < NR;
    const int q = on ? threadIdx.x : 0;
    double mx = s->maxrr[q];
    const double rr = s->rr_s[q], eps = s->eps[q], delta2 = s->delta2;
    int done = s->done[q], rel = s->rel[q];
    const int step = s->step[q] + 1, max_steps = s->max_steps;
    final_sums<NR>(partials, nchunks, tot);
    if (threadIdx.x >= 64) return;
    if (on && !done) {
        const double rn = tot[q];
        if (rn > mx) s->maxrr[q] = mx = rn;
        // due reliable updates run at the next reliable-update slot
        if (rn < delta2 * mx || rn < eps) s->rel[q] = rel = 1;
        s->beta[q] = rn / rr;
        s->rr_s[q] = rn;
        s->step[q] = step;
        if (step >= max_steps) s->done[q] = done = 1;
    }
    const int any = __any(on && rel && !done), all = __all(!on || done);
    if (threadIdx.x == 0) {
        s->any_rel = any;
        s->skip_rel = any ? 0 : 1;
        s->all_done = all;
    }
}

// reliable update, part 1, for the RHS with a due update: x += x_s, x_s = 0
template <int NR>
__global__ void k_brel_accum(const BState* s, zd* x, cplx<float>* xs, long nsites, int stride) {
    if (s->skip_rel) return;
    PAIR_LOOP(j, q, NR, nsites) {
        if (!s->rel[q]) continue;
        zd a[12];
        cplx<float> f[12];
        ld_lane(x, nsites, stride, j, (int)q, a);
        bg_load<cplx<float>, NR>(xs, stride, j, (int)q, f);
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            a[k] = a[k] + mk((double)f[k].re, (double)f[k].im);
            f[k] = mk(0.f, 0.f);
        }
        st_lane(x, nsites, stride, j, (int)q, a);
        bg_store<cplx<float>, NR>(xs, stride, j, (int)q, f);
    }
}

// reliable update, part 2: r = b - Ax (FP64), r_s = r, |r|^2
template <int NR>
__global__ __launch_bounds__(BC * NR) void k_brel_resid(const BState* s, zd* r, cplx<float>* rs, const zd* b,
                                                        const zd* Ax, long nsites, int stride, double* partials,
                                                        long nchunks) {
    if (s->skip_rel) return;
    long j;
    int q;
    double v = 0;
    if (chunk_pair<NR>(nsites, j, q) && s->rel[q]) {
        zd bb[12], ax[12];
        cplx<float> f[12];
        ld_lane(b, nsites, stride, j, q, bb);
        ld_lane(Ax, nsites, stride, j, q, ax);
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            bb[k] = bb[k] - ax[k];
            v += bb[k].re * bb[k].re + bb[k].im * bb[k].im;
            f[k] = mk((float)bb[k].re, (float)bb[k].im);
        }
        st_lane(r, nsites, stride, j, q, bb);
        bg_store<cplx<float>, NR>(rs, stride, j, q, f);
    }
    chunk_store<NR>(v, partials, nchunks);
}

template <int NR>
__global__ __launch_bounds__(FT) void k_brel_final(BState* s, const double* partials, long nchunks) {
    if (s->skip_rel) return;
    __shared__ double tot[NR];
    const bool on = threadIdx.x < NR;
    const int q = on ? threadIdx.x : 0;
    int done = s->done[q];
    const int rel = s->rel[q], nrel = s->nrel[q] + 1;
    const double eps = s->eps[q];
    final_sums<NR>(partials, nchunks, tot);
    if (threadIdx.x >= 64) return;
    if (on && rel) {
        const double rt = tot[q];
        s->rr_true[q] = rt;
        s->nrel[q] = nrel;
        s->rel[q] = 0;
        if (rt < eps) {
            s->done[q] = done = 1;
            s->conv[q] = 1;
        } else {
            s->rr_s[q] = rt;
            s->maxrr[q] = rt;
        }
    }
    const int all = __all(!on || done);
    if (threadIdx.x == 0) {
        s->any_rel = 0;
        s->skip_rel = 1;
        s->all_done = all;
    }
}

template <int PR, int NR>
__global__ void k_bcg_p(const BState* s, typename Prec<PR>::S* p, float* p_sc, const cplx<float>* rs, long nsites,
                        int stride) {
    if (s->all_done) return;
    PAIR_LOOP(j, q, NR, nsites) {
        if (s->done[q]) continue;
        const float be = (float)s->beta[q];
        cplx<float> a[12], r[12];
        bs_load<PR, NR>(p, p_sc, stride, j, (int)q, a);
        bg_load<cplx<float>, NR>(rs, stride, j, (int)q, r);
#pragma unroll
        for (int k = 0; k < 12; ++k) a[k] = r[k] + be * a[k];
        bs_store<PR, NR>(p, p_sc, stride, j, (int)q, a);
    }
}

// x += x_s for the RHS that stopped between reliable updates (mask may be null: every lane)
template <int NR>
__global__ void k_baccum(const BState* s, zd* x, const cplx<float>* xs, long nsites, int stride, const int* mask) {
    PAIR_LOOP(j, q, NR, nsites) {
        if (s->conv[q] || (mask && !mask[q])) continue;
        zd a[12];
        cplx<float> f[12];
        ld_lane(x, nsites, stride, j, (int)q, a);
        bg_load<cplx<float>, NR>(xs, stride, j, (int)q, f);
#pragma unroll
        for (int k = 0; k < 12; ++k) a[k] = a[k] + mk((double)f[k].re, (double)f[k].im);
        st_lane(x, nsites, stride, j, (int)q, a);
    }
}

// pack / unpack single full fields <-> an nr-field (a null pointer leaves
// its lane alone); also multi-RHS clover block apply
__global__ void k_pack(const zd* const* srcs, int nr, zd* multi, long n) {
    BSITE_LOOP(i, n) {
        for (int r = 0; r < nr; ++r)
            if (srcs[r]) multi[i * nr + r] = srcs[r][i];
    }
}
__global__ void k_unpack(const zd* multi, int nr, zd* const* dsts, long n) {
    BSITE_LOOP(i, n) {
        for (int r = 0; r < nr; ++r)
            if (dsts[r]) dsts[r][i] = multi[i * nr + r];
    }
}

// ---------------------------------------------------------------- lanes
// FP64 lane fields: one grid row per lane
__global__ void k_lane_copy(zd* dst, long dst_lane, const zd* src, long src_lane, long n, const int* mask) {
    const int l = blockIdx.y;
    if (mask && !mask[l]) return;
    BSITE_LOOP(i, n) { dst[l * dst_lane + i] = src[l * src_lane + i]; }
}
__global__ void k_lane_sub(zd* out, const zd* a, const zd* b, long lane, long n, const int* mask) {
    const int l = blockIdx.y;
    if (mask && !mask[l]) return;
    BSITE_LOOP(i, n) { out[l * lane + i] = a[l * lane + i] - b[l * lane + i]; }
}
__global__ void k_lane_gather(const zd* const* srcs, zd* dst, long n) {
    const zd* s = srcs[blockIdx.y];
    if (!s) return;
    BSITE_LOOP(i, n) { dst[blockIdx.y * n + i] = s[i]; }
}
__global__ void k_lane_scatter(const zd* src, zd* const* dsts, long n) {
    zd* d = dsts[blockIdx.y];
    if (!d) return;
    BSITE_LOOP(i, n) { d[i] = src[blockIdx.y * n + i]; }
}
// An interleaved field is rows x nr elements, lane fastest.
// out (width w_new) from in (width w_old): lane j keeps its index, lanes
// j >= w_old are zero
template <class E>
__global__ void k_relayout(const E* in, E* out, long rows, int w_old, int w_new) {
    BSITE_LOOP(t, rows * w_new) {
        const long i = t / w_new;
        const int j = (int)(t - i * w_new);
        E e;
        if (j < w_old) e = in[i * w_old + j];
        else __builtin_memset(&e, 0, sizeof(E));
        out[t] = e;
    }
}

// ---------------------------------------------------------------- launchers
static inline int bsite_blocks(long n) {
    long b = (n + 255) / 256;
    return (int)(b < 4096 ? b : 4096);
}

static inline int pair_blocks(long pairs) {
    long b = (pairs + 255) / 256;
    return (int)(b < 8192 ? b : 8192);
}

template <int PR, int NR>
static void bcg_step_impl(int which, BState* s, const BcgArgs& a, hipStream_t st) {
    typedef typename Prec<PR>::S S;
    S* p = reinterpret_cast<S*>(a.p);
    S* Ap = reinterpret_cast<S*>(a.Ap);
    const long nch = (a.nsites + BC - 1) / BC;
    const dim3 cg((unsigned)nch), cb(BC * NR), fb(FT);
    const int eb = pair_blocks(a.nsites * NR);
    const dim3 sg(chunk_wave<NR> ? (unsigned)((nch + CHUNK_WAVES - 1) / CHUNK_WAVES) : (unsigned)nch);
    const dim3 sb(chunk_wave<NR> ? 64 * CHUNK_WAVES : BC * NR);
    switch (which) {
        case 0:
            hipLaunchKernelGGL((k_bcg_init<PR, NR>), cg, cb, 0, st, a.r, a.rs, a.xs, p, a.p_sc, a.nsites, a.stride,
                               a.partials, nch, a.mask);
            hipLaunchKernelGGL((k_bcg_init_final<NR>), dim3(1), fb, 0, st, s, a.partials, nch, a.max_steps, a.mask);
            break;
        case 1:
            hipLaunchKernelGGL((k_bcg_dot<PR, NR>), cg, cb, 0, st, s, p, a.p_sc, Ap, a.Ap_sc, a.nsites, a.stride,
                               a.partials, nch);
            hipLaunchKernelGGL((k_bcg_alpha_final<NR>), dim3(1), fb, 0, st, s, a.partials, nch);
            break;
        case 2:
            hipLaunchKernelGGL((k_bcg_update<PR, NR>), cg, cb, 0, st, s, a.xs, a.rs, p, a.p_sc, Ap, a.Ap_sc, a.nsites,
                               a.stride, a.partials, nch);
            hipLaunchKernelGGL((k_bcg_update_final<NR>), dim3(1), fb, 0, st, s, a.partials, nch);
            break;
        case 3:
            hipLaunchKernelGGL((k_brel_accum<NR>), dim3(eb), dim3(256), 0, st, s, a.x, a.xs, a.nsites, a.stride);
            break;
        case 4:
            hipLaunchKernelGGL((k_brel_resid<NR>), cg, cb, 0, st, s, a.r, a.rs, a.b, a.Ax, a.nsites, a.stride,
                               a.partials, nch);
            hipLaunchKernelGGL((k_brel_final<NR>), dim3(1), fb, 0, st, s, a.partials, nch);
            break;
        case 5:
            hipLaunchKernelGGL((k_bcg_p<PR, NR>), dim3(eb), dim3(256), 0, st, s, p, a.p_sc, a.rs, a.nsites, a.stride);
            break;
        case 7:
            hipLaunchKernelGGL((k_bcg_chunksum<NR>), sg, sb, 0, st, s, a.bsite, a.nsites, a.stride, a.vh, a.partials,
                               nch);
            hipLaunchKernelGGL((k_bcg_alpha_final<NR>), dim3(1), fb, 0, st, s, a.partials, nch);
            break;
        case 8:
            hipLaunchKernelGGL((k_bcg_chunksum<NR>), sg, sb, 0, st, s, a.bsite, a.nsites, a.stride, a.vh, a.partials,
                               nch);
            hipLaunchKernelGGL((k_bcg_update_final<NR>), dim3(1), fb, 0, st, s, a.partials, nch);
            break;
        default:
            hipLaunchKernelGGL((k_baccum<NR>), dim3(eb), dim3(256), 0, st, s, a.x, a.xs, a.nsites, a.stride, a.mask);
            break;
    }
}

template <int PR>
static bool bcg_step_pr(int which, int nr, BState* s, const BcgArgs& a, hipStream_t st) {
    switch (nr) {
        case 1: bcg_step_impl<PR, 1>(which, s, a, st); return true;
        case 2: bcg_step_impl<PR, 2>(which, s, a, st); return true;
        case 3: bcg_step_impl<PR, 3>(which, s, a, st); return true;
        case 4: bcg_step_impl<PR, 4>(which, s, a, st); return true;
        case 6: bcg_step_impl<PR, 6>(which, s, a, st); return true;
        case 8: bcg_step_impl<PR, 8>(which, s, a, st); return true;
        case 12: bcg_step_impl<PR, 12>(which, s, a, st); return true;
        case 16: bcg_step_impl<PR, 16>(which, s, a, st); return true;
        default: return false;
    }
}

bool launch_bcg_step(int which, int prec, int nr, BState* s, const BcgArgs& a, hipStream_t st) {
    return prec == 1 ? bcg_step_pr<1>(which, nr, s, a, st) : bcg_step_pr<2>(which, nr, s, a, st);
}

bool batch_nr_supported(int nr) { return nr == 1 || nr == 2 || nr == 3 || nr == 4 || nr == 6 || nr == 8 || nr == 12 || nr == 16; }

void launch_pack(const zd* const* srcs_dev, int nr, zd* multi, long n, hipStream_t st) {
    hipLaunchKernelGGL(k_pack, dim3(bsite_blocks(n)), dim3(256), 0, st, srcs_dev, nr, multi, n);
}
void launch_unpack(const zd* multi, int nr, zd* const* dsts_dev, long n, hipStream_t st) {
    hipLaunchKernelGGL(k_unpack, dim3(bsite_blocks(n)), dim3(256), 0, st, multi, nr, dsts_dev, n);
}

static inline dim3 lane_dim(long n, int lanes) { return dim3((unsigned)bsite_blocks(n), (unsigned)lanes); }
void launch_lane_copy(zd* dst, long dst_lane, const zd* src, long src_lane, long n, int lanes, const int* mask,
                      hipStream_t st) {
    hipLaunchKernelGGL(k_lane_copy, lane_dim(n, lanes), dim3(256), 0, st, dst, dst_lane, src, src_lane, n, mask);
}
void launch_lane_sub(zd* out, const zd* a, const zd* b, long lane, long n, int lanes, const int* mask, hipStream_t st) {
    hipLaunchKernelGGL(k_lane_sub, lane_dim(n, lanes), dim3(256), 0, st, out, a, b, lane, n, mask);
}
void launch_lane_gather(const zd* const* srcs_dev, zd* dst, long n, int lanes, hipStream_t st) {
    hipLaunchKernelGGL(k_lane_gather, lane_dim(n, lanes), dim3(256), 0, st, srcs_dev, dst, n);
}
void launch_lane_scatter(const zd* src, zd* const* dsts_dev, long n, int lanes, hipStream_t st) {
    hipLaunchKernelGGL(k_lane_scatter, lane_dim(n, lanes), dim3(256), 0, st, src, dsts_dev, n);
}
void launch_relayout(int esize, const void* in, void* out, long rows, int w_old, int w_new, hipStream_t st) {
    const dim3 g(bsite_blocks(rows * w_new)), b(256);
    switch (esize) {
        case 16:
            hipLaunchKernelGGL(k_relayout<V16>, g, b, 0, st, (const V16*)in, (V16*)out, rows, w_old, w_new);
            break;
        case 8:
            hipLaunchKernelGGL(k_relayout<cplx<float>>, g, b, 0, st, (const cplx<float>*)in, (cplx<float>*)out, rows,
                               w_old, w_new);
            break;
        default:
            hipLaunchKernelGGL(k_relayout<float>, g, b, 0, st, (const float*)in, (float*)out, rows, w_old, w_new);
            break;
    }
}
// padding slots of an nr-field: sites vh..stride-1 of each of `groups` groups
// of stride * nr elements (lane fastest)
template <class E>
__global__ void k_zero_padding(E* buf, long groups, int stride, int vh, int nr) {
    const long per = (long)(stride - vh) * nr;
    const E z{};
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < groups * per; t += (long)gridDim.x * blockDim.x) {
        const long g = t / per;
        buf[(g * stride + vh) * nr + (t - g * per)] = z;
    }
}
void launch_zero_padding(int esize, void* buf, long groups, int stride, int vh, int nr, hipStream_t st) {
    if (!buf || stride <= vh) return;
    const dim3 g(bsite_blocks(groups * (stride - vh) * nr)), b(256);
    switch (esize) {
        case 16: hipLaunchKernelGGL(k_zero_padding<V16>, g, b, 0, st, (V16*)buf, groups, stride, vh, nr); break;
        case 8:
            hipLaunchKernelGGL(k_zero_padding<cplx<float>>, g, b, 0, st, (cplx<float>*)buf, groups, stride, vh, nr);
            break;
        default: hipLaunchKernelGGL(k_zero_padding<float>, g, b, 0, st, (float*)buf, groups, stride, vh, nr); break;
    }
}

}  // namespace lym
