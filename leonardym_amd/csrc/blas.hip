// blas.hip -- spinor BLAS-1 and the device-resident CG / BiCGStab state machines.
//
// Reductions (AlgebraUtils::squaredNorm, dot, gamma5dot, differenceNorm,
// source/algebra_utils/AlgebraUtils.h:17-27,182-254) run on a fixed grid of
// RED_BLOCKS workgroups: each wavefront folds its lanes with xor-shuffles,
// the workgroup folds its waves through LDS and writes one partial per
// workgroup; a single-workgroup second pass folds the partials in a fixed
// tree.  The order of every addition is therefore fixed, so a result does not
// depend on what else runs on the device (the reference sums in long double;
// here every sum is FP64).
//
// The solver kernels keep all scalars (alpha, beta, rho, omega, |r|^2) in a
// device state block, so an iteration needs no host round trip; every kernel
// returns at once when the state says `done`, which makes the iteration
// count and stopping point those of the reference loops
// (source/inverters/ConjugateGradient.cpp:33-67, BiConjugateGradient.cpp:364-501)
// however many iterations the host has queued.
#include "lym_kernels.h"

namespace lym {

constexpr int RB_THREADS = 256;

template <int NV>
__device__ __forceinline__ void wave_sum(double v[NV]) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < NV; ++k) v[k] += __shfl_xor(v[k], off, 64);
}

// block of RB_THREADS threads -> partials[k * stride + blockIdx.x]
template <int NV>
__device__ __forceinline__ void block_store(double v[NV], double* partials, int stride = RED_BLOCKS) {
    __shared__ double sh[NV][RB_THREADS / 64];
    wave_sum<NV>(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[k][w] = v[k];
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            double s = 0;
#pragma unroll
            for (int j = 0; j < RB_THREADS / 64; ++j) s += sh[k][j];
            partials[(size_t)k * stride + blockIdx.x] = s;
        }
    }
}

// one block of RED_BLOCKS threads folds the partials; thread 0 returns totals
template <int NV>
__device__ __forceinline__ void final_sum(const double* partials, double out[NV]) {
    __shared__ double sh[NV][RED_BLOCKS / 64];
    double v[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = partials[k * RED_BLOCKS + threadIdx.x];
    wave_sum<NV>(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[k][w] = v[k];
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            double s = 0;
#pragma unroll
            for (int j = 0; j < RED_BLOCKS / 64; ++j) s += sh[k][j];
            out[k] = s;
        }
}

// The totals of NV sums of n <= FOLD_MAX partials each (sum k of workgroup b at
// partials[k * stride + b]), folded by every workgroup of RB_THREADS threads that
// needs them (the same fixed order in each, so all get the same values): the
// partials are loaded first (fold_load), the caller may then issue its own
// loads, and fold_block folds across the workgroup (result in every thread).
template <int NV>
__device__ __forceinline__ void fold_load(const double* partials, int stride, int n, double pl[NV]) {
#pragma unroll
    for (int k = 0; k < NV; ++k) pl[k] = 0;
    for (int i = (int)threadIdx.x; i < n; i += RB_THREADS)
#pragma unroll
        for (int k = 0; k < NV; ++k) pl[k] += partials[(size_t)k * stride + i];
}
template <int NV>
__device__ __forceinline__ void fold_block(const double pl[NV], double out[NV]) {
    __shared__ double sh[NV][RB_THREADS / 64];
    double v[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = pl[k];
    wave_sum<NV>(v);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[k][threadIdx.x >> 6] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        double t = 0;
#pragma unroll
        for (int j = 0; j < RB_THREADS / 64; ++j) t += sh[k][j];
        out[k] = t;
    }
    __syncthreads();
}

// more than FOLD_MAX partials: one workgroup folds each sum into one
template <int NV>
__global__ __launch_bounds__(1024) void k_fold(const double* partials, int stride, int n, double* out,
                                               const int* skip) {
    if (skip && *skip) return;
    __shared__ double sh[NV][16];
    double v[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = 0;
    for (int i = (int)threadIdx.x; i < n; i += 1024)
#pragma unroll
        for (int k = 0; k < NV; ++k) v[k] += partials[(size_t)k * stride + i];
    wave_sum<NV>(v);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[k][threadIdx.x >> 6] = v[k];
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            double t = 0;
            for (int j = 0; j < 16; ++j) t += sh[k][j];
            out[(size_t)k * stride] = t;
        }
}

void launch_fold(int nv, const double*& part, int stride, int& npart, double* out, const int* skip, hipStream_t st) {
    if (npart <= FOLD_MAX) return;
    if (nv == 1) hipLaunchKernelGGL(k_fold<1>, dim3(1), dim3(1024), 0, st, part, stride, npart, out, skip);
    else hipLaunchKernelGGL(k_fold<3>, dim3(1), dim3(1024), 0, st, part, stride, npart, out, skip);
    part = out;
    npart = 1;
}

#define GRID_LOOP(i, n) for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += (long)gridDim.x * blockDim.x)

// ---------------------------------------------------------------- plain reductions
__global__ __launch_bounds__(RB_THREADS) void k_norm2(const zd* __restrict__ a, long n, double* partials) {
    double v[1] = {0};
    GRID_LOOP(i, n) {
        zd x = a[i];
        v[0] += x.re * x.re + x.im * x.im;
    }
    block_store<1>(v, partials);
}

__global__ __launch_bounds__(RB_THREADS) void k_dot(const zd* __restrict__ a, const zd* __restrict__ b, long n,
                                                    double* partials) {
    double v[2] = {0, 0};
    GRID_LOOP(i, n) {
        zd x = a[i], y = b[i];
        v[0] += x.re * y.re + x.im * y.im;
        v[1] += x.re * y.im - x.im * y.re;
    }
    block_store<2>(v, partials);
}

__global__ __launch_bounds__(RB_THREADS) void k_gamma5dot(const zd* __restrict__ a, const zd* __restrict__ b, long n,
                                                          int stride, double* partials) {
    double v[2] = {0, 0};
    GRID_LOOP(i, n) {
        zd x = a[i], y = b[i];
        double s = ((i / stride) % 12) < 6 ? 1.0 : -1.0;
        v[0] += s * (x.re * y.re + x.im * y.im);
        v[1] += s * (x.re * y.im - x.im * y.re);
    }
    block_store<2>(v, partials);
}

__global__ __launch_bounds__(RB_THREADS) void k_diffnorm(const zd* __restrict__ a, const zd* __restrict__ b, long n,
                                                         double* partials) {
    double v[1] = {0};
    GRID_LOOP(i, n) {
        zd d = a[i] - b[i];
        v[0] += d.re * d.re + d.im * d.im;
    }
    block_store<1>(v, partials);
}

template <int NV>
__global__ __launch_bounds__(RED_BLOCKS) void k_final(const double* partials, double* result) {
    double out[NV];
    final_sum<NV>(partials, out);
    if (threadIdx.x == 0)
        for (int k = 0; k < NV; ++k) result[k] = out[k];
}

void launch_norm2(const zd* a, long n, double* partials, double* result, hipStream_t st) {
    hipLaunchKernelGGL(k_norm2, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, a, n, partials);
    hipLaunchKernelGGL(k_final<1>, dim3(1), dim3(RED_BLOCKS), 0, st, partials, result);
}
void launch_dot(const zd* a, const zd* b, long n, double* partials, double* result, hipStream_t st) {
    hipLaunchKernelGGL(k_dot, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, a, b, n, partials);
    hipLaunchKernelGGL(k_final<2>, dim3(1), dim3(RED_BLOCKS), 0, st, partials, result);
}
void launch_gamma5dot(const zd* a, const zd* b, long n, int nparity, int stride, double* partials, double* result,
                      hipStream_t st) {
    (void)nparity;
    hipLaunchKernelGGL(k_gamma5dot, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, a, b, n, stride, partials);
    hipLaunchKernelGGL(k_final<2>, dim3(1), dim3(RED_BLOCKS), 0, st, partials, result);
}
void launch_diffnorm(const zd* a, const zd* b, long n, double* partials, double* result, hipStream_t st) {
    hipLaunchKernelGGL(k_diffnorm, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, a, b, n, partials);
    hipLaunchKernelGGL(k_final<1>, dim3(1), dim3(RED_BLOCKS), 0, st, partials, result);
}

// ---------------------------------------------------------------- elementwise
// one element per thread (grid-stride only beyond 2^28 elements): on the
// MI355X a copy with one element per thread streams at 6.2 TB/s, the same
// copy as a grid-stride loop over 8192 workgroups at 5.1 TB/s
static inline int ew_blocks(long n) {
    long b = (n + 255) / 256;
    return (int)(b < (1L << 20) ? b : (1L << 20));
}

__global__ void k_axpy(zd* __restrict__ y, zd a, const zd* __restrict__ x, long n) {
    GRID_LOOP(i, n) { y[i] = y[i] + a * x[i]; }
}
__global__ void k_xpay(zd* __restrict__ y, const zd* __restrict__ x, zd a, long n) {
    GRID_LOOP(i, n) { y[i] = x[i] + a * y[i]; }
}
__global__ void k_g5(zd* __restrict__ y, long n, int stride) {
    GRID_LOOP(i, n) {
        if (((i / stride) % 12) >= 6) y[i] = -y[i];
    }
}
__global__ void k_copy(zd* __restrict__ y, const zd* __restrict__ x, long n) {
    GRID_LOOP(i, n) { y[i] = x[i]; }
}
__global__ void k_sub(zd* __restrict__ o, const zd* __restrict__ a, const zd* __restrict__ b, long n) {
    GRID_LOOP(i, n) { o[i] = a[i] - b[i]; }
}

void launch_axpy(zd* y, zd a, const zd* x, long n, hipStream_t st) {
    hipLaunchKernelGGL(k_axpy, dim3(ew_blocks(n)), dim3(256), 0, st, y, a, x, n);
}
void launch_xpay(zd* y, const zd* x, zd a, long n, hipStream_t st) {
    hipLaunchKernelGGL(k_xpay, dim3(ew_blocks(n)), dim3(256), 0, st, y, x, a, n);
}
void launch_scale_g5(zd* y, int nparity, int stride, hipStream_t st) {
    long n = (long)nparity * 12 * stride;
    hipLaunchKernelGGL(k_g5, dim3(ew_blocks(n)), dim3(256), 0, st, y, n, stride);
}
__global__ void k_set_double(double* p, double v) { *p = v; }
void launch_set_double(double* p, double v, hipStream_t st) {
    hipLaunchKernelGGL(k_set_double, dim3(1), dim3(1), 0, st, p, v);
}

void launch_copy(zd* y, const zd* x, long n, hipStream_t st) {
    hipLaunchKernelGGL(k_copy, dim3(ew_blocks(n)), dim3(256), 0, st, y, x, n);
}
void launch_sub(zd* o, const zd* a, const zd* b, long n, hipStream_t st) {
    hipLaunchKernelGGL(k_sub, dim3(ew_blocks(n)), dim3(256), 0, st, o, a, b, n);
}

// ---------------------------------------------------------------- CG
__global__ __launch_bounds__(RED_BLOCKS) void k_cg_init_final(CGState* s, const double* partials, double eps,
                                                              int max_steps) {
    double out[1];
    final_sum<1>(partials, out);
    if (threadIdx.x == 0) {
        s->rr = out[0];
        s->rr_new = out[0];
        s->eps = eps;
        s->max_steps = max_steps;
        s->step = 0;
        s->converged = 0;
        s->done = max_steps <= 0 ? 1 : 0;
        s->alpha_re = s->alpha_im = s->beta = 0;
    }
}

void launch_cg_init(CGState* s, const zd* r, long n, double* partials, double eps, int max_steps, hipStream_t st) {
    hipLaunchKernelGGL(k_norm2, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, r, n, partials);
    hipLaunchKernelGGL(k_cg_init_final, dim3(1), dim3(RED_BLOCKS), 0, st, s, partials, eps, max_steps);
}

__global__ __launch_bounds__(RB_THREADS) void k_cg_dot(const CGState* s, const zd* __restrict__ p,
                                                       const zd* __restrict__ Ap, long n, double* partials) {
    if (s->done) return;
    double v[2] = {0, 0};
    GRID_LOOP(i, n) {
        zd x = p[i], y = Ap[i];
        v[0] += x.re * y.re + x.im * y.im;
        v[1] += x.re * y.im - x.im * y.re;
    }
    block_store<2>(v, partials);
}

void launch_cg_alpha(CGState* s, const zd* p, const zd* Ap, long n, double* partials, hipStream_t st) {
    hipLaunchKernelGGL(k_cg_dot, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, s, p, Ap, n, partials);
}

// alpha = |r|^2 / <p, A p> (complex, ConjugateGradient.cpp:36), folded by
// every workgroup from the <p, Ap> partials; then x += alpha p, r -= alpha Ap,
// partial |r|^2.  Workgroup 0 records alpha and the |r|^2 the p update
// divides by.
__global__ __launch_bounds__(RB_THREADS) void k_cg_update(CGState* s, zd* __restrict__ x, zd* __restrict__ r,
                                                          const zd* __restrict__ p, const zd* __restrict__ Ap, long n,
                                                          const double* dot_partials, double* partials) {
    if (s->done) return;
    double pl[2];
    fold_load<2>(dot_partials, RED_BLOCKS, RED_BLOCKS, pl);
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long istep = (long)gridDim.x * blockDim.x;
    zd xv, rv, pv, av;
    if (i < n) {
        xv = x[i];
        rv = r[i];
        pv = p[i];
        av = Ap[i];
    }
    double d[2];
    fold_block<2>(pl, d);
    const double den = d[0] * d[0] + d[1] * d[1];
    const zd al = mk(s->rr * d[0] / den, -s->rr * d[1] / den);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        s->alpha_re = al.re;
        s->alpha_im = al.im;
        s->rr_prev = s->rr;
    }
    double v[1] = {0};
    while (i < n) {
        x[i] = xv + al * pv;
        const zd rn = rv - al * av;
        r[i] = rn;
        v[0] += rn.re * rn.re + rn.im * rn.im;
        i += istep;
        if (i < n) {
            xv = x[i];
            rv = r[i];
            pv = p[i];
            av = Ap[i];
        }
    }
    block_store<1>(v, partials);
}

void launch_cg_update(CGState* s, zd* x, zd* r, const zd* p, const zd* Ap, long n, double* partials,
                      hipStream_t st) {
    // <p, Ap> partials in slots 0 and 1 (launch_cg_alpha), |r|^2 in slot 2
    hipLaunchKernelGGL(k_cg_update, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, s, x, r, p, Ap, n, partials,
                       partials + 2 * RED_BLOCKS);
}

// |r|^2 folded by every workgroup from the update's partials; workgroup 0
// advances the state (ConjugateGradient.cpp:49-50: stop at |r|^2 < eps, else
// beta = |r|^2 / |r_prev|^2, step + 1); then p = r + beta p.  Only workgroup 0
// writes the state and no workgroup reads what it writes except `done` at the
// start (read once per workgroup: after a stop decided here p may be left
// partly updated, which nothing reads).
__global__ __launch_bounds__(RB_THREADS) void k_cg_p(CGState* s, zd* __restrict__ p, const zd* __restrict__ r, long n,
                                                     const double* rpart, int npart) {
    __shared__ int stop;
    if (threadIdx.x == 0) stop = s->done;
    __syncthreads();
    if (stop) return;
    double pl[1];
    fold_load<1>(rpart, 0, npart, pl);
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long istep = (long)gridDim.x * blockDim.x;
    zd pv, rv;
    if (i < n) {
        pv = p[i];
        rv = r[i];
    }
    double rn[1];
    fold_block<1>(pl, rn);
    const double b = rn[0] / s->rr_prev;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        s->rr_new = rn[0];
        if (rn[0] < s->eps) {
            s->done = 1;
            s->converged = 1;
        } else {
            s->beta = b;
            s->rr = rn[0];
            s->step += 1;
            if (s->step >= s->max_steps) s->done = 1;
        }
    }
    while (i < n) {
        p[i] = rv + b * pv;
        i += istep;
        if (i < n) {
            pv = p[i];
            rv = r[i];
        }
    }
}

void launch_cg_p(CGState* s, zd* p, const zd* r, long n, const double* part, int npart, hipStream_t st) {
    hipLaunchKernelGGL(k_cg_p, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, s, p, r, n, part, npart);
}

// ---------------------------------------------------------------- BiCGStab
__device__ __forceinline__ zd zdiv(zd a, zd b) {
    double den = b.re * b.re + b.im * b.im;
    return mk((a.re * b.re + a.im * b.im) / den, (a.im * b.re - a.re * b.im) / den);
}

__global__ void k_bicg_init(BiCGState* s, double precision, int max_steps) {
    s->rho_re = 1; s->rho_im = 0;
    s->alpha_re = 1; s->alpha_im = 0;
    s->omega_re = 1; s->omega_im = 0;
    s->rhon_re = s->rhon_im = s->beta_re = s->beta_im = 0;
    s->norm = 0;
    s->precision = precision;
    s->max_steps = max_steps;
    s->step = 0;
    s->converged = 0;
    s->breakdown = 0;
    s->copy_b = 0;
    s->phase = BICG_FIRST;
    s->done = max_steps <= 0 ? 1 : 0;
}

void launch_bicg_init(BiCGState* s, double precision, int max_steps, hipStream_t st) {
    hipLaunchKernelGGL(k_bicg_init, dim3(1), dim3(1), 0, st, s, precision, max_steps);
}

// v += <rh, r> and |r|^2 of one element
__device__ __forceinline__ void bicg_terms(zd rh, zd r, double v[3]) {
    v[0] += rh.re * r.re + rh.im * r.im;
    v[1] += rh.re * r.im - rh.im * r.re;
    v[2] += r.re * r.re + r.im * r.im;
}

__global__ __launch_bounds__(RB_THREADS) void k_bicg_setup(zd* __restrict__ r, zd* __restrict__ rh,
                                                           zd* __restrict__ p, zd* __restrict__ nu,
                                                           const zd* __restrict__ b, const zd* __restrict__ Ax,
                                                           long n, double* partials, int stride) {
    double v[3] = {0, 0, 0};
    GRID_LOOP(i, n) {
        const zd bb = b[i], ax = Ax[i], ri = bb - ax, hi = bb + ax;
        r[i] = ri;
        rh[i] = hi;
        p[i] = mk(0.0, 0.0);
        nu[i] = mk(0.0, 0.0);
        bicg_terms(hi, ri, v);
    }
    block_store<3>(v, partials, stride);
}

void launch_bicg_setup(zd* r, zd* rh, zd* p, zd* nu, const zd* b, const zd* Ax, long n, double* partials, int stride,
                       hipStream_t st) {
    hipLaunchKernelGGL(k_bicg_setup, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, r, rh, p, nu, b, Ax, n, partials,
                       stride);
}

__global__ __launch_bounds__(RB_THREADS) void k_bicg_dot(const BiCGState* s, const zd* __restrict__ w,
                                                         const zd* __restrict__ v, long n, double* partials,
                                                         int stride) {
    if (s->done) return;
    double t[3] = {0, 0, 0};
    GRID_LOOP(i, n) { bicg_terms(w[i], v[i], t); }
    block_store<3>(t, partials, stride);
}

void launch_bicg_dot(const BiCGState* s, const zd* w, const zd* v, long n, double* partials, int stride,
                     hipStream_t st) {
    hipLaunchKernelGGL(k_bicg_dot, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, s, w, v, n, partials, stride);
}

// Each of the p, s and x/r updates below folds the partial sums of the step
// before it in every workgroup (a fixed order, so all get the same value);
// workgroup 0 writes the state.  No other workgroup reads what it writes, but for
// two members: `done` (once per workgroup, at the start: a workgroup that starts
// after a stop returns at once and leaves its part of a vector as it was, so a
// kernel whose vector is still to be read never sets it), and `step` in the p
// update, which changes there only when every workgroup returns without updating.
#define BICG_STOP_CHECK()                        \
    __shared__ int stop_;                        \
    if (threadIdx.x == 0) stop_ = s->done;      \
    __syncthreads();                             \
    if (stop_) return

// |r|^2 < precision after the last update: converged at its step; else that step
// is over, at most max_steps of them (BiConjugateGradient.cpp:480-501).  Returns
// whether the solve stops; wr: this thread writes the state.
__device__ __forceinline__ bool bicg_stop(BiCGState* s, double norm, int step, bool wr) {
    const bool conv = norm < s->precision, last = step + 1 >= s->max_steps;
    if (wr) {
        s->norm = norm;
        if (conv) {
            s->converged = 1;
            s->done = 1;
        } else if (last) {
            s->step = step + 1;
            s->done = 1;
        }
    }
    return conv || last;
}

// The last update's stopping rule, then rho_next = <rh, r>; breakdown if zero;
// beta = (rho_next / rho)(alpha / omega); p = r + beta (p - omega nu)
__global__ __launch_bounds__(RB_THREADS) void k_bicg_p(BiCGState* s, zd* __restrict__ p, const zd* __restrict__ r,
                                                       const zd* __restrict__ nu, long n, const double* partials,
                                                       int stride, int npart) {
    BICG_STOP_CHECK();
    const bool wr = blockIdx.x == 0 && threadIdx.x == 0;
    if (s->copy_b) {  // the last update copied the source into x: the solve is over
        if (wr) s->done = 1;
        return;
    }
    const int phase = s->phase, step = s->step;
    double pl[3];
    fold_load<3>(partials, stride, npart, pl);
    double out[3];
    fold_block<3>(pl, out);
    if (phase == BICG_FOLD && bicg_stop(s, out[2], step, wr)) return;
    const zd rn = mk(out[0], out[1]);
    const bool brk = rn.re * rn.re + rn.im * rn.im == 0.0;
    const zd om = mk(s->omega_re, s->omega_im);
    const zd beta = zdiv(rn, mk(s->rho_re, s->rho_im)) * zdiv(mk(s->alpha_re, s->alpha_im), om);
    if (wr) {
        s->rhon_re = rn.re;
        s->rhon_im = rn.im;
        if (brk) {
            if (phase == BICG_FOLD) s->step = step + 1;
            s->done = 1;
            s->breakdown = 1;
            s->converged = 0;
        } else {
            s->beta_re = beta.re;
            s->beta_im = beta.im;
        }
    }
    if (brk) return;
    GRID_LOOP(i, n) { p[i] = r[i] + beta * (p[i] - om * nu[i]); }
}

void launch_bicg_p(BiCGState* s, zd* p, const zd* r, const zd* nu, long n, const double* partials, int stride,
                   hipStream_t st) {
    hipLaunchKernelGGL(k_bicg_p, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, s, p, r, nu, n, partials, stride,
                       RED_BLOCKS);
}

// alpha = rho_next / <rh, nu>; s = r - alpha nu.  Workgroup 0 also moves rho_next
// to rho and counts the step the p update has closed.
__global__ __launch_bounds__(RB_THREADS) void k_bicg_s(BiCGState* s, zd* __restrict__ sv, const zd* __restrict__ r,
                                                       const zd* __restrict__ nu, long n, const double* part,
                                                       int stride, int npart) {
    BICG_STOP_CHECK();
    double pl[2];
    fold_load<2>(part, stride, npart, pl);
    double out[2];
    fold_block<2>(pl, out);
    const zd rhon = mk(s->rhon_re, s->rhon_im), al = zdiv(rhon, mk(out[0], out[1]));
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        s->alpha_re = al.re;
        s->alpha_im = al.im;
        s->rho_re = rhon.re;
        s->rho_im = rhon.im;
        if (s->phase == BICG_FOLD) s->step += 1;
        s->phase = BICG_FOLD;
    }
    GRID_LOOP(i, n) { sv[i] = r[i] - al * nu[i]; }
}

void launch_bicg_s(BiCGState* s, zd* sv, const zd* r, const zd* nu, long n, const double* part, int stride, int npart,
                   hipStream_t st) {
    hipLaunchKernelGGL(k_bicg_s, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, s, sv, r, nu, n, part, stride, npart);
}

// omega = <t,s>/<t,t> from <s,t> and |t|^2; <t,t> == 0 -> solution = source
// (BiConjugateGradient.cpp:449-458); x += alpha p + omega s, r = s - omega t,
// partial <rh, r> and |r|^2
__global__ __launch_bounds__(RB_THREADS) void k_bicg_update(BiCGState* s, zd* __restrict__ x, zd* __restrict__ r,
                                                            const zd* __restrict__ rh, const zd* __restrict__ p,
                                                            const zd* __restrict__ sv, const zd* __restrict__ t,
                                                            const zd* __restrict__ b, long n, const double* part,
                                                            int stride, int npart, double* partials) {
    BICG_STOP_CHECK();
    double pl[3];
    fold_load<3>(part, stride, npart, pl);
    double out[3];
    fold_block<3>(pl, out);
    if (out[2] == 0.0) {
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            s->copy_b = 1;  // (`done` by the next p update or launch_bicg_check)
            s->converged = 1;
        }
        GRID_LOOP(i, n) { x[i] = b[i]; }
        return;
    }
    const zd om = mk(out[0] / out[2], -out[1] / out[2]);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        s->omega_re = om.re;
        s->omega_im = om.im;
    }
    const zd al = mk(s->alpha_re, s->alpha_im);
    double v[3] = {0, 0, 0};
    GRID_LOOP(i, n) {
        const zd sv_i = sv[i];
        x[i] = x[i] + al * p[i] + om * sv_i;
        const zd rn = sv_i - om * t[i];
        r[i] = rn;
        bicg_terms(rh[i], rn, v);
    }
    block_store<3>(v, partials, stride);
}

void launch_bicg_update(BiCGState* s, zd* x, zd* r, const zd* rh, const zd* p, const zd* sv, const zd* t, const zd* b,
                        long n, const double* part, int stride, int npart, double* partials, hipStream_t st) {
    hipLaunchKernelGGL(k_bicg_update, dim3(RED_BLOCKS), dim3(RB_THREADS), 0, st, s, x, r, rh, p, sv, t, b, n, part,
                       stride, npart, partials);
}

__global__ __launch_bounds__(RB_THREADS) void k_bicg_check(BiCGState* s, const double* partials, int stride,
                                                           int npart) {
    if (s->done || s->phase != BICG_FOLD) return;
    if (s->copy_b) {
        if (threadIdx.x == 0) s->done = 1;
        return;
    }
    double pl[3], out[3];
    fold_load<3>(partials, stride, npart, pl);
    fold_block<3>(pl, out);
    if (threadIdx.x == 0 && !bicg_stop(s, out[2], s->step, true)) {
        s->step += 1;
        s->phase = BICG_CHECKED;
    }
}

void launch_bicg_check(BiCGState* s, const double* partials, int stride, hipStream_t st) {
    hipLaunchKernelGGL(k_bicg_check, dim3(1), dim3(RB_THREADS), 0, st, s, partials, stride, RED_BLOCKS);
}

}  // namespace lym

namespace lym {

__device__ __forceinline__ uint64_t mix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__global__ void k_fill_uniform(zd* x, long n, int stride, int Vh, uint64_t seed) {
    GRID_LOOP(i, n) {
        if ((int)(i % stride) >= Vh) {
            x[i] = mk(0.0, 0.0);
        } else {
            uint64_t a = mix64(seed ^ mix64(2 * (uint64_t)i)), b = mix64(seed ^ mix64(2 * (uint64_t)i + 1));
            x[i] = mk((a >> 11) * 0x1.0p-53, (b >> 11) * 0x1.0p-53);
        }
    }
}

void launch_fill_uniform(zd* x, int nparity, int stride, int Vh, uint64_t seed, hipStream_t st) {
    long n = (long)nparity * 12 * stride;
    hipLaunchKernelGGL(k_fill_uniform, dim3(ew_blocks(n)), dim3(256), 0, st, x, n, stride, Vh, seed);
}

}  // namespace lym
