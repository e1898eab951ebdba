// lym_device.h -- device-side field access shared by the stencil, the clover
// builder and the solver kernels, generic over the storage precision and the
// number of right-hand sides.
//
// Storage precisions (PR):
//   0  FP64: spinor double2, links double2 / double, clover double2
//   1  FP32: float2 / float, computed in FP32
//   2  FP16: _Float16 pairs, computed in FP32; spinors and clover blocks carry
//      one FP32 scale per site (and right-hand side) = the largest |real|
//      component, so the stored values lie in [-1, 1]; links are unitary
//      (or orthogonal), their entries already lie in [-1, 1] and need no scale.
// Multi-RHS fields store the right-hand side fastest:
//   element (component k, site s, rhs r) at (k * stride + s) * NR + r,
// so the NR lanes that handle one site read one link (a single broadcast
// transaction) and NR consecutive spinor elements.
#pragma once

#include <type_traits>

#include "lym_kernels.h"

#ifndef LYM_NT_LINKS
#define LYM_NT_LINKS 0
#endif

namespace lym {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));

template <int PR>
struct Prec;
template <>
struct Prec<0> {
    typedef double T;
    typedef cplx<double> S;  // complex storage element
    typedef double R;        // real storage element
};
template <>
struct Prec<1> {
    typedef float T;
    typedef cplx<float> S;
    typedef float R;
};
template <>
struct Prec<2> {
    typedef float T;
    typedef h2_t S;
    typedef _Float16 R;
};

// Non-temporal access for data touched once per launch (clover blocks, axpy
// operands, outputs): it streams past L2 instead of evicting the neighbour
// spinors and links that other sites of the launch reuse.
template <class E>
__device__ __forceinline__ E ld_nt_raw(const E* p) {
    if constexpr (sizeof(E) == 16) {
        typedef double v2 __attribute__((ext_vector_type(2)));
        v2 v = __builtin_nontemporal_load(reinterpret_cast<const v2*>(p));
        E e;
        __builtin_memcpy(&e, &v, 16);
        return e;
    } else if constexpr (sizeof(E) == 8) {
        typedef float v2 __attribute__((ext_vector_type(2)));
        v2 v = __builtin_nontemporal_load(reinterpret_cast<const v2*>(p));
        E e;
        __builtin_memcpy(&e, &v, 8);
        return e;
    } else {
        static_assert(sizeof(E) == 4, "element size");
        unsigned v = __builtin_nontemporal_load(reinterpret_cast<const unsigned*>(p));
        E e;
        __builtin_memcpy(&e, &v, 4);
        return e;
    }
}
template <class E>
__device__ __forceinline__ void st_nt_raw(E* p, E e) {
    if constexpr (sizeof(E) == 16) {
        typedef double v2 __attribute__((ext_vector_type(2)));
        v2 v;
        __builtin_memcpy(&v, &e, 16);
        __builtin_nontemporal_store(v, reinterpret_cast<v2*>(p));
    } else if constexpr (sizeof(E) == 8) {
        typedef float v2 __attribute__((ext_vector_type(2)));
        v2 v;
        __builtin_memcpy(&v, &e, 8);
        __builtin_nontemporal_store(v, reinterpret_cast<v2*>(p));
    } else {
        unsigned v;
        __builtin_memcpy(&v, &e, 4);
        __builtin_nontemporal_store(v, reinterpret_cast<unsigned*>(p));
    }
}

__device__ __forceinline__ cplx<double> ld_nt(const cplx<double>* p) { return ld_nt_raw(p); }
__device__ __forceinline__ void st_nt(cplx<double>* p, cplx<double> z) { st_nt_raw(p, z); }

// storage element -> compute complex
template <int PR>
__device__ __forceinline__ cplx<typename Prec<PR>::T> to_c(typename Prec<PR>::S s) {
    if constexpr (PR == 2) return {(float)s.x, (float)s.y};
    else return s;
}
template <int PR>
__device__ __forceinline__ typename Prec<PR>::S from_c(cplx<typename Prec<PR>::T> z) {
    if constexpr (PR == 2) {
        h2_t h;
        h.x = (_Float16)z.re;
        h.y = (_Float16)z.im;
        return h;
    } else {
        return z;
    }
}

// Field access through buffer instructions: a wave-uniform 128-bit resource
// (base address in SGPRs) per component stream plus one 32-bit per-lane byte
// offset shared by all streams of a site index.  Plain pointer arithmetic
// leaves a 64-bit VGPR address per stream (v_lshl_add_u64 for each of the ~230
// loads of a stencil site), which costs registers and occupancy.  Each
// component stream is < 2 GiB.  LYM_BUFFER_LOADS=0 keeps plain loads.
#ifndef LYM_BUFFER_LOADS
#define LYM_BUFFER_LOADS 1
#endif

template <class E>
__device__ __forceinline__ const E* lane_at(const E* ubase, unsigned lane_elems) {
    return reinterpret_cast<const E*>(reinterpret_cast<const char*>(ubase) + lane_elems * (unsigned)sizeof(E));
}
template <class E>
__device__ __forceinline__ E* lane_at(E* ubase, unsigned lane_elems) {
    return reinterpret_cast<E*>(reinterpret_cast<char*>(ubase) + lane_elems * (unsigned)sizeof(E));
}

#if LYM_BUFFER_LOADS
// raw buffer resource for gfx9-family (gfx950): stride 0, 2 GiB range
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)BUF_RANGE, 0x00020000);
}
// cache policy bits of the buffer instructions: 2 = non-temporal
template <class E, int AUX = 0>
__device__ __forceinline__ E buf_ld(const E* ubase, unsigned lane_elems) {
    const __amdgpu_buffer_rsrc_t r = rsrc_of(ubase);
    const unsigned off = lane_elems * (unsigned)sizeof(E);
    E e;
    if constexpr (sizeof(E) == 16) {
        auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, AUX);
        __builtin_memcpy(&e, &v, 16);
    } else if constexpr (sizeof(E) == 8) {
        auto v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, AUX);
        __builtin_memcpy(&e, &v, 8);
    } else if constexpr (sizeof(E) == 4) {
        auto v = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, AUX);
        __builtin_memcpy(&e, &v, 4);
    } else {
        static_assert(sizeof(E) == 2, "element size");
        auto v = __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, AUX);
        __builtin_memcpy(&e, &v, 2);
    }
    return e;
}
template <class E, int AUX = 0>
__device__ __forceinline__ void buf_st(E* ubase, unsigned lane_elems, E e) {
    const __amdgpu_buffer_rsrc_t r = rsrc_of(ubase);
    const unsigned off = lane_elems * (unsigned)sizeof(E);
    if constexpr (sizeof(E) == 16) {
        typedef unsigned v4u __attribute__((ext_vector_type(4)));
        v4u v;
        __builtin_memcpy(&v, &e, 16);
        __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, AUX);
    } else if constexpr (sizeof(E) == 8) {
        typedef unsigned v2u __attribute__((ext_vector_type(2)));
        v2u v;
        __builtin_memcpy(&v, &e, 8);
        __builtin_amdgcn_raw_buffer_store_b64(v, r, off, 0, AUX);
    } else {
        static_assert(sizeof(E) == 4, "element size");
        unsigned v;
        __builtin_memcpy(&v, &e, 4);
        __builtin_amdgcn_raw_buffer_store_b32(v, r, off, 0, AUX);
    }
}
#endif

// element (ubase)[lane] through the chosen path; NT = non-temporal
template <class E, bool NT = false>
__device__ __forceinline__ E fld(const E* ubase, unsigned lane) {
#if LYM_BUFFER_LOADS
    return buf_ld<E, NT ? 2 : 0>(ubase, lane);
#else
    if constexpr (NT && sizeof(E) >= 4) return ld_nt_raw(lane_at(ubase, lane));
    else return *lane_at(ubase, lane);
#endif
}
template <class E, bool NT = true>
__device__ __forceinline__ void fst(E* ubase, unsigned lane, E e) {
#if LYM_BUFFER_LOADS
    buf_st<E, NT ? 2 : 0>(ubase, lane, e);
#else
    if constexpr (NT && sizeof(E) >= 4) st_nt_raw(lane_at(ubase, lane), e);
    else *lane_at(ubase, lane) = e;
#endif
}

// ---------------------------------------------------------------- packed low-precision spinors
// FP32 and FP16 spinor fields store 16-byte vectors of consecutive
// spin-colour components: per parity [G][stride * nr] vectors, G = 6 (two
// float2) or 3 (four half2), lane element (site * nr + rhs).  A lane reads a
// site's spinor with G 16-byte loads instead of 12 8- or 4-byte ones; the
// bytes per site are those of the unpacked [12][stride * nr] layout, so the
// buffers keep their sizes.  FP64 spinors stay [12][stride * nr] double2.
struct alignas(16) V16 {
    unsigned w[4];
};
struct alignas(8) V8 {
    unsigned w[2];
};
template <int PR>
struct Packed {
    static constexpr int PER = 16 / (int)sizeof(typename Prec<PR>::S);  // components per vector
    static constexpr int G = 12 / PER;
};

// parity base pbase (element type S), group stride ks = stride * nr vectors, lane o
template <int PR, bool NT = false>
__device__ __forceinline__ void load_packed(const typename Prec<PR>::S* pbase, size_t ks, unsigned o,
                                            typename Prec<PR>::S e[12]) {
    constexpr int PER = Packed<PR>::PER;
    const V16* b = reinterpret_cast<const V16*>(pbase);
#pragma unroll
    for (int g = 0; g < Packed<PR>::G; ++g) {
        V16 v = fld<V16, NT>(b + g * ks, o);
        __builtin_memcpy(e + g * PER, &v, 16);
    }
}
template <int PR, bool NT = true>
__device__ __forceinline__ void store_packed(typename Prec<PR>::S* pbase, size_t ks, unsigned o,
                                             const typename Prec<PR>::S e[12]) {
    constexpr int PER = Packed<PR>::PER;
    V16* b = reinterpret_cast<V16*>(pbase);
#pragma unroll
    for (int g = 0; g < Packed<PR>::G; ++g) {
        V16 v;
        __builtin_memcpy(&v, e + g * PER, 16);
        fst<V16, NT>(b + g * ks, o, v);
    }
}

// ---------------------------------------------------------------- spinors
// One parity of a (multi-RHS) spinor field.
template <int PR>
struct SpinorRef {
    const typename Prec<PR>::S* base;
    const float* scale;  // PR == 2 only: [stride][NR]
};
template <int PR>
struct SpinorOut {
    typename Prec<PR>::S* base;
    float* scale;
};

template <int PR, bool NT = false>
__device__ __forceinline__ void load_spinor(SpinorRef<PR> f, int stride, int nr, int site, int r,
                                            cplx<typename Prec<PR>::T> s[12]) {
    const unsigned o = (unsigned)site * (unsigned)nr + (unsigned)r;
    const size_t ks = (size_t)stride * nr;
    if constexpr (PR == 0) {
#pragma unroll
        for (int k = 0; k < 12; ++k) s[k] = to_c<PR>(fld<typename Prec<PR>::S, NT>(f.base + k * ks, o));
    } else {
        typename Prec<PR>::S e[12];
        load_packed<PR, NT>(f.base, ks, o, e);
#pragma unroll
        for (int k = 0; k < 12; ++k) s[k] = to_c<PR>(e[k]);
    }
    if constexpr (PR == 2) {
        const float sc = fld<float>(f.scale, o);
#pragma unroll
        for (int k = 0; k < 12; ++k) s[k] = sc * s[k];
    }
}

// The same without the FP16 per-site scale: sc receives it (1 for FP64/FP32),
// so a caller can apply it to a product of fewer components (the stencil
// scales the two projected colour vectors after the link multiply: 12 real
// multiplies per hop instead of 24).
template <int PR>
__device__ __forceinline__ void load_spinor_unscaled(SpinorRef<PR> f, int stride, int nr, int site, int r,
                                                     cplx<typename Prec<PR>::T> s[12], typename Prec<PR>::T& sc) {
    const unsigned o = (unsigned)site * (unsigned)nr + (unsigned)r;
    const size_t ks = (size_t)stride * nr;
    if constexpr (PR == 0) {
#pragma unroll
        for (int k = 0; k < 12; ++k) s[k] = fld<typename Prec<PR>::S>(f.base + k * ks, o);
    } else {
        typename Prec<PR>::S e[12];
        load_packed<PR>(f.base, ks, o, e);
#pragma unroll
        for (int k = 0; k < 12; ++k) s[k] = to_c<PR>(e[k]);
    }
    if constexpr (PR == 2) sc = fld<float>(f.scale, o);
    else sc = (typename Prec<PR>::T)1;
}

// Reciprocal of a per-site FP16 scale m (the site's largest |component|).  A
// site whose m is below the smallest normal float is stored as zero: 1/m of a
// subnormal overflows to inf, and inf * 0 = NaN would poison the vector.  Such
// sites appear where a localised vector (a point source after a few hops)
// decays below 1e-38; they are negligible in FP32 arithmetic anyway.
__device__ __forceinline__ float fp16_site_inv(float& m) {
    if (!(m >= 1.17549435e-38f)) {
        m = 0.f;
        return 0.f;
    }
    return 1.0f / m;
}

template <int PR>
__device__ __forceinline__ void store_spinor(SpinorOut<PR> f, int stride, int nr, int site, int r,
                                             const cplx<typename Prec<PR>::T> v[12]) {
    const unsigned o = (unsigned)site * (unsigned)nr + (unsigned)r;
    const size_t ks = (size_t)stride * nr;
    if constexpr (PR == 2) {
        float m = 0.f;
#pragma unroll
        for (int k = 0; k < 12; ++k) m = fmaxf(m, fmaxf(fabsf(v[k].re), fabsf(v[k].im)));
        const float inv = fp16_site_inv(m);
        typename Prec<PR>::S e[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) e[k] = from_c<PR>(inv * v[k]);
        store_packed<PR>(f.base, ks, o, e);
        fst<float, false>(f.scale, o, m);
    } else if constexpr (PR == 1) {
        typename Prec<PR>::S e[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) e[k] = from_c<PR>(v[k]);
        store_packed<PR>(f.base, ks, o, e);
    } else {
#pragma unroll
        for (int k = 0; k < 12; ++k) fst(f.base + k * ks, o, v[k]);
    }
}

// ---------------------------------------------------------------- link loaders
// LK: 0 complex 18-real, 1 complex 12-real (row 2 = conj(row0 x row1)),
//     2 real 9 (adjoint), 3 real 6 (row 2 = row0 x row1)
template <int LK, class T>
struct LinkMat;
template <class T>
struct LinkMat<0, T> { cplx<T> m[9]; };
template <class T>
struct LinkMat<1, T> { cplx<T> m[9]; };
template <class T>
struct LinkMat<2, T> { T m[9]; };
template <class T>
struct LinkMat<3, T> { T m[9]; };

// ---------------------------------------------------------------- one chirality of a low-precision spinor
// Components 6h .. 6h+5 (spins 2h, 2h+1) of a packed FP32/FP16 spinor, for
// the two-threads-per-site stencil; h must be wave-uniform.  FP32 vectors hold
// components (2g, 2g+1): a chirality is three whole vectors.  FP16 vectors
// hold (4g .. 4g+3): chirality 0 is vector 0 and the low half of vector 1,
// chirality 1 the high half of vector 1 and vector 2.  No scale applied.
template <int PR, bool NT = false>
__device__ __forceinline__ void load_half_lp(const typename Prec<PR>::S* pbase, size_t ks, unsigned o, int h,
                                             typename Prec<PR>::S e[6]) {
    static_assert(PR >= 1, "low precision only");
    const V16* b = reinterpret_cast<const V16*>(pbase);
    if constexpr (PR == 1) {
#pragma unroll
        for (int g = 0; g < 3; ++g) {
            V16 v = fld<V16, NT>(b + (3 * h + g) * ks, o);
            __builtin_memcpy(e + 2 * g, &v, 16);
        }
    } else {
        const V8* b8 = reinterpret_cast<const V8*>(b + ks);  // vector 1 as 8-byte halves
        if (h == 0) {
            V16 v = fld<V16, NT>(b, o);
            V8 w = fld<V8, NT>(b8, 2 * o);
            __builtin_memcpy(e, &v, 16);
            __builtin_memcpy(e + 4, &w, 8);
        } else {
            V8 w = fld<V8, NT>(b8, 2 * o + 1);
            V16 v = fld<V16, NT>(b + 2 * ks, o);
            __builtin_memcpy(e, &w, 8);
            __builtin_memcpy(e + 2, &v, 16);
        }
    }
}
template <int PR>
__device__ __forceinline__ void store_half_lp(typename Prec<PR>::S* pbase, size_t ks, unsigned o, int h,
                                              const typename Prec<PR>::S e[6]) {
    static_assert(PR >= 1, "low precision only");
    V16* b = reinterpret_cast<V16*>(pbase);
    if constexpr (PR == 1) {
#pragma unroll
        for (int g = 0; g < 3; ++g) {
            V16 v;
            __builtin_memcpy(&v, e + 2 * g, 16);
            fst<V16>(b + (3 * h + g) * ks, o, v);
        }
    } else {
        V8* b8 = reinterpret_cast<V8*>(b + ks);
        V16 v;
        V8 w;
        if (h == 0) {
            __builtin_memcpy(&v, e, 16);
            __builtin_memcpy(&w, e + 4, 8);
            fst<V16>(b, o, v);
            fst<V8>(b8, 2 * o, w);
        } else {
            __builtin_memcpy(&w, e, 8);
            __builtin_memcpy(&v, e + 2, 16);
            fst<V8>(b8, 2 * o + 1, w);
            fst<V16>(b + 2 * ks, o, v);
        }
    }
}

// ---------------------------------------------------------------- packed low-precision links
// FP32/FP16 links, rows 0 and 1 (kinds 1 and 3; row 2 is rebuilt: conj(row0 x row1)
// for SU(3), row0 x row1 for the real adjoint links) or all three (kinds 0 and 2),
// packed into 16-, 8- and 4-byte vectors.  Group g of the field is an
// array [2 parity][4 mu][stride] of vectors of its size; the groups follow
// one another.  Bytes per link of two rows: FP32 complex 48 (16+16+16), FP16 complex
// 24 (16+8), FP32 real 24 (16+8), FP16 real 12 (8+4); of three: 72 (4 x 16 + 8), 36
// (16+16+4), 36 (16+16+4), 20 (16+4, the last 2 unused).
// Three rows as 9 single entries took 9 loads a link (72 a site), which the batched
// launches, whose lanes share the links, spent much of their time issuing: the clover
// Schur launches of 8 right-hand sides on 32^3x64 went from 488 to 450 us at FP16 and
// from 1090 to 970 at FP32, on 24^3x48 adjoint links from 150 to 124 at FP16.  (Two
// rows and the rebuild: 456 and 856; the batches keep all rows, which are the FP64
// links rounded once.)
template <int PR, bool REAL, int ROWS>
struct PackedLink {
    static_assert(PR >= 1, "packed links are low-precision only");
    typedef typename std::conditional<REAL, typename Prec<PR>::R, typename Prec<PR>::S>::type E;
    static constexpr int BYTES = link_bytes(PR, REAL, ROWS);
    static constexpr int NE = BYTES / (int)sizeof(E);  // 3 ROWS and the padding
    static constexpr int N16 = BYTES / 16;
    static constexpr bool H8 = (BYTES - 16 * N16) >= 8;
    static constexpr bool H4 = (BYTES - 16 * N16) % 8 == 4;
};

template <int PR, bool REAL, int ROWS>
__device__ __forceinline__ void load_link_rows(const void* base, int stride, int p, int mu, int idx,
                                               typename PackedLink<PR, REAL, ROWS>::E e[3 * ROWS]) {
    typedef PackedLink<PR, REAL, ROWS> P;
    const char* gb = reinterpret_cast<const char*>(base);
    const size_t plane = (size_t)(p * 4 + mu) * stride;
    unsigned char buf[P::BYTES];
    int off = 0;
#pragma unroll
    for (int g = 0; g < P::N16; ++g) {
        V16 v = fld<V16, LYM_NT_LINKS != 0>(reinterpret_cast<const V16*>(gb) + plane, (unsigned)idx);
        __builtin_memcpy(buf + off, &v, 16);
        off += 16;
        gb += (size_t)8 * stride * 16;
    }
    if constexpr (P::H8) {
        V8 v = fld<V8, LYM_NT_LINKS != 0>(reinterpret_cast<const V8*>(gb) + plane, (unsigned)idx);
        __builtin_memcpy(buf + off, &v, 8);
        off += 8;
        gb += (size_t)8 * stride * 8;
    }
    if constexpr (P::H4) {
        unsigned v = fld<unsigned, LYM_NT_LINKS != 0>(reinterpret_cast<const unsigned*>(gb) + plane, (unsigned)idx);
        __builtin_memcpy(buf + off, &v, 4);
    }
    __builtin_memcpy(e, buf, 3 * ROWS * sizeof(typename P::E));
}

// row 2 from rows 0 and 1: conj(row0 x row1), for real links row0 x row1
template <class T>
__device__ __forceinline__ void rebuild_row2(cplx<T> m[9]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int i = (k + 1) % 3, j = (k + 2) % 3;
        cplx<T> t = cmul(m[i], m[3 + j]);
        cfma(t, -m[j], m[3 + i]);
        m[6 + k] = conj(t);
    }
}
template <class T>
__device__ __forceinline__ void rebuild_row2(T m[9]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int i = (k + 1) % 3, j = (k + 2) % 3;
        m[6 + k] = fmadd(-m[j], m[3 + i], m[i] * m[3 + j]);
    }
}

template <int PR, int LK>
__device__ __forceinline__ void load_link(const void* base, int stride, int p, int mu, int idx,
                                          LinkMat<LK, typename Prec<PR>::T>& L) {
    typedef typename Prec<PR>::T T;
    if constexpr (PR >= 1) {
        constexpr bool REAL = LK >= 2;
        constexpr int ROWS = LK & 1 ? 2 : 3;
        typename PackedLink<PR, REAL, ROWS>::E e[3 * ROWS];
        load_link_rows<PR, REAL, ROWS>(base, stride, p, mu, idx, e);
#pragma unroll
        for (int k = 0; k < 3 * ROWS; ++k) {
            if constexpr (REAL) L.m[k] = (T)e[k];
            else L.m[k] = to_c<PR>(e[k]);
        }
        if constexpr (ROWS == 2) rebuild_row2(L.m);
    } else if constexpr (LK == 0 || LK == 1) {
        constexpr int NC = (LK == 0) ? 9 : 6;
        const typename Prec<PR>::S* b =
            reinterpret_cast<const typename Prec<PR>::S*>(base) + (size_t)((p * 4 + mu) * NC) * stride;
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            L.m[k] = to_c<PR>(fld<typename Prec<PR>::S, LYM_NT_LINKS != 0>(b + (size_t)k * stride, (unsigned)idx));
        }
        if constexpr (LK == 1) {
            rebuild_row2(L.m);
        }
    } else {
        constexpr int NC = (LK == 2) ? 9 : 6;
        const typename Prec<PR>::R* b =
            reinterpret_cast<const typename Prec<PR>::R*>(base) + (size_t)((p * 4 + mu) * NC) * stride;
#pragma unroll
        for (int k = 0; k < NC; ++k) L.m[k] = (T)fld<typename Prec<PR>::R, LYM_NT_LINKS != 0>(b + (size_t)k * stride, (unsigned)idx);
        if constexpr (LK == 3) {
            rebuild_row2(L.m);
        }
    }
}

template <int LK, class T>
__device__ __forceinline__ void matvec(const LinkMat<LK, T>& L, const cplx<T> h[3], cplx<T> o[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        if constexpr (LK <= 1) {
            cplx<T> s = cmul(L.m[3 * i], h[0]);
            cfma(s, L.m[3 * i + 1], h[1]);
            cfma(s, L.m[3 * i + 2], h[2]);
            o[i] = s;
        } else {
            o[i] = axpy1(L.m[3 * i + 2], h[2], axpy1(L.m[3 * i + 1], h[1], L.m[3 * i] * h[0]));
        }
    }
}

template <int LK, class T>
__device__ __forceinline__ void matvec_dag(const LinkMat<LK, T>& L, const cplx<T> h[3], cplx<T> o[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        if constexpr (LK <= 1) {
            cplx<T> s = cmulcj(L.m[i], h[0]);
            cfmac(s, L.m[3 + i], h[1]);
            cfmac(s, L.m[6 + i], h[2]);
            o[i] = s;
        } else {
            o[i] = axpy1(L.m[6 + i], h[2], axpy1(L.m[3 + i], h[1], L.m[i] * h[0]));
        }
    }
}

// FP64 single-RHS spinor load (layout.hip, clover.hip)
__device__ __forceinline__ void load_spinor(const cplx<double>* f, int stride, int idx, cplx<double> s[12]) {
#pragma unroll
    for (int k = 0; k < 12; ++k) s[k] = f[(size_t)k * stride + idx];
}

// ---------------------------------------------------------------- clover blocks
// A site's diagonal term is one hermitian 6x6 block per chirality (spins 2h, 2h + 1;
// rows 3 spin + colour), and it is stored as the numbers it is made of.
//  BLK_A       D's block: 1 + [[D, X^H], [X, -D]], D hermitian 3x3, X any 3x3:
//              27 reals (D's diagonal, D_10 D_20 D_21, X by rows)
//  BLK_INV     its inverse: 36 reals (six diagonal entries, the lower ones by rows)
//  BLK_A_REAL, BLK_INV_REAL  the same for real links, whose field strengths are real
//              and antisymmetric: D = i T and X antisymmetric (T real, X complex):
//              9 reals (T_10 T_20 T_21, X_10 X_20 X_21); the inverse
//              [[S + i T, X^H], [X, S - i T]], S real symmetric: 15 reals (S's
//              diagonal, S_10 S_20 S_21, then as above)
// The stencil is bound by memory, and stored as general hermitian blocks (36 reals)
// they were 576 of the 1536 bytes of an FP64 clover apply's site (432 of 1392 now:
// 32^3x64 761 -> 717 us) and 576 of the 1536 and 1728 of a Schur complement's even and
// odd sites on real links (240 and 144 now: 24^3x48 Qhat^2 471 -> 389 us; its FP16
// two-threads-per-site clover launch 59 -> 43 us).
// D and X are stored without the 1, so the FP16 form's per-site scale is theirs.
//
// Layout, for every precision: a plane's block as 16-byte vectors and an 8- and
// a 4-byte rest, piece k of every (plane, site) in one array [nplanes][stride],
// the arrays one after the other (plane = 2 parity + h; h for the inverse).
template <int BK>
inline constexpr bool block_is_A = BK == BLK_A || BK == BLK_A_REAL;

template <int PR, int BK>
struct BlockStore {
    typedef typename Prec<PR>::T T;
    static constexpr int N = block_reals(BK);
    static constexpr int BYTES = block_bytes(PR, BK);
    static constexpr int N16 = BYTES / 16;
    static constexpr bool H8 = (BYTES & 8) != 0, H4 = (BYTES & 4) != 0;
    static constexpr int SLOTS = BYTES / (PR == 0 ? 8 : PR == 1 ? 4 : 2);  // N and the FP16 form's padding
};
template <int PR>
struct BlockReal {
    typedef double E;
};
template <>
struct BlockReal<1> {
    typedef float E;
};
template <>
struct BlockReal<2> {
    typedef _Float16 E;
};

// the block's numbers as stored (FP16: without the site's scale)
template <int PR, int BK, bool NT = true>
__device__ __forceinline__ void load_block(const void* base, int nplanes, int stride, int plane, int idx,
                                           typename Prec<PR>::T e[block_reals(BK)]) {
    typedef BlockStore<PR, BK> P;
    const char* gb = reinterpret_cast<const char*>(base);
    const size_t na = (size_t)nplanes * stride, po = (size_t)plane * stride;
    unsigned char buf[P::BYTES];
#pragma unroll
    for (int k = 0; k < P::N16; ++k) {
        const V16 w = fld<V16, NT>(reinterpret_cast<const V16*>(gb + 16 * na * k) + po, (unsigned)idx);
        __builtin_memcpy(buf + 16 * k, &w, 16);
    }
    gb += 16 * na * P::N16;
    if constexpr (P::H8) {
        const V8 w = fld<V8, NT>(reinterpret_cast<const V8*>(gb) + po, (unsigned)idx);
        __builtin_memcpy(buf + 16 * P::N16, &w, 8);
        gb += 8 * na;
    }
    if constexpr (P::H4) {
        const float w = fld<float, NT>(reinterpret_cast<const float*>(gb) + po, (unsigned)idx);
        __builtin_memcpy(buf + P::BYTES - 4, &w, 4);
    }
    typename BlockReal<PR>::E s[P::SLOTS];
    __builtin_memcpy(s, buf, P::BYTES);
#pragma unroll
    for (int k = 0; k < P::N; ++k) e[k] = (typename Prec<PR>::T)s[k];
}
template <int PR, int BK>
__device__ __forceinline__ void store_block(void* base, int nplanes, int stride, int plane, int idx,
                                            const typename Prec<PR>::T e[block_reals(BK)]) {
    typedef BlockStore<PR, BK> P;
    typename BlockReal<PR>::E s[P::SLOTS];
#pragma unroll
    for (int k = 0; k < P::SLOTS; ++k) s[k] = (typename BlockReal<PR>::E)(k < P::N ? e[k < P::N ? k : 0] : 0);
    char* gb = reinterpret_cast<char*>(base);
    const size_t na = (size_t)nplanes * stride, o = (size_t)plane * stride + idx;
    const char* buf = reinterpret_cast<const char*>(s);
#pragma unroll
    for (int k = 0; k < P::N16; ++k) __builtin_memcpy(gb + 16 * (na * k + o), buf + 16 * k, 16);
    gb += 16 * na * P::N16;
    if constexpr (P::H8) {
        __builtin_memcpy(gb + 8 * o, buf + 16 * P::N16, 8);
        gb += 8 * na;
    }
    if constexpr (P::H4) __builtin_memcpy(gb + 4 * o, buf + P::BYTES - 4, 4);
}

// s += i t b (t real)
template <class T>
__device__ __forceinline__ void ifma(cplx<T>& s, T t, cplx<T> b) {
    s.re = fmadd(-t, b.im, s.re);
    s.im = fmadd(t, b.re, s.im);
}

// o = E v for the numbers e of a block (BLK_A: without the 1)
template <int BK, class T>
__device__ __forceinline__ void block_mul(const T e[block_reals(BK)], const cplx<T> v[6], cplx<T> o[6]) {
    if constexpr (BK == BLK_INV) {
#pragma unroll
        for (int i = 0; i < 6; ++i) o[i] = e[i] * v[i];
        int k = 6;
#pragma unroll
        for (int i = 1; i < 6; ++i) {
#pragma unroll
            for (int j = 0; j < i; ++j) {
                const cplx<T> a = mk(e[k], e[k + 1]);
                cfma(o[i], a, v[j]);
                cfmac(o[j], a, v[i]);
                k += 2;
            }
        }
    } else if constexpr (BK == BLK_A) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            o[i] = e[i] * v[i];
            o[3 + i] = -e[i] * v[3 + i];
        }
        int k = 3;
#pragma unroll
        for (int i = 1; i < 3; ++i) {
#pragma unroll
            for (int j = 0; j < i; ++j) {
                const cplx<T> d = mk(e[k], e[k + 1]), m = mk(-e[k], -e[k + 1]);
                cfma(o[i], d, v[j]);
                cfmac(o[j], d, v[i]);
                cfma(o[3 + i], m, v[3 + j]);
                cfmac(o[3 + j], m, v[3 + i]);
                k += 2;
            }
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) {
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const cplx<T> x = mk(e[k], e[k + 1]);
                cfma(o[3 + i], x, v[j]);
                cfmac(o[j], x, v[3 + i]);
                k += 2;
            }
        }
    } else {
        int k = 0;
        if constexpr (BK == BLK_INV_REAL) {
#pragma unroll
            for (int i = 0; i < 6; ++i) o[i] = e[i % 3] * v[i];
            k = 3;
#pragma unroll
            for (int i = 1; i < 3; ++i) {
#pragma unroll
                for (int j = 0; j < i; ++j) {
#pragma unroll
                    for (int s = 0; s < 6; s += 3) {
                        o[s + i] = axpy1(e[k], v[s + j], o[s + i]);
                        o[s + j] = axpy1(e[k], v[s + i], o[s + j]);
                    }
                    ++k;
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < 6; ++i) o[i] = mk((T)0, (T)0);
        }
#pragma unroll
        for (int i = 1; i < 3; ++i) {
#pragma unroll
            for (int j = 0; j < i; ++j) {
                ifma(o[i], e[k], v[j]);
                ifma(o[j], -e[k], v[i]);
                ifma(o[3 + i], -e[k], v[3 + j]);
                ifma(o[3 + j], e[k], v[3 + i]);
                ++k;
            }
        }
#pragma unroll
        for (int i = 1; i < 3; ++i) {
#pragma unroll
            for (int j = 0; j < i; ++j) {
                const cplx<T> x = mk(e[k], e[k + 1]), m = mk(-e[k], -e[k + 1]);
                cfma(o[3 + i], x, v[j]);
                cfma(o[3 + j], m, v[i]);
                cfmac(o[j], x, v[3 + i]);
                cfmac(o[i], m, v[3 + j]);
                k += 2;
            }
        }
    }
}
// o = the block times v; FP16: sc is the site's scale, put on the outputs.  The 1 is
// added last: the sum's roundings are then those of E v (the FP64 clover apply's
// error 1.6e-16; 2.0e-16 with it first, 1.9e-16 with the 1 stored in the diagonal).
template <int PR, int BK>
__device__ __forceinline__ void block_apply(const typename Prec<PR>::T e[block_reals(BK)], typename Prec<PR>::T sc,
                                            const cplx<typename Prec<PR>::T> v[6], cplx<typename Prec<PR>::T> o[6]) {
    constexpr bool A = block_is_A<BK>;
    block_mul<BK>(e, v, o);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        if constexpr (PR == 2) o[i] = A ? axpy1(sc, o[i], v[i]) : sc * o[i];
        else if constexpr (A) o[i] = v[i] + o[i];
    }
}
template <int PR, int BK, bool NT = true>
__device__ __forceinline__ void block_apply_at(const void* base, int nplanes, int stride, int plane, int idx,
                                               typename Prec<PR>::T sc, const cplx<typename Prec<PR>::T> v[6],
                                               cplx<typename Prec<PR>::T> o[6]) {
    typename Prec<PR>::T e[block_reals(BK)];
    load_block<PR, BK, NT>(base, nplanes, stride, plane, idx, e);
    block_apply<PR, BK>(e, sc, v, o);
}

}  // namespace lym
