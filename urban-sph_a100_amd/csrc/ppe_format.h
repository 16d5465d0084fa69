// Sliced-ELLPACK storage of the PPE operator and its row product, shared
// by the Krylov kernels and the multigrid preconditioner.
#pragma once
#include "sph_internal.h"

namespace sph {

// V-cycle weights of the multigrid preconditioner: damped Jacobi smoothing
// x = w b / diag, and the over-correction of unsmoothed aggregation
constexpr double MG_OMEGA = 0.9;
constexpr double MG_SCALE = 1.5;

// 16-bit column entries: 10 offset bits, up to 64 window groups per slice
constexpr int EC_OFF_BITS = 10;
constexpr int EC_OFF_MASK = (1 << EC_OFF_BITS) - 1;
constexpr int EC_MAX_GROUPS = 64;
constexpr int EC_MAX_WORDS = (65536 * 256 >> 10) >> 5;   // window bitmap words for 16.7M unknowns

// Matrix layout: sliced ELLPACK over 64-row slices, one wave64 per slice,
// entries column-major within a slice: entry k of row r lives at
//     sl_off[r / 64] + k * 64 + r % 64,
// so the wave's loads of one slot are one contiguous block.
__host__ __device__ __forceinline__ long long prow(const long long* sl_off, int r) {
    return sl_off[r >> 6] + (r & 63);
}
__host__ __device__ __forceinline__ long long pslot(int k) { return (long long)k * SLICE; }

// Off-diagonal part of one row, sum_k vals[k] * x[col[k]], accumulated in
// double in entry order: ld(k) loads entry k's operands, mac(s, operands)
// adds its term.  U entries' loads are issued before the
// first of their terms is added, in the remainder too (entries past the
// row's end reload the last one and add nothing): a small case has about
// a wave a SIMD, and its product takes the number of such rounds times the
// memory latency.  Measured with 4 (and a remainder entry by entry), 8, 16
// and 24 entries a round, HIP events, operators read past the caches: float
// product 29.9, 21.4, 16.9, 16.0 us on 20,609 particles and 137, 132, 131,
// 143 us on the 2.13 M canyon, whose level-0 passes (half values) take 94, 83,
// 83, 104 us; double product (150 k canyon) 36.3, 36.9, 39.9, 43.5 us, through
// the caches with 8 and 16: 27.9, 30.9, and 21.3, 20.8 us on the 32^3 box.
// Giving a row to four waves (an LDS sum) was slower from 200 k particles on
// and no faster below.
constexpr int ROW_U = 16;        // float and half values
constexpr int ROW_U_F64 = 8;
template <class T, int U, class LD, class MAC>
__device__ __forceinline__ double row_sum(int m, LD&& ld, MAC&& mac) {
    double s = 0.0;
    int k = 0;
    for (; k + U <= m; k += U) {
        T t[U];
#pragma unroll
        for (int u = 0; u < U; u++) t[u] = ld(k + u);
#pragma unroll
        for (int u = 0; u < U; u++) s = mac(s, t[u]);
    }
    if (k < m) {
        T t[U];
#pragma unroll
        for (int u = 0; u < U; u++) t[u] = ld(min(k + u, m - 1));
#pragma unroll
        for (int u = 0; u < U; u++) s = k + u < m ? mac(s, t[u]) : s;
    }
    return s;
}
template <class V, class X> struct Term { V v; X x; };
template <class V> constexpr int row_u() { return sizeof(V) == 8 ? ROW_U_F64 : ROW_U; }
// The same for double entries with stored columns: while a round's x values
// are gathered, the next round's entries are on their way, so a round costs one
// memory latency, not two.  32^3 box 21.3 -> 18.8 us a product, 4 k 15.9 -> 15.3,
// 150 k canyon the same 27; the float products, 16 entries a round, lose more
// waves to the registers than they gain (35 -> 40 us on 300 k, 130 -> 148 on
// 2.13 M).  ld(k): entry k; x_of(entry): its x; val(entry): its value.
template <class E, class X, int U, class LD, class XOF, class VAL>
__device__ __forceinline__ double row_sum_cols(int m, LD&& ld, XOF&& x_of, VAL&& val) {
    double s = 0.0;
    if (m <= 0) return s;
    E a[U];
#pragma unroll
    for (int u = 0; u < U; u++) a[u] = ld(min(u, m - 1));
    int k = 0;
    for (; k + U < m; k += U) {
        X x[U];
        E b[U];
#pragma unroll
        for (int u = 0; u < U; u++) x[u] = x_of(a[u]);
#pragma unroll
        for (int u = 0; u < U; u++) b[u] = ld(min(k + U + u, m - 1));
#pragma unroll
        for (int u = 0; u < U; u++) s += (double)val(a[u]) * (double)x[u];
#pragma unroll
        for (int u = 0; u < U; u++) a[u] = b[u];
    }
    X x[U];
#pragma unroll
    for (int u = 0; u < U; u++) x[u] = x_of(a[u]);
#pragma unroll
    for (int u = 0; u < U; u++) s = k + u < m ? s + (double)val(a[u]) * (double)x[u] : s;
    return s;
}
template <class V, class C> struct Entry { V v; C c; };
template <class V, class X, bool NT>
__device__ __forceinline__ double offdiag_i32(const int* cp, const V* vp, int m, const X* x) {
    if constexpr (sizeof(V) == 8) {
        typedef Entry<V, int> E;
        return row_sum_cols<E, X, row_u<V>()>(
            m, [&](int k) { return E{ld_matrix<NT>(vp + pslot(k)), ld_matrix<NT>(cp + pslot(k))}; },
            [&](const E& e) { return x[e.c]; }, [](const E& e) { return e.v; });
    } else {
        return row_sum<Term<V, X>, row_u<V>()>(
            m, [&](int k) { return Term<V, X>{ld_matrix<NT>(vp + pslot(k)), x[ld_matrix<NT>(cp + pslot(k))]}; },
            [](double s, const Term<V, X>& t) { return s + (double)t.v * (double)t.x; });
    }
}
// The same over 16-bit columns: entry e = (group << EC_OFF_BITS) | offset,
// column = wb[group] + offset, wb = the slice's group bases (in LDS).
__device__ __forceinline__ int ecol(const int* wb, int e) { return wb[e >> EC_OFF_BITS] + (e & EC_OFF_MASK); }
template <class V, class X, bool NT>
__device__ __forceinline__ double offdiag_u16(const unsigned short* ep, const V* vp, int m, const int* wb,
                                              const X* x) {
    if constexpr (sizeof(V) == 8) {
        typedef Entry<V, unsigned short> E;
        return row_sum_cols<E, X, row_u<V>()>(
            m, [&](int k) { return E{ld_matrix<NT>(vp + pslot(k)), ld_matrix<NT>(ep + pslot(k))}; },
            [&](const E& e) { return x[ecol(wb, e.c)]; }, [](const E& e) { return e.v; });
    } else {
        return row_sum<Term<V, X>, row_u<V>()>(
            m, [&](int k) { return Term<V, X>{ld_matrix<NT>(vp + pslot(k)), x[ecol(wb, ld_matrix<NT>(ep + pslot(k)))]}; },
            [](double s, const Term<V, X>& t) { return s + (double)t.v * (double)t.x; });
    }
}

// The same over a stencil slice: column row + off[k], off the slice's
// ascending offsets, so a slot's x gathers are one contiguous run of the
// wave's rows; the stored zeros add exact zeros.  The offsets are the same
// for the whole wave and constant during the launch: read through the
// constant address space they become scalar loads.  Values and x through the
// global address space.
template <class T> using gmem = const __attribute__((address_space(1))) T*;
template <class T> using cmem = const __attribute__((address_space(4))) T*;
template <class V, class X, bool NT>
__device__ __forceinline__ double offdiag_stencil(const V* vals, int m, const int* offs, int r, const X* xv) {
    const gmem<V> vp = (gmem<V>)vals;
    const gmem<X> x = (gmem<X>)(xv + r);
    const cmem<int> off = (cmem<int>)offs;
    return row_sum<Term<V, X>, row_u<V>()>(
        m, [&](int k) { return Term<V, X>{ld_matrix<NT>(vp + pslot(k)), x[off[k]]}; },
        [](double s, const Term<V, X>& t) { return s + (double)t.v * (double)t.x; });
}
// Row r's slice: the first of its stencil offsets in pp.poff, or -1.  Every
// active lane of the calling wave holds a row of the same slice (rows are
// handed out in whole slices), so the value is read as wave-uniform.
__device__ __forceinline__ int stencil_of(const PPEView& pp, int r) {
    return pp.spat ? __builtin_amdgcn_readfirstlane(pp.spat[r >> 6]) : -1;
}

// Bitonic sort of a wave's Q * 64 keys held in registers, key t = lane +
// 64 q ascending: partners in other lanes through cross-lane moves, partners
// in the same lane (distance 64 and more) by register.
template <class K, int Q>
__device__ __forceinline__ void bitonic_wave(K (&v)[Q], int lane) {
    constexpr int W = Q * SLICE;
#pragma unroll
    for (int k = 2; k <= W; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j >= SLICE) {
                const int qj = j / SLICE;
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    if ((q & qj) == 0) {
                        const bool up = ((lane + q * SLICE) & k) == 0;
                        const K a = v[q], b = v[q | qj];
                        const bool sw = (a > b) == up;
                        v[q] = sw ? b : a;
                        v[q | qj] = sw ? a : b;
                    }
                }
            } else {
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const K o = __shfl_xor(v[q], j, SLICE);
                    const bool up = ((lane + q * SLICE) & k) == 0;
                    const bool take_min = ((lane & j) == 0) == up;
                    v[q] = take_min ? (o < v[q] ? o : v[q]) : (o > v[q] ? o : v[q]);
                }
            }
        }
    }
}
// Group bases of the block's slices into LDS (every thread of the block
// takes part; call before the row guard).
__device__ __forceinline__ void load_group_bases(const PPEView& pp, int first, int* wbase) {
    if (pp.ecols) wbase[threadIdx.x] = pp.gbase[first + (int)threadIdx.x];
    __syncthreads();
}

// y_r = diag_r x_r - offdiag_r(x); dg = the diagonal of this operator
template <bool NT, class V, class X>
__device__ __forceinline__ double offdiag_row(const PPEView& pp, int r, const V* vals, const X* x, const int* wbase) {
    const long long base = prow(pp.sl_off, r);
    const int st = stencil_of(pp, r);
    if (st >= 0) {
        // a stencil slice's rows all hold its offsets: a uniform count
        const int m = __builtin_amdgcn_readfirstlane(pp.cnt[r]);
        return offdiag_stencil<V, X, NT>(vals + base, m, pp.poff + st, r, x);
    }
    const int m = pp.cnt[r];
    if (pp.ecols) return offdiag_u16<V, X, NT>(pp.ecols + base, vals + base, m, wbase + (threadIdx.x & ~63), x);
    return offdiag_i32<V, X, NT>(pp.cols + base, vals + base, m, x);
}
template <class V, class X, class DG>
__device__ __forceinline__ double spmv_row(const PPEView& pp, int r, const V* vals, const DG* dg, const X* x,
                                           const int* wbase) {
    double s = (pp.stream & STREAM_KRYLOV) ? offdiag_row<true>(pp, r, vals, x, wbase)
                                           : offdiag_row<false>(pp, r, vals, x, wbase);
    if (pp.ltail) {
        const int u = pp.ltail[r];
        if (u >= 0) s += pp.lsum[u];
    }
    return (double)dg[r] * (double)x[r] - s;
}

}  // namespace sph
