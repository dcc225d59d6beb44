// herk_elem.h -- output elements and QC row loads shared by the pipelined and the direct HERK.
#pragma once
#include "herk_common.h"

namespace ftdx {

template <typename OutT>
struct Elem;  // one complex output element
template <>
struct Elem<float> {
    typedef float v2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ v2 make(float r, float i) {
        v2 v;
        v[0] = r;
        v[1] = i;
        return v;
    }
};
template <>
struct Elem<_Float16> {
    typedef _Float16 v2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ v2 make(float r, float i) {
        v2 v;
        v[0] = (_Float16)r;
        v[1] = (_Float16)i;
        return v;
    }
};
template <>
struct Elem<double> {
    typedef double v2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ v2 make(float r, float i) {
        v2 v;
        v[0] = r;
        v[1] = i;
        return v;
    }
};

// C = alpha * (r, i) + beta * C for one element: alpha first, then fma(beta, old, .), one
// rounding each, as the other HERK kernels.
template <typename OutT>
__device__ __forceinline__ void put_element(typename Elem<OutT>::v2* c, float r, float i, float alpha, float beta) {
    r *= alpha;
    i *= alpha;
    if (beta != 0.0f) {
        const typename Elem<OutT>::v2 old = *c;
        r = __builtin_fmaf(beta, (float)old[0], r);
        i = __builtin_fmaf(beta, (float)old[1], i);
    }
    *c = Elem<OutT>::make(r, i);
}

// A block wholly below the diagonal and inside the matrix, beta = 0: no element is tested, and a
// row's offset is the last row's plus a lane constant (row d of a block starting at row w lies
// d w + d (d + 1) / 2 elements after row 0).  The general form below spends about 15 VALU
// operations per element, 5 of them on 64-bit index arithmetic (K = 128, FP16 output: 214
// against 269 us for the whole launch).
template <typename OutT, bool SCALE, bool NT, int FM, int FN>
__device__ __forceinline__ void store_inside(OutT* C, int w, int col, float alpha, const v16f (&re)[FM][FN],
                                             const v16f (&im)[FM][FN], int lane) {
    typedef typename Elem<OutT>::v2 v2;
    constexpr uint32_t ES = sizeof(v2);
    const int n = lane & 31, g4 = (lane >> 5) * 4;
    uint8_t* base = reinterpret_cast<uint8_t*>(reinterpret_cast<v2*>(C) + tri_index(w, col));
    uint32_t off = (uint32_t)(g4 * w + g4 * (g4 + 1) / 2 + n) * ES;
    const uint32_t step = (uint32_t)(w + g4) * ES;  // row d + g4 -> d + 1 + g4 adds step + (d + 1) ES
    // Where a kernel holds both forms the compiler would otherwise merge them into one of plain
    // stores, or compute the offsets and elements of both ahead of the choice and spill them.
    if constexpr (NT) __asm__ __volatile__("; non-temporal stores" : "+v"(off), "+v"(alpha));
    else __asm__ __volatile__("; plain stores" : "+v"(off), "+v"(alpha));
#pragma unroll
    for (int x = 0; x < FM; ++x)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int d = x * 32 + (q >> 2) * 8 + (q & 3);
            v2* p = reinterpret_cast<v2*>(base + off);
#pragma unroll
            for (int y = 0; y < FN; ++y) {
                const v2 e = SCALE ? Elem<OutT>::make(re[x][y][q] * alpha, im[x][y][q] * alpha)
                                  : Elem<OutT>::make(re[x][y][q], im[x][y][q]);
                if constexpr (NT) __builtin_nontemporal_store(e, p + y * 32);
                else p[y * 32] = e;
            }
            off += (q & 3) != 3 ? step + (uint32_t)(d + 1) * ES : 5 * step + (uint32_t)(5 * d + 15) * ES;
        }
    if constexpr (NT) __asm__ __volatile__("; stored");
}

typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(1)));

// Samples k .. k + 15 of a row of K >= 16 samples at any address; zeros past K.  A segment that
// crosses the row's end is taken from its last 16 bytes and shifted down, so nothing past the
// row is read.
__device__ __forceinline__ uint4 row_segment(const uint8_t* row, int k, int K) {
    const int over = k + 16 - K;
    if (over >= 16) return make_uint4(0u, 0u, 0u, 0u);
    const u32x4_any v = *reinterpret_cast<const u32x4_any*>(row + (over > 0 ? K - 16 : k));
    uint64_t lo = ((uint64_t)v[1] << 32) | v[0], hi = ((uint64_t)v[3] << 32) | v[2];
    if (over > 0) {
        const int s = over * 8;
        if (s >= 64) {
            lo = hi >> (s - 64);
            hi = 0;
        } else {
            lo = (lo >> s) | (hi << (64 - s));
            hi >>= s;
        }
    }
    return make_uint4((uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32));
}

}  // namespace ftdx
