// herk_pipe_dev.h -- device code shared by the pipelined HERK kernels (herk_pipe.hip, herk_mxpipe.hip).
#pragma once
#include "herk_common.h"
#include "herk_elem.h"

namespace ftdx {

constexpr int PT = 128;                      // tile rows and columns
constexpr int P_BLOCK = 4;                   // tile order: blocks of 4 x 4 tiles

typedef int v6i __attribute__((ext_vector_type(6)));

__device__ __forceinline__ v8i op8(v6i a) { return __builtin_shufflevector(a, a, 0, 1, 2, 3, 4, 5, -1, -1); }

template <int VM>
__device__ __forceinline__ void wait_vm() {  // vmcnt(VM), other counters free
    __builtin_amdgcn_s_waitcnt((VM & 0xF) | (0x7 << 4) | (0xF << 8) | (((VM >> 4) & 0x3) << 14));
}

__device__ __forceinline__ void wg_barrier() {
    __asm__ __volatile__("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ __volatile__("" ::: "memory");
}

// Tile t of the lower triangle of nb x nb tiles, in square blocks of H x H tiles (row-major
// inside a block, blocks row-major): the tiles that one XCD runs together then share H row and
// H column blocks in its L2 instead of one and many.
__device__ __forceinline__ void tri_decode_blocked(int t, int nb, int H, int& I, int& J) {
    const int full = H * H, diag = H * (H + 1) / 2;
    // block row S starts at full S (S - 1) / 2 + diag S
    const float a = 0.5f * full, b = diag - a;
    int S = (int)((__builtin_sqrtf(b * b + 4.0f * a * (float)t) - b) / (2.0f * a));
    while (S > 0 && full * S * (S - 1) / 2 + diag * S > t) --S;
    while (full * (S + 1) * S / 2 + diag * (S + 1) <= t) ++S;
    int u = t - (full * S * (S - 1) / 2 + diag * S);
    const int h = nb - S * H < H ? nb - S * H : H;  // rows of this block row
    if (u < h * H * S) {
        const int SJ = u / (h * H), v = u - SJ * (h * H);
        I = S * H + v / H;
        J = SJ * H + v % H;
    } else {
        int i;
        tri_decode(u - h * H * S, i, u);
        I = S * H + i;
        J = S * H + u;
    }
}

// Paired rows (herk_pipe.h): element (x, y, register q) of a wave's block at
// (w, col) is row w + 2 (8 (q / 4) + 4 (lane / 32) + q % 4) + x, column col + 2 (lane % 32) + y, so a
// lane stores the two column groups' elements at once and a half wave a run of 64.
template <typename OutT>
struct Elem2 {  // two neighbouring elements
    typedef OutT v4 __attribute__((ext_vector_type(4), aligned(2 * sizeof(OutT))));
    static __device__ __forceinline__ v4 make(float r0, float i0, float r1, float i1) {
        v4 v;
        v[0] = (OutT)r0;
        v[1] = (OutT)i0;
        v[2] = (OutT)r1;
        v[3] = (OutT)i1;
        return v;
    }
};

// A block wholly below the diagonal and inside the matrix, beta = 0: as store_inside of
// herk_elem.h.  Half the store instructions pay where they are non-temporal (us, 32-row groups /
// paired: 4096 x 96, K = 2048 4145 / 4060; 2048 x 16, K = 512, FP16 73.7 / 71.4; 1024 x 40, K = 384,
// FP16 52.6 / 51.2), not where plain ones meet in the L2 (1664 x 128, K = 128, FP16 213 / 216).
template <typename OutT, bool SCALE, bool NT>
__device__ __forceinline__ void store_pairs(OutT* C, int w, int col, float alpha, const v16f (&re)[2][2],
                                            const v16f (&im)[2][2], int lane) {
    constexpr uint32_t ES = 2 * sizeof(OutT);
    const int n = lane & 31, g8 = (lane >> 5) * 8;
    uint8_t* base = reinterpret_cast<uint8_t*>(C) + tri_index(w, col) * ES;
    uint32_t off = (uint32_t)(g8 * w + g8 * (g8 + 1) / 2 + 2 * n) * ES;
    const uint32_t step = (uint32_t)(w + g8) * ES;  // row d + g8 -> d + 1 + g8 adds step + (d + 1) ES
#pragma unroll
    for (int q = 0; q < 16; ++q)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int d = 2 * ((q >> 2) * 8 + (q & 3)) + x;
            const float a = SCALE ? alpha : 1.0f;
            const auto e = Elem2<OutT>::make(re[x][0][q] * a, im[x][0][q] * a, re[x][1][q] * a, im[x][1][q] * a);
            auto* p = reinterpret_cast<typename Elem2<OutT>::v4*>(base + off);
            if constexpr (NT) __builtin_nontemporal_store(e, p);
            else *p = e;
            off += (q & 3) != 3 || x == 0 ? step + (uint32_t)(d + 1) * ES : 9 * step + (uint32_t)(9 * d + 45) * ES;
        }
}

// Any block: elements (i, j <= i) with i < N; Im = 0 on the diagonal, then alpha, then
// fma(beta, old, .), as the other HERK kernels.
template <typename OutT, bool PAIRED = false>
__device__ __forceinline__ void store_any(OutT* C, int N, int w, int col, float alpha, float beta,
                                          const v16f (&re)[2][2], const v16f (&im)[2][2], int lane) {
    typedef typename Elem<OutT>::v2 v2;
    const int n = lane & 31, g4 = (lane >> 5) * 4;
    v2* base = reinterpret_cast<v2*>(C);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int r = (q >> 2) * 8 + g4 + (q & 3), i = w + (PAIRED ? 2 * r + x : x * 32 + r);
            v2* row = base + tri_index(i, 0);
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                const int j = col + (PAIRED ? 2 * n + y : y * 32 + n);
                if (i < N && j <= i)
                    put_element<OutT>(row + j, re[x][y][q], i == j ? 0.0f : im[x][y][q], alpha, beta);
            }
        }
}

}  // namespace ftdx
