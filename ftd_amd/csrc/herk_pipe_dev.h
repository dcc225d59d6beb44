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

// Any block: elements (i, j <= i) with i < N; Im = 0 on the diagonal, then alpha, then
// fma(beta, old, .), as the other HERK kernels.
template <typename OutT>
__device__ __forceinline__ void store_any(OutT* C, int N, int w, int col, float alpha, float beta,
                                          const v16f (&re)[2][2], const v16f (&im)[2][2], int lane) {
    typedef typename Elem<OutT>::v2 v2;
    const int n = lane & 31, g4 = (lane >> 5) * 4;
    v2* base = reinterpret_cast<v2*>(C);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int i = w + x * 32 + (q >> 2) * 8 + g4 + (q & 3);
            v2* row = base + tri_index(i, 0);
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                const int j = col + y * 32 + n;
                if (i < N && j <= i)
                    put_element<OutT>(row + j, re[x][y][q], i == j ? 0.0f : im[x][y][q], alpha, beta);
            }
        }
}

}  // namespace ftdx
