// herk_grid.h -- gridding epilogue (OUT_GRID) of the HERK kernels: the pillbox scatter of the
// reference (visibility_bf.cuh:259-370) on each element of an accumulator block instead of a store.
#pragma once
#include "herk_common.h"
#include "herk_fp8.h"

namespace ftdx {

struct GridJob {
    float* grid;      // this channel's plane [Ng][Ng][2]
    float* half;      // scratch of half_grid_cells(Ng) cells, zero before the launch, or nullptr
    const float* uv;  // baseline UV (metres), packed lower index
    double lambda;    // wavelength (metres)
    int Ng;
    float cell;       // radians
};

// A cross-correlation V at (u, v) also adds conj(V) at (-u, -v).  With cells numbered iv Ng + iu,
// that cell is Ng^2 + Ng - c wherever both are on the grid and rounding is symmetric.  Such a
// pair adds once, to the smaller of the two in a half plane, which launch_half_grid_add later
// adds to both: the same terms per cell, half the scattered atomics.
__host__ __device__ inline int64_t mirror_sum(int Ng) { return (int64_t)Ng * Ng + Ng; }
__host__ __device__ inline int64_t half_grid_cells(int Ng) { return mirror_sum(Ng) / 2 + 1; }

// Batch b of a launch.
__device__ __forceinline__ GridJob grid_job(const HerkPlainArgs& p, int b) {
    GridJob g;
    g.grid = static_cast<float*>(p.C) + (int64_t)b * p.c_bstride;
    g.half = p.half ? p.half + (int64_t)b * 2 * half_grid_cells(p.Ng) : nullptr;
    g.uv = p.uv_m;
    g.lambda = 299792458.0 / p.freq_hz[p.freq_offset + b];  // speed of light / frequency
    g.Ng = p.Ng;
    g.cell = p.cell;
    return g;
}

// uv / lambda rounded to float as the double division rounds it: from the reciprocal y of
// lambda, q = uv y and one correction by the exact remainder give the correctly rounded
// quotient (Markstein, Computation of elementary functions on the IBM RISC System/6000
// processor, 1990) where neither operand is zero's or infinity's neighbour; `plain` (the
// same for the whole launch) and an infinite uv take the division.
__device__ __forceinline__ float over_lambda(float uv, double lambda, double y, bool plain) {
    const double a = (double)uv;
    if (plain) return (float)(a / lambda);
    const double q = a * y;
    const double r = __builtin_fma(-q, lambda, a);
    const float f = (float)__builtin_fma(r, y, q);
    return __builtin_fabsf(uv) < __builtin_inff() ? f : uv;
}

// Cell of (iu, iv), -1 off the grid.
__device__ __forceinline__ int64_t grid_cell(int Ng, float x, float y) {
    const int iu = (int)__builtin_roundf(x), iv = (int)__builtin_roundf(y);
    return iu >= 0 && iu < Ng && iv >= 0 && iv < Ng ? (int64_t)iv * Ng + iu : -1;
}

typedef float uv_pair __attribute__((ext_vector_type(2), aligned(4)));

// LDS bytes of one wave below: 16 rows of 32 FN columns, [re, im].
template <int FN>
constexpr int grid_lds_bytes() { return 16 * (32 * FN * 8 + 16); }

// Elements (i, j <= i), i < N, of the block at (w, col), times alpha; Im = 0 on the diagonal.
// UV in wavelengths = float(uv_m / lambda) (double division).  Whole waves call it.  The block
// goes through LDS 16 rows at a time so that a loop over elements can serve them all: unrolled
// over the accumulators the cell arithmetic is 64 bodies, past the instruction cache, and the UV
// loads of few resident waves were waited for one by one.  Eight at a time against four: 128 x 4
// channels, K = 2 x 512, 68 against 73 us; 1024 x 8 308 against 304.
template <int FM, int FN>
__device__ __forceinline__ void grid_block(const GridJob& g, int N, int w, int col, float alpha,
                                           const v16f (&re)[FM][FN], const v16f (&im)[FM][FN], uint8_t* lds, int lane) {
    constexpr int COLS = 32 * FN, PITCH = COLS * 8 + 16, BATCH = 8;  // BATCH: UV loads in flight
    const float half_ng = 0.5f * g.Ng;
    const int64_t sum = mirror_sum(g.Ng);
    const double y = 1.0 / g.lambda;
    const bool plain = !(__builtin_fabs(g.lambda) > 1e-100 && __builtin_fabs(g.lambda) < 1e100);
    const int n = lane & 31, g4 = (lane >> 5) * 4;
    float* auto_at = nullptr;  // a lane meets at most one element of the diagonal
    float auto_re = 0.0f;
#pragma unroll
    for (int x = 0; x < FM; ++x)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int y = 0; y < FN; ++y)
#pragma unroll
                for (int q = 8 * h; q < 8 * h + 8; ++q)
                    *reinterpret_cast<float2*>(lds + ((q >> 2) * 8 + g4 + (q & 3) - 16 * h) * PITCH + (y * 32 + n) * 8) =
                        make_float2(re[x][y][q] * alpha, im[x][y][q] * alpha);
            __builtin_amdgcn_wave_barrier();
#pragma unroll 1
            for (int e0 = lane; e0 < 16 * COLS; e0 += 64 * BATCH) {
                uv_pair uv[BATCH];
#pragma unroll
                for (int b = 0; b < BATCH; ++b) {
                    const int e = e0 + 64 * b, i = w + x * 32 + h * 16 + e / COLS, j = col + e % COLS;
                    uv[b] = 0.0f;
                    if (i < N && j <= i) uv[b] = *reinterpret_cast<const uv_pair*>(g.uv + 2 * tri_index(i, j));
                }
#pragma unroll
                for (int b = 0; b < BATCH; ++b) {
                    const int e = e0 + 64 * b, i = w + x * 32 + h * 16 + e / COLS, j = col + e % COLS;
                    const float2 v = *reinterpret_cast<const float2*>(lds + (e / COLS) * PITCH + (e % COLS) * 8);
                    float vim = i == j ? 0.0f : v.y;
                    float *p = nullptr, *c = nullptr;
                    if (i < N && j <= i) {
                        const float u = over_lambda(uv[b][0], g.lambda, y, plain) / g.cell;
                        const float t = over_lambda(uv[b][1], g.lambda, y, plain) / g.cell;
                        const int64_t at = grid_cell(g.Ng, half_ng + u, half_ng + t);
                        const int64_t conj = i != j ? grid_cell(g.Ng, half_ng - u, half_ng - t) : -1;
                        if (g.half && at >= 0 && conj == sum - at) {
                            p = g.half + 2 * (at < conj ? at : conj);
                            if (conj < at) vim = -vim;
                        } else if (i == j) {
                            if (at >= 0) {
                                auto_at = g.grid + 2 * at;
                                auto_re = v.x;
                            }
                        } else {
                            if (at >= 0) p = g.grid + 2 * at;
                            if (conj >= 0) c = g.grid + 2 * conj;
                        }
                    }
                    grid_add(p, v.x, vim);
                    if (__ballot(c != nullptr)) grid_add(c, v.x, -vim);
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    // Autocorrelations mostly share the centre cell, one address for all their atomics and a
    // long sum: those of a wave are summed first where they do.
    const uint64_t autos = __ballot(auto_at != nullptr);
    if (autos == 0) return;
    const int src = __builtin_ctzll(autos);
    float* first = reinterpret_cast<float*>(__shfl(reinterpret_cast<uint64_t>(auto_at), src));
    if (__ballot(auto_at != nullptr && auto_at != first) == 0) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) auto_re += __shfl_xor(auto_re, d);
        if (lane != src) auto_at = nullptr;
    }
    grid_add(auto_at, auto_re, 0.0f);
}

}  // namespace ftdx
