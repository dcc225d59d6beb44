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

// LDS bytes of one wave below: 16 rows of 64 columns, [re, im].
constexpr int kGridRegion = 16 * (64 * 8 + 16);

// Elements (i, j <= i), i < N, of the tile at (row0, col0), times alpha; Im = 0 on the diagonal.
// UV in wavelengths = float(uv_m / lambda) (double division).  Every wave of the workgroup calls it,
// W of them in rows of WN, each with the 64 x 64 block of its place (active: it has elements).  The
// blocks go through LDS 16 rows at a time so that a loop over rows can serve them all: unrolled
// over the accumulators the cell arithmetic is 64 bodies, past the instruction cache, and the UV
// loads of few resident waves were waited for one by one.  Eight at a time against four: 128 x 4
// channels, K = 2 x 512, 68 against 73 us; 1024 x 8 308 against 304.
// What bounds launches of few tiles is one wave's instructions, about 250 a row.  Where every wave has
// 64 rows each takes its own; on the diagonal and at the matrix's edge, where some have few or none,
// the workgroup shares the rows that exist, and rows without an element are skipped (us, each wave its
// own 64 / shared: 48 x 1 channel, K = 64 40 / 17; 64 x 16, K = 2 x 512 58 / 30; 128 x 16 61 / 54;
// 256 x 8 73 / 74; 1024 x 8 307 / 300).
template <int W, int WN, int FM, int FN>
__device__ __forceinline__ void grid_tile(const GridJob& g, int N, int row0, int col0, bool active, float alpha,
                                          const v16f (&re)[FM][FN], const v16f (&im)[FM][FN], uint8_t* lds, int wave,
                                          int lane) {
    static_assert(FM == 2 && FN == 2 && 16 % W == 0, "blocks of 64 x 64, whole rows per wave");
    constexpr int PITCH = 64 * 8 + 16, BATCH = 8;  // BATCH: UV loads in flight
    const bool shared = col0 + WN * 64 > row0 || row0 + W / WN * 64 > N;
    const float half_ng = 0.5f * g.Ng;
    const int64_t sum = mirror_sum(g.Ng);
    const double y = 1.0 / g.lambda;
    const bool plain = !(__builtin_fabs(g.lambda) > 1e-100 && __builtin_fabs(g.lambda) < 1e100);
    const int n = lane & 31, g4 = (lane >> 5) * 4;
    uint8_t* mine = lds + wave * kGridRegion;
    // A wave's 16 rows go in groups of R.  Shared: a group or two of every block, of another part of
    // each, so that a lane still meets at most one element of the diagonal.
    constexpr int PART = 16 / W, R = PART < BATCH ? PART : BATCH;
    auto place = [&](int q, int& i, int& j, int& at) {  // group q: first row of its rows, first column, LDS
        const int r = shared ? q / (PART / R) : wave;
        const int row = shared ? ((wave + r) & (W - 1)) * PART + q % (PART / R) * R : q * R;
        i = r / WN * 64 + row;
        j = col0 + r % WN * 64;
        at = r * kGridRegion + row * PITCH;
    };
    auto wait = [&] {
        if (shared) __syncthreads();
        else __builtin_amdgcn_wave_barrier();
    };
    float* auto_at = nullptr;  // a lane meets at most one element of the diagonal
    float auto_re = 0.0f;
#pragma unroll
    for (int x = 0; x < FM; ++x)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int first = x * 32 + h * 16;  // of each block's rows
            if (row0 + first >= N) continue;    // the same for the workgroup
            if (active) {
#pragma unroll
                for (int y = 0; y < FN; ++y)
#pragma unroll
                    for (int q = 8 * h; q < 8 * h + 8; ++q)
                        *reinterpret_cast<float2*>(mine + ((q >> 2) * 8 + g4 + (q & 3) - 16 * h) * PITCH + (y * 32 + n) * 8) =
                            make_float2(re[x][y][q] * alpha, im[x][y][q] * alpha);
            }
            wait();
#pragma unroll 1
            for (int k0 = 0; k0 < 16; k0 += BATCH) {
                int i0[BATCH / R], j0[BATCH / R], at0[BATCH / R];
                uv_pair uv[BATCH];
#pragma unroll
                for (int q = 0; q < BATCH / R; ++q) {
                    place(k0 / R + q, i0[q], j0[q], at0[q]);
                    i0[q] += row0 + first;
                }
#pragma unroll
                for (int b = 0; b < BATCH; ++b) {
                    const int i = i0[b / R] + b % R, j = j0[b / R] + lane;
                    uv[b] = 0.0f;
                    if (i < N && j <= i) uv[b] = *reinterpret_cast<const uv_pair*>(g.uv + 2 * tri_index(i, j));
                }
#pragma unroll
                for (int b = 0; b < BATCH; ++b) {
                    const int i = i0[b / R] + b % R, j = j0[b / R] + lane;
                    if (i >= N || j0[b / R] > i) continue;  // no element in this row
                    const float2 v = *reinterpret_cast<const float2*>(lds + at0[b / R] + b % R * PITCH + lane * 8);
                    float vim = i == j ? 0.0f : v.y;
                    float *p = nullptr, *c = nullptr;
                    if (j <= i) {
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
            wait();
        }
    if (!shared) return;  // no diagonal in it
    // Autocorrelations mostly share the centre cell, one address for all their atomics and a
    // long sum: those of the tile are summed first where they do.
    const uint64_t autos = __ballot(auto_at != nullptr);
    const int src = autos ? __builtin_ctzll(autos) : 0;
    float* at = reinterpret_cast<float*>(__shfl(reinterpret_cast<uint64_t>(auto_at), src));  // nullptr: none
    const bool one = __ballot(auto_at != nullptr && auto_at != at) == 0;
    if (one) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) auto_re += __shfl_xor(auto_re, d);
        if (lane != src) auto_at = nullptr;
    }
    struct Sum {
        float* at;
        float re;
        int one;
    }* sums = reinterpret_cast<Sum*>(lds);
    if (lane == 0) sums[wave] = {at, auto_re, one};
    __syncthreads();
    bool same = true;
    at = nullptr;
    float total = 0.0f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
        const Sum t = sums[w];
        if (!at) at = t.at;
        same = same && t.one && (!t.at || t.at == at);
        total += t.re;
    }
    if (same) {
        auto_at = wave == 0 && lane == 0 ? at : nullptr;
        auto_re = total;
    }
    grid_add(auto_at, auto_re, 0.0f);
}

}  // namespace ftdx
