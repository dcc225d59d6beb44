// herk_direct.hip -- HERK of QC voltages for problems too small to fill the chip with tiles.
//
// What bounds such a call is latency: a 128 x 128 tile of K = 1024 is one workgroup's chain of 16
// load / unpack / barrier / MFMA stages, and few CUs have one.  Here a workgroup computes one
// 32 x 32 tile with its waves splitting K, each wave reading its operands straight from the QC
// rows (16 bytes of a row are a lane's 16 samples of an MFMA step) with no LDS and no barrier;
// the waves' sums meet in LDS once.  The voltages are integers, so the order of the sums does
// not change them (below 2^24).  128 inputs x 16, K = 1024: 24.9 -> 5.7 us, kernel time.
#include "herk_direct.h"
#include "herk_elem.h"
#include "herk_tile.h"

namespace ftdx {

namespace {

constexpr int DT = 32;  // tile rows and columns

__device__ __forceinline__ v8i unpack16(uint4 g) {
    uint32_t d[8];
    qc4_to_fp8_planar(g.x, d[0], d[1]);
    qc4_to_fp8_planar(g.y, d[2], d[3]);
    qc4_to_fp8_planar(g.z, d[4], d[5]);
    qc4_to_fp8_planar(g.w, d[6], d[7]);
    v8i r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = (int)d[i];
    return r;
}

// Samples k .. k + 15 of a row; VEC: K % 16 == 0 and 16-byte aligned rows
template <bool VEC>
__device__ __forceinline__ uint4 load_samples(const uint8_t* row, int k, int K) {
    if constexpr (VEC) return k < K ? *reinterpret_cast<const uint4*>(row + k) : make_uint4(0u, 0u, 0u, 0u);
    else return row_segment(row, k, K);
}

// KS waves per workgroup; wave w takes its share of the 64-sample stages (lane half h: samples
// 32 h .. 32 h + 31 of a stage, the same for both operands).
template <int KS, typename OutT, bool VEC>
__global__ void __launch_bounds__(64 * KS)
herk_direct_kernel(HerkPlainArgs p, int tiles) {
    __shared__ __attribute__((aligned(16))) float sum[KS][8][256];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w = xcd_logical((int)blockIdx.x, (int)gridDim.x);
    const int b = w / tiles, t = w - b * tiles;
    int I, J;
    tri_decode(t, I, J);
    const uint8_t* A = p.A + (int64_t)b * p.a_bstride;
    const int r = lane & 31, h = lane >> 5;
    const int gi = I * DT + r < p.N ? I * DT + r : p.N - 1, gj = J * DT + r < p.N ? J * DT + r : p.N - 1;
    const uint8_t* ra = A + (int64_t)gi * p.K;
    const uint8_t* rb = A + (int64_t)gj * p.K;
    v16f re, im;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        re[q] = 0.0f;
        im[q] = 0.0f;
    }
    const int nst = (p.K + 63) / 64, per = (nst + KS - 1) / KS;
    const int s0 = wave * per, s1 = s0 + per < nst ? s0 + per : nst;
    uint4 ga[2], gb[2];
    auto load = [&](int s) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            ga[e] = load_samples<VEC>(ra, s * 64 + h * 32 + e * 16, p.K);
            gb[e] = load_samples<VEC>(rb, s * 64 + h * 32 + e * 16, p.K);
        }
    };
    if (s0 < s1) load(s0);
    for (int s = s0; s < s1; ++s) {
        v8i ua[2], ub[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            ua[e] = unpack16(ga[e]);
            ub[e] = unpack16(gb[e]);
        }
        if (s + 1 < s1) load(s + 1);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            re = mfma_32x32x64<OPF_FP8>(ua[e], ub[e], re);
            im = mfma_32x32x64<OPF_FP8>(conj_planar(ua[e]), ub[e], im);
        }
    }
    // four accumulator registers (rows 8 q + 4 (lane / 32) .. + 3 of column lane % 32) per group
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        v4f a, c;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            a[e] = re[q * 4 + e];
            c[e] = im[q * 4 + e];
        }
        *reinterpret_cast<v4f*>(&sum[wave][2 * q][lane * 4]) = a;
        *reinterpret_cast<v4f*>(&sum[wave][2 * q + 1][lane * 4]) = c;
    }
    __syncthreads();
    typedef typename Elem<OutT>::v2 v2;
    v2* C = reinterpret_cast<v2*>(static_cast<OutT*>(p.C) + (int64_t)b * p.c_bstride);
    // 16 rows per lane, spread over the waves
#pragma unroll
    for (int u = wave; u < 16; u += KS) {
        float sr = 0.0f, si = 0.0f;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            sr += sum[s][2 * (u >> 2)][lane * 4 + (u & 3)];
            si += sum[s][2 * (u >> 2) + 1][lane * 4 + (u & 3)];
        }
        const int i = I * DT + (u >> 2) * 8 + h * 4 + (u & 3), j = J * DT + r;
        if (i < p.N && j <= i) put_element<OutT>(C + tri_index(i, j), sr, i == j ? 0.0f : si, p.alpha, p.beta);
    }
}

template <int KS, typename OutT>
void launch_ks(const HerkPlainArgs& a, int tiles, hipStream_t stream) {
    const dim3 grid((unsigned)(tiles * a.batch)), block(64 * KS);
    if (a.K % 16 == 0 && (reinterpret_cast<uintptr_t>(a.A) & 15u) == 0)
        hipLaunchKernelGGL((herk_direct_kernel<KS, OutT, true>), grid, block, 0, stream, a, tiles);
    else
        hipLaunchKernelGGL((herk_direct_kernel<KS, OutT, false>), grid, block, 0, stream, a, tiles);
}

}  // namespace

int direct_tiles(int N) {
    const int nb = (N + DT - 1) / DT;
    return nb * (nb + 1) / 2;
}

bool direct_supported(int N, int K, int batch) {
    return N > 0 && K >= 16 && batch > 0 && N <= (1 << 18) && (int64_t)direct_tiles(N) * batch <= 0x7FFFFFFF;
}

hipError_t launch_herk_direct(const HerkPlainArgs& a, bool out_fp16, hipStream_t stream) {
    if (a.N <= 0 || a.batch <= 0) return hipSuccess;
    if (!direct_supported(a.N, a.K, a.batch) || a.nseg != 1) return hipErrorInvalidValue;
    const int tiles = direct_tiles(a.N);
    // 16 waves where K has a stage for each and the chip's wave slots (16 per CU at this
    // kernel's registers) hold them all; else 4
    const bool deep = a.K > 15 * 64 && (int64_t)tiles * a.batch <= 256;
    if (out_fp16) {
        if (deep) launch_ks<16, _Float16>(a, tiles, stream);
        else launch_ks<4, _Float16>(a, tiles, stream);
    } else {
        if (deep) launch_ks<16, float>(a, tiles, stream);
        else launch_ks<4, float>(a, tiles, stream);
    }
    return hipGetLastError();
}

}  // namespace ftdx
