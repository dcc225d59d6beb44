// herk_mxpipe.hip -- block-scaled (MX) HERK over operand fragments (layout: herk_mxpipe.h).
//
// Bound as herk_pipe.hip is, by the energy of the MFMAs and the operand traffic; same tile, stages,
// buffers and stores.  What differs is the Im product's operand V = [Im | -Re] of U = [Re | Im]:
// the two halves of a wave trade places with their scales.  The two blocks of a stage do it
// together, two v_permlane32_swap and one sign flip per dword pair:
//   (U0, U1) = ([R0|I0], [R1|I1])  ->  ([R0|R1], [I0|I1])  ->  ([I0|-R0], [I1|-R1]) = (V0, V1)
// which needs both blocks' row operands at once, so a stage runs Re first (column blocks y = 0,
// 1), then Im from V, and reads each next operand where the last use of its registers is past:
// the rows' after Re, a column block's after its Im.  Each output is summed block by block, Re
// and Im of a block in one MFMA, as the tile kernel sums it: the same bits.
#include "herk_mxpipe.h"
#include "herk_pipe.h"
#include "herk_pipe_dev.h"

namespace ftdx {

namespace {

constexpr int M_THREADS = 256;  // 4 waves, 2 x 2, of 64 x 64
constexpr int M_GROUPS = 2 * PT / 32;
constexpr int M_BUFS = 3;

template <int FMT>
struct Mx {
    static constexpr int FB = mxfrag_bytes(FMT), DW = FB / 256;  // bytes, dwords per lane of a block
    static constexpr int CODE = FMT == MX_FP4_E2M1 ? 4 : 3;      // cbsz / blgp
    static constexpr int SRC = 2 * FB + 128;                     // bytes of one group and stage
    static constexpr int PIECES = 2 * FB / 1024;                 // kilobytes of codes
    static constexpr int GSTRIDE = 2 * FB + 16;                  // as P_GSTRIDE of herk_pipe.hip
    static constexpr int SCALES = M_GROUPS * GSTRIDE;            // then 128 bytes per group
    static constexpr int STAGE = SCALES + M_GROUPS * 128;
    static constexpr int LOADS = M_GROUPS * PIECES / 4 + 1;      // copies per wave and stage
    static_assert(M_BUFS * STAGE * 2 <= 160 * 1024, "LDS of two workgroups per CU");
    // sign bits of dword d of an operand
    static __device__ __forceinline__ uint32_t neg(int d) {
        if (FMT == MX_FP4_E2M1) return 0x88888888u;
        return d % 3 == 0 ? 0x20820820u : d % 3 == 1 ? 0x08208208u : 0x82082082u;
    }
};

typedef int v4i __attribute__((ext_vector_type(4)));
typedef v6i Pair[2];  // one operand of a stage's two blocks

template <int FMT>
__device__ __forceinline__ void pin(Pair& f) {  // consecutive registers, here
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        if constexpr (FMT == MX_FP4_E2M1) {
            v4i t = __builtin_shufflevector(f[k], f[k], 0, 1, 2, 3);
            __asm__ __volatile__("" : "+v"(t));
            f[k] = __builtin_shufflevector(t, t, 0, 1, 2, 3, -1, -1);
        } else {
            __asm__ __volatile__("" : "+v"(f[k]));
        }
    }
}

template <int FMT>
__device__ __forceinline__ void read_pair(const uint8_t* __restrict__ g, int lane, Pair& f) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint4 u = *reinterpret_cast<const uint4*>(g + k * Mx<FMT>::FB + lane * 16);
        f[k][0] = (int)u.x;
        f[k][1] = (int)u.y;
        f[k][2] = (int)u.z;
        f[k][3] = (int)u.w;
        if constexpr (FMT != MX_FP4_E2M1) {
            const uint2 v = *reinterpret_cast<const uint2*>(g + k * Mx<FMT>::FB + 1024 + lane * 8);
            f[k][4] = (int)v.x;
            f[k][5] = (int)v.y;
        }
    }
}

[[maybe_unused]] __device__ __forceinline__ int read_scales(const uint8_t* __restrict__ sc, int group, int lane) {
    return *reinterpret_cast<const uint16_t*>(sc + group * 128 + lane * 2);
}

template <int FMT>
__device__ __forceinline__ void partner(const Pair& u, Pair& v) {
#pragma unroll
    for (int d = 0; d < Mx<FMT>::DW; ++d) {
        const auto w = __builtin_amdgcn_permlane32_swap((unsigned)u[0][d], (unsigned)u[1][d], false, false);
        const auto x = __builtin_amdgcn_permlane32_swap(w[1], w[0] ^ Mx<FMT>::neg(d), false, false);
        v[0][d] = (int)x[0];
        v[1][d] = (int)x[1];
    }
}

template <int FMT>
__device__ __forceinline__ void mfma_pair(const Pair& a, int sa, const Pair& b, int sb, v16f& c) {
    constexpr int F = Mx<FMT>::CODE;
    c = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(op8(a[0]), op8(b[0]), c, F, F, 0, sa, 0, sb);
    c = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(op8(a[1]), op8(b[1]), c, F, F, 1, sa, 1, sb);
}

// This wave's share of one stage: code kilobytes, and the scales of two groups.
template <int FMT>
__device__ __forceinline__ void copy_stage(__amdgpu_buffer_rsrc_t rows, int at, uint8_t* st, int wave,
                                           const uint32_t (&off)[Mx<FMT>::LOADS]) {
    using M = Mx<FMT>;
#pragma unroll
    for (int q = 0; q < M::LOADS - 1; ++q) {
        const int p = q * 4 + wave;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rows, (void __attribute__((address_space(3)))*)(st + (p / M::PIECES) * M::GSTRIDE + (p % M::PIECES) * 1024),
            16, off[q], at, 0, 0);
    }
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rows, (void __attribute__((address_space(3)))*)(st + M::SCALES + wave * 256), 4, off[M::LOADS - 1], at, 0, 0);
}

struct Ops {  // a wave's operands: two row groups, two column groups
    Pair a[2], b[2], v[2];
    int sa[2], sb[2], sv[2];
};

template <int FMT>
__device__ __forceinline__ void read_rows(const uint8_t* __restrict__ st, int ga, int lane, Ops& o) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        read_pair<FMT>(st + (ga + x) * Mx<FMT>::GSTRIDE, lane, o.a[x]);
        o.sa[x] = read_scales(st + Mx<FMT>::SCALES, ga + x, lane);
    }
}

template <int FMT>
__device__ __forceinline__ void read_col(const uint8_t* __restrict__ st, int gb, int y, int lane, Ops& o) {
    read_pair<FMT>(st + (gb + y) * Mx<FMT>::GSTRIDE, lane, o.b[y]);
    o.sb[y] = read_scales(st + Mx<FMT>::SCALES, gb + y, lane);
}

// Stage in `cur`: on entry its row operands and its first column block are read (or in flight).
template <int FMT>
__device__ __forceinline__ void stage_body(const uint8_t* __restrict__ cur, const uint8_t* __restrict__ nxt, int ga,
                                           int gb, int lane, Ops& o, v16f (&re)[2][2], v16f (&im)[2][2]) {
    read_col<FMT>(cur, gb, 1, lane, o);
#pragma unroll
    for (int x = 0; x < 2; ++x) o.sv[x] = read_scales(cur + Mx<FMT>::SCALES, ga + x, lane ^ 32);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < 2; ++x) pin<FMT>(o.a[x]);
    pin<FMT>(o.b[0]);
#pragma unroll
    for (int x = 0; x < 2; ++x) mfma_pair<FMT>(o.a[x], o.sa[x], o.b[0], o.sb[0], re[x][0]);
#pragma unroll
    for (int x = 0; x < 2; ++x) partner<FMT>(o.a[x], o.v[x]);
    __builtin_amdgcn_sched_barrier(0);
    pin<FMT>(o.b[1]);
#pragma unroll
    for (int x = 0; x < 2; ++x) mfma_pair<FMT>(o.a[x], o.sa[x], o.b[1], o.sb[1], re[x][1]);
    __builtin_amdgcn_sched_barrier(0);
    read_rows<FMT>(nxt, ga, lane, o);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < 2; ++x) pin<FMT>(o.v[x]);
#pragma unroll
    for (int x = 0; x < 2; ++x) mfma_pair<FMT>(o.v[x], o.sv[x], o.b[0], o.sb[0], im[x][0]);
    __builtin_amdgcn_sched_barrier(0);
    read_col<FMT>(nxt, gb, 0, lane, o);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int x = 0; x < 2; ++x) mfma_pair<FMT>(o.v[x], o.sv[x], o.b[1], o.sb[1], im[x][1]);
    __builtin_amdgcn_sched_barrier(0);
}

// Buffers and barriers as tile_loop of herk_pipe.hip: the barrier that opens stage s publishes
// stage s + 1, whose operands stage s reads at its end; the copies of stage s + 2 go where
// stage s - 1 was.
template <int FMT, bool ACTIVE>
__device__ __forceinline__ void tile_loop(__amdgpu_buffer_rsrc_t rows, uint8_t* lds, int nst,
                                          const uint32_t (&off)[Mx<FMT>::LOADS], int lane, int wave, int ga, int gb,
                                          v16f (&re)[2][2], v16f (&im)[2][2]) {
    using M = Mx<FMT>;
    copy_stage<FMT>(rows, 0, lds, wave, off);
    copy_stage<FMT>(rows, nst > 1 ? M::SRC : 0, lds + M::STAGE, wave, off);
    Ops o;
    wait_vm<M::LOADS>();  // stage 0 landed
    wg_barrier();
    if constexpr (ACTIVE) {
        read_rows<FMT>(lds, ga, lane, o);
        read_col<FMT>(lds, gb, 0, lane, o);
    }
    int c = 0;  // buffer of stage s
    for (int s = 0; s < nst; ++s) {
        wait_vm<0>();  // this wave's copies of stage s + 1
        wg_barrier();
        const int n = c == M_BUFS - 1 ? 0 : c + 1, f = c == 0 ? M_BUFS - 1 : c - 1;
        // past the end the last stage is copied again, into a buffer that is not read
        copy_stage<FMT>(rows, (s + 2 < nst ? s + 2 : nst - 1) * M::SRC, lds + f * M::STAGE, wave, off);
        if constexpr (ACTIVE) stage_body<FMT>(lds + c * M::STAGE, lds + n * M::STAGE, ga, gb, lane, o, re, im);
        c = n;
    }
    wait_vm<0>();  // no copy may land after the workgroup's LDS is given back
}

template <int FMT, typename OutT, bool NT>
__global__ void __launch_bounds__(M_THREADS, 2) herk_mxpipe_kernel(HerkPlainArgs p, int nst, int tiles) {
#if defined(__HIP_DEVICE_COMPILE__)  // clang's host pass deduces no template with a buffer descriptor
    using M = Mx<FMT>;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[M_BUFS * M::STAGE];
    const int w = xcd_logical((int)blockIdx.x, tiles * p.batch);
    const int b = w / tiles, t = w - b * tiles;
    int I, J;
    tri_decode_blocked(t, (p.N + PT - 1) / PT, P_BLOCK, I, J);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int wrow = I * PT + wm * 64, wcol = J * PT + wn * 64;
    const bool active = wrow < p.N && wrow + 63 >= wcol;
    // groups past N (edge tiles) read the last group; their products are not stored
    const int ng = (p.N + 31) / 32;
    uint32_t off[M::LOADS];
#pragma unroll
    for (int q = 0; q < M::LOADS; ++q) {
        const bool codes = q < M::LOADS - 1;
        const int k = q * 4 + wave, g = codes ? k / M::PIECES : wave * 2 + (lane >> 5);
        const int want = g < M_GROUPS / 2 ? I * (PT / 32) + g : J * (PT / 32) + g - M_GROUPS / 2;
        off[q] = (uint32_t)(want < ng ? want : ng - 1) * (uint32_t)(nst * M::SRC) +
                 (uint32_t)(codes ? (k % M::PIECES) * 1024 + lane * 16 : 2 * M::FB + (lane & 31) * 4);
    }
    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(p.A) + (int64_t)b * p.a_bstride, 0, (int)((uint32_t)ng * (uint32_t)(nst * M::SRC)), 0x00027000);
    v16f re[2][2], im[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                re[x][y][r] = 0.0f;
                im[x][y][r] = 0.0f;
            }
    const int ga = wm * 2, gb = M_GROUPS / 2 + wn * 2;
    if (!active) {
        tile_loop<FMT, false>(rows, lds, nst, off, lane, wave, ga, gb, re, im);
        return;
    }
    tile_loop<FMT, true>(rows, lds, nst, off, lane, wave, ga, gb, re, im);
    OutT* C = static_cast<OutT*>(p.C) + (int64_t)b * p.c_bstride;
    if (wcol + 63 < wrow && wrow + 64 <= p.N && p.beta == 0.0f)
        store_inside<OutT, true, NT>(C, wrow, wcol, p.alpha, re, im, lane);
    else
        store_any<OutT>(C, p.N, wrow, wcol, p.alpha, p.beta, re, im, lane);
#endif
}

template <int FMT, typename OutT>
void launch(const HerkPlainArgs& a, int nst, int tiles, bool nt, hipStream_t s) {
    const dim3 grid((unsigned)((int64_t)tiles * a.batch)), block(M_THREADS);
    if (nt)
        hipLaunchKernelGGL((herk_mxpipe_kernel<FMT, OutT, true>), grid, block, 0, s, a, nst, tiles);
    else
        hipLaunchKernelGGL((herk_mxpipe_kernel<FMT, OutT, false>), grid, block, 0, s, a, nst, tiles);
}

}  // namespace

hipError_t launch_herk_mxpipe(const HerkPlainArgs& a, int fmt, bool out_fp16, hipStream_t s) {
    if (a.N <= 0 || a.batch <= 0) return hipSuccess;
    const int tiles = pipe_tiles(a.N), nst = (a.K + 63) / 64;
    if ((int64_t)tiles * a.batch > 0x7FFFFFFF || !mxpipe_supported(a.N, a.K, fmt)) return hipErrorInvalidValue;
    const bool nt = pipe_nontemporal(a.N, a.K, out_fp16);
    if (fmt == MX_FP4_E2M1) {
        if (out_fp16) launch<MX_FP4_E2M1, _Float16>(a, nst, tiles, nt, s);
        else launch<MX_FP4_E2M1, float>(a, nst, tiles, nt, s);
    } else {
        if (out_fp16) launch<MX_FP6_E3M2, _Float16>(a, nst, tiles, nt, s);
        else launch<MX_FP6_E3M2, float>(a, nst, tiles, nt, s);
    }
    return hipGetLastError();
}

}  // namespace ftdx
