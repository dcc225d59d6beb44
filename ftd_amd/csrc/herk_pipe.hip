// herk_pipe.hip -- HERK of QC voltages on E3M2 MFMA over fragment rows (layout: herk_pipe.h).
//
// What bounds it: at 4096 x 96, K = 2048 the matrix cores are busy about 60% of the cycles, and
// under that load the chip runs at 1.5 - 1.9 instead of 2.4 GHz: the time is the energy of the
// MFMAs, then of the operand traffic.  So the operands are the smallest exact ones (6 bits,
// half the MFMA time of FP8 and 0.75 of its bytes), tiles go in square blocks that one XCD's L2
// serves, and the loop keeps both pipes fed:
//   * 128 x 128 tile, 4 waves of 64 x 64, two workgroups per CU, so that one workgroup's
//     stores overlap the other's MFMAs (256 x 128 with one per CU: 4.39 against 4.25 ms);
//   * stages of 64 samples in three LDS buffers, copied by buffer_load ... lds.  (The
//     global_load form is a FLAT instruction to the compiler, which then waits for every
//     outstanding LDS and memory operation at the next use of either.)
//   * operands one 32-sample step ahead in a second register set, across the barrier too: a
//     stage's first step is read during the previous stage, whose barrier already published
//     it, so no MFMA waits for an LDS read that was not issued a step earlier.
// Stores go to the packed rows straight from the accumulators.  With few samples they are runs of 32
// lanes, plain, so that the L2 joins the partial lines of neighbouring runs (1664 inputs x 128, K = 128,
// FP32: 303 against 478 us non-temporal; written bytes within 2% of the output's); with more, runs of 64
// elements from paired rows, non-temporal (pipe_nontemporal below has both sides).
#include "herk_common.h"
#include "herk_elem.h"
#include "herk_grid.h"
#include "herk_pipe.h"
#include "herk_pipe_dev.h"

namespace ftdx {

namespace {

constexpr int P_THREADS = 256;               // 4 waves, 2 x 2
constexpr int P_GROUPS = 2 * PT / 32;        // row groups of a stage: 4 of the rows, 4 of the columns
constexpr int P_GSTRIDE = 2 * kFragBytes + 16;  // LDS bytes per group and stage; not a multiple of
                                             // 512, or the compiler pairs the 8-byte reads of two
                                             // groups and copies the halves into place
constexpr int P_STAGE = P_GROUPS * P_GSTRIDE;
constexpr int P_BUFS = 3;
constexpr int P_LOADS = P_GROUPS * 3 / 4;    // kilobyte copies per wave and stage
constexpr int P_WG_PER_CU = 2;
static_assert(P_BUFS * P_STAGE * P_WG_PER_CU <= 160 * 1024, "LDS of the resident workgroups");

typedef v6i Frags[2];

// v = [im | -re] of u = [re | im]: the halves swapped, bit 5 of every Re code flipped
__device__ __forceinline__ v6i conj6(v6i a) {
    v6i r;
    r[0] = a[3];
    r[1] = a[4];
    r[2] = a[5];
    r[3] = a[0] ^ (int)0x20820820u;
    r[4] = a[1] ^ (int)0x08208208u;
    r[5] = a[2] ^ (int)0x82082082u;
    return r;
}

template <int L>
__device__ __forceinline__ void wait_lgkm() {  // lgkmcnt(L), other counters free
    __builtin_amdgcn_s_waitcnt(0xF | (0x7 << 4) | (L << 8) | (3 << 14));
}

// The operands of step ks (0, 1) of a stage: two groups at `a`, two at `b`.
__device__ __forceinline__ void read_frags(const uint8_t* __restrict__ st, int a, int b, int lane, int ks, Frags& fa,
                                           Frags& fb) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            const int off = (m ? b : a) + x * P_GSTRIDE + ks * kFragBytes;
            const uint4 u = *reinterpret_cast<const uint4*>(st + off + lane * 16);
            const uint2 v = *reinterpret_cast<const uint2*>(st + off + 1024 + lane * 8);
            v6i& f = m ? fb[x] : fa[x];
            f[0] = (int)u.x;
            f[1] = (int)u.y;
            f[2] = (int)u.z;
            f[3] = (int)u.w;
            f[4] = (int)v.x;
            f[5] = (int)v.y;
        }
}

// One step: 8 MFMAs; TRANS: the accumulators hold the transposed block, same values.  The empty
// asm keeps each operand in six consecutive registers here.
template <bool TRANS>
__device__ __forceinline__ void mfma_step(Frags& fa, Frags& fb, v16f (&re)[2][2], v16f (&im)[2][2]) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        __asm__ __volatile__("" : "+v"(fa[x]));
        __asm__ __volatile__("" : "+v"(fb[x]));
    }
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const v6i v = conj6(fa[x]);
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            re[x][y] = TRANS ? mfma_32x32x64<OPF_BF6>(op8(fb[y]), op8(fa[x]), re[x][y])
                             : mfma_32x32x64<OPF_BF6>(op8(fa[x]), op8(fb[y]), re[x][y]);
            im[x][y] = TRANS ? mfma_32x32x64<OPF_BF6>(op8(fb[y]), op8(v), im[x][y])
                             : mfma_32x32x64<OPF_BF6>(op8(v), op8(fb[y]), im[x][y]);
        }
    }
}

// This wave's share of one stage: kilobyte q * 4 + wave of the stage's 24, three per group.
__device__ __forceinline__ void copy_stage(__amdgpu_buffer_rsrc_t rows, int at, uint8_t* st, int wave,
                                           const uint32_t (&off)[P_LOADS]) {
#pragma unroll
    for (int q = 0; q < P_LOADS; ++q) {
        const int p = q * 4 + wave;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rows, (void __attribute__((address_space(3)))*)(st + (p / 3) * P_GSTRIDE + (p % 3) * 1024), 16, off[q], at,
            0, 0);
    }
}

// Stage s in `cur`: its second step's operands are read while the first step (f0, read a stage
// ago) multiplies, the next stage's first step while the second one does.  The copies of
// stage s + 2 go into `fre`, the buffer of stage s - 1, which every wave finished reading
// before this stage's barrier.
template <bool ACTIVE, bool TRANS>
__device__ __forceinline__ void stage_body(const uint8_t* __restrict__ cur, const uint8_t* __restrict__ nxt,
                                           uint8_t* __restrict__ fre, __amdgpu_buffer_rsrc_t rows, int at,
                                           const uint32_t (&off)[P_LOADS], int lane, int wave, int a, int b, Frags& a0,
                                           Frags& b0, Frags& a1, Frags& b1, v16f (&re)[2][2], v16f (&im)[2][2]) {
    copy_stage(rows, at, fre, wave, off);
    if constexpr (ACTIVE) {
        read_frags(cur, a, b, lane, 1, a1, b1);
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkm<8>();  // all but the eight reads just issued
        mfma_step<TRANS>(a0, b0, re, im);
        __builtin_amdgcn_sched_barrier(0);
        read_frags(nxt, a, b, lane, 0, a0, b0);
        __builtin_amdgcn_sched_barrier(0);
        wait_lgkm<8>();
        mfma_step<TRANS>(a1, b1, re, im);
        __builtin_amdgcn_sched_barrier(0);
    }
}

template <bool ACTIVE, bool TRANS>
__device__ __forceinline__ void tile_loop(__amdgpu_buffer_rsrc_t rows, uint8_t* lds, int nst,
                                          const uint32_t (&off)[P_LOADS], int lane, int wave, int a, int b,
                                          v16f (&re)[2][2], v16f (&im)[2][2]) {
    constexpr int SRC = 2 * kFragBytes;  // bytes of one group and stage
    copy_stage(rows, 0, lds, wave, off);
    copy_stage(rows, nst > 1 ? SRC : 0, lds + P_STAGE, wave, off);
    Frags a0, b0, a1, b1;
    wait_vm<P_LOADS>();  // stage 0 landed
    wg_barrier();
    if constexpr (ACTIVE) read_frags(lds, a, b, lane, 0, a0, b0);
    int c = 0;  // buffer of stage s
    for (int s = 0; s < nst; ++s) {
        wait_vm<0>();  // this wave's copies of stage s + 1
        wg_barrier();
        const int n = c == P_BUFS - 1 ? 0 : c + 1, f = c == 0 ? P_BUFS - 1 : c - 1;
        // past the end the last stage is copied again, into a buffer that is not read
        const int t = s + 2 < nst ? s + 2 : nst - 1;
        stage_body<ACTIVE, TRANS>(lds + c * P_STAGE, lds + n * P_STAGE, lds + f * P_STAGE, rows, t * SRC, off, lane,
                                  wave, a, b, a0, b0, a1, b1, re, im);
        c = n;
    }
    wait_vm<0>();  // no copy may land after the workgroup's LDS is given back
}

// ---- GGP layouts (herk_tile.h), from the transposed accumulators: lane = row i ----
// Block x, y, register q: i = w + 32 x + lane % 32, j = col + 32 y + 8 (q / 4) + 4 (lane / 32) + q % 4.
// Upper packed rows (j, i >= j) are 32-lane runs, so is the upper half of the full matrix; its
// lower half takes the four consecutive j of a lane at a time, which the L2 joins to lines.
template <typename OutT, int FMT>
__device__ __forceinline__ void store_ggp_inside(OutT* C, int N, int w, int col, const v16f (&re)[2][2],
                                                 const v16f (&im)[2][2], int lane) {
    typedef typename Elem<OutT>::v2 v2;
    constexpr uint32_t ES = sizeof(v2);
    constexpr bool TRI = FMT == OUT_UPPER_PACKED;
    const int n = lane & 31, g4 = (lane >> 5) * 4;
    const int64_t row = (int64_t)col * N - (TRI ? (int64_t)col * (col + 1) / 2 : 0);
    uint8_t* base = reinterpret_cast<uint8_t*>(reinterpret_cast<v2*>(C) + row + w);
    // row col + d starts d (N - col) - d (d + 1) / 2 elements on (TRI), d N (full)
    const uint32_t pitch = (uint32_t)(N - (TRI ? col + g4 : 0)) * ES;  // row d + g4 -> d + 1 + g4: less (d + 1) ES
    uint32_t off = (uint32_t)(TRI ? g4 * (N - col) - g4 * (g4 + 1) / 2 + n : g4 * N + n) * ES;
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int d = y * 32 + (q >> 2) * 8 + (q & 3);
            v2* p = reinterpret_cast<v2*>(base + off);
#pragma unroll
            for (int x = 0; x < 2; ++x) p[x * 32] = Elem<OutT>::make(re[x][y][q], im[x][y][q]);
            const bool next = (q & 3) != 3;
            off += (next ? 1u : 5u) * pitch - (TRI ? (uint32_t)(next ? d + 1 : 5 * d + 15) * ES : 0u);
        }
    if constexpr (FMT == OUT_HERM_FULL) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            v2* p = reinterpret_cast<v2*>(C) + (int64_t)(w + x * 32 + n) * N + col + g4;
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    float r = re[x][y][q], m = -im[x][y][q];
                    // converted anew: kept from the first loop, FP64 values would spill
                    if constexpr (sizeof(OutT) == 8) __asm__ __volatile__("" : "+v"(r), "+v"(m));
                    p[y * 32 + (q >> 2) * 8 + (q & 3)] = Elem<OutT>::make(r, m);
                }
        }
    }
}

template <typename OutT, int FMT>
__device__ __forceinline__ void store_ggp_any(OutT* C, int N, int w, int col, const v16f (&re)[2][2],
                                              const v16f (&im)[2][2], int lane) {
    typedef typename Elem<OutT>::v2 v2;
    const int n = lane & 31, g4 = (lane >> 5) * 4;
    v2* base = reinterpret_cast<v2*>(C);
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int j = col + y * 32 + (q >> 2) * 8 + g4 + (q & 3);
            v2* row = base + ((int64_t)j * N - (FMT == OUT_UPPER_PACKED ? (int64_t)j * (j + 1) / 2 : 0));
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const int i = w + x * 32 + n;
                if (i >= N || j > i) continue;
                const float r = re[x][y][q], m = i == j ? 0.0f : im[x][y][q];
                row[i] = Elem<OutT>::make(r, m);
                if (FMT == OUT_HERM_FULL && i != j) base[(int64_t)i * N + j] = Elem<OutT>::make(r, -m);
            }
        }
}

// Tile (I, J) of one problem: `base` its fragment rows, `steps` per row.  GGP layouts: alpha 1,
// beta 0; OUT_GRID: `grid` in place of C.
template <typename OutT, int FMT = OUT_LOWER_PACKED>
__device__ __forceinline__ void pipe_tile(uint8_t* lds, const uint8_t* base, int N, int steps, int I, int J, OutT* C,
                                          float alpha, float beta, bool nt, const GridJob* grid = nullptr) {
    // wave index in an SGPR: the conditions on it are scalar branches
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int wrow = I * PT + wm * 64, wcol = J * PT + wn * 64;
    const bool active = wrow < N && wrow + 63 >= wcol;
    // groups past N (edge tiles) read the last group; their products are not stored
    const int ng = frag_groups(N);
    uint32_t off[P_LOADS];
#pragma unroll
    for (int q = 0; q < P_LOADS; ++q) {
        const int k = q * 4 + wave, g = k / 3;
        const int want = g < P_GROUPS / 2 ? I * (PT / 32) + g : J * (PT / 32) + g - P_GROUPS / 2;
        off[q] = (uint32_t)(want < ng ? want : ng - 1) * (uint32_t)(steps * kFragBytes) + (uint32_t)((k % 3) * 1024 + lane * 16);
    }
    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(base), 0, (int)((uint32_t)ng * (uint32_t)(steps * kFragBytes)), 0x00027000);
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
    const int a = wm * 2 * P_GSTRIDE, bo = (P_GROUPS / 2 + wn * 2) * P_GSTRIDE;
    if (!active) {
        tile_loop<false, false>(rows, lds, steps / 2, off, lane, wave, a, bo, re, im);
        if constexpr (FMT != OUT_GRID) return;
    } else {
        tile_loop<true, FMT == OUT_UPPER_PACKED || FMT == OUT_HERM_FULL>(rows, lds, steps / 2, off, lane, wave, a, bo, re, im);
    }
    const bool inside = wcol + 63 < wrow && wrow + 64 <= N;
    if constexpr (FMT == OUT_GRID) {
        static_assert(4 * kGridRegion <= P_BUFS * P_STAGE, "gridding regions");
        __syncthreads();  // the last stage is read
        grid_tile<4, 2>(*grid, N, I * PT, J * PT, active, alpha, re, im, lds, wave, lane);
    } else if constexpr (FMT != OUT_LOWER_PACKED) {
        if (inside) store_ggp_inside<OutT, FMT>(C, N, wrow, wcol, re, im, lane);
        else store_ggp_any<OutT, FMT>(C, N, wrow, wcol, re, im, lane);
    } else if (inside && beta == 0.0f) {
        if (nt) {
            if (alpha == 1.0f) store_pairs<OutT, false, true>(C, wrow, wcol, alpha, re, im, lane);
            else store_pairs<OutT, true, true>(C, wrow, wcol, alpha, re, im, lane);
        } else {
            if (alpha == 1.0f) store_inside<OutT, false, false>(C, wrow, wcol, alpha, re, im, lane);
            else store_inside<OutT, true, false>(C, wrow, wcol, alpha, re, im, lane);
        }
    } else if (nt) {
        store_any<OutT, true>(C, N, wrow, wcol, alpha, beta, re, im, lane);
    } else {
        store_any<OutT>(C, N, wrow, wcol, alpha, beta, re, im, lane);
    }
}

template <typename OutT, bool NT, int FMT = OUT_LOWER_PACKED>
__global__ void __launch_bounds__(P_THREADS, 2) herk_pipe_kernel(HerkPlainArgs p, int steps, int tiles) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[P_BUFS * P_STAGE];
    const int w = xcd_logical((int)blockIdx.x, tiles * p.batch);
    const int b = w / tiles, t = w - b * tiles;
    int I, J;
    // Launches that are bound by their stores go 2 x 2 tiles at a time (longer runs of each output
    // row together), those bound by operands 4 x 4; us for 1 / 2 / 4 / 8: 4096 x 16, K = 256 255 /
    // 261 / 276 / 281; 2500 x 20, K = 128 122 / 124 / 129 / 130; 3000 x 20, K = 64, FP16 79 / 78 / 83 /
    // 81; 1664 x 128, K = 128, FP16 212 / 205 / 207 / 206; 4096 x 96, K = 2048 4364 / 4203 / 4150 / 4160.
    tri_decode_blocked(t, (p.N + PT - 1) / PT, NT ? P_BLOCK : 2, I, J);
    const uint8_t* rows = p.A + (int64_t)b * p.a_bstride;
    if constexpr (FMT == OUT_GRID) {
        const GridJob g = grid_job(p, b);
        pipe_tile<OutT, FMT>(lds, rows, p.N, steps, I, J, nullptr, p.alpha, 0.0f, NT, &g);
    } else {
        pipe_tile<OutT, FMT>(lds, rows, p.N, steps, I, J, static_cast<OutT*>(p.C) + (int64_t)b * p.c_bstride, p.alpha,
                             p.beta, NT);
    }
}

// Tiles of many problems: workgroup b runs tiles[b].
template <typename OutT>
__global__ void __launch_bounds__(P_THREADS, 2)
herk_pipe_grouped_kernel(const PipeProblem* __restrict__ probs, const GroupItemDev* __restrict__ tiles) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[P_BUFS * P_STAGE];
    const GroupItemDev it = tiles[blockIdx.x];
    if (it.prob < 0) return;  // this XCD's list is shorter than the longest
    const PipeProblem p = probs[it.prob];
    int I, J;
    tri_decode_blocked(it.tile, (p.N + PT - 1) / PT, P_BLOCK, I, J);
    pipe_tile<OutT>(lds, p.rows, p.N, p.steps, I, J, static_cast<OutT*>(p.C), p.alpha, p.beta, p.nt != 0);
}

// ---- QC rows -> fragment rows ----
// HBM-bound (1 byte read, 1.5 written per sample).  A thread converts 16 samples of one row; a
// wave covers S segments x 64 / S rows, so it reads runs of 16 S bytes and writes runs of
// 64 / S x 16 bytes.

// 4 QC bytes -> E3M2 codes of their Re and Im nibbles, one per byte (bits 5:0)
__device__ __forceinline__ void qc4_codes(uint32_t x, uint32_t& re, uint32_t& im) {
    const uint32_t TLO = 0x12100C00u;  // e3m2(0..3)
    const uint32_t THI = 0x17161514u;  // e3m2(4..7)
    re = __builtin_amdgcn_perm(THI, TLO, (x >> 4) & 0x07070707u) | ((x >> 2) & 0x20202020u);
    im = __builtin_amdgcn_perm(THI, TLO, x & 0x07070707u) | ((x << 2) & 0x20202020u);
}

__device__ __forceinline__ uint32_t pack4(uint32_t c) {  // four byte-wide codes -> 24 bits
    return (c & 0x3Fu) | ((c >> 2) & 0xFC0u) | ((c >> 4) & 0x3F000u) | ((c >> 6) & 0xFC0000u);
}

__device__ __forceinline__ void pack16(const uint32_t (&c)[4], uint32_t& d0, uint32_t& d1, uint32_t& d2) {
    const uint32_t p0 = pack4(c[0]), p1 = pack4(c[1]), p2 = pack4(c[2]), p3 = pack4(c[3]);
    d0 = p0 | (p1 << 24);
    d1 = (p1 >> 8) | (p2 << 16);
    d2 = (p2 >> 16) | (p3 << 8);
}

// Four two's complement nibbles, one per byte -> their E3M2 codes: a 16-entry table over two
// lookups (0 .. 7, -8 .. -1) and a select on bit 3.
__device__ __forceinline__ uint32_t ggp_nib4_codes(uint32_t nib) {
    const uint32_t sel = nib & 0x07070707u;
    const uint32_t pos = __builtin_amdgcn_perm(0x17161514u, 0x12100C00u, sel);  // 4 .. 7, 0 .. 3
    const uint32_t neg = __builtin_amdgcn_perm(0x2C303234u, 0x35363738u, sel);  // -4 .. -1, -8 .. -5
    const uint32_t m = ((nib >> 3) & 0x01010101u) * 0xFFu;
    return (pos & ~m) | (neg & m);
}

// 16 samples' codes -> their place in the fragment step at dst (lane as in herk_pipe.h)
__device__ __forceinline__ void put_codes(const uint32_t (&re)[4], const uint32_t (&im)[4], uint8_t* dst, int lane) {
    uint4 a;
    uint2 b;
    pack16(re, a.x, a.y, a.z);
    pack16(im, a.w, b.x, b.y);
    *reinterpret_cast<uint4*>(dst + lane * 16) = a;
    *reinterpret_cast<uint2*>(dst + 1024 + lane * 8) = b;
}

// 16 QC samples -> their place in the fragment step at dst 
__device__ __forceinline__ void put_frag(uint4 w, uint8_t* dst, int lane) {
    uint32_t re[4], im[4];
    qc4_codes(w.x, re[0], im[0]);
    qc4_codes(w.y, re[1], im[1]);
    qc4_codes(w.z, re[2], im[2]);
    qc4_codes(w.w, re[3], im[3]);
    put_codes(re, im, dst, lane);
}

// Row and 16-sample segment of conversion thread t: waves of S segments x 64 / S rows, of one parity
// where paired.
__device__ __forceinline__ void conv_place(uint32_t t, int segs, int S, bool paired, int& r, int& s) {
    const uint32_t v = t / 64u, per = (uint32_t)(segs / S);
    const uint32_t rb = v / per, sb = v - rb * per;
    s = (int)sb * S + (int)(t % S);
    const int R = 64 / S, u = (int)(t / S) % R;
    r = paired ? (int)(rb >> 1) * 2 * R + 2 * u + (int)(rb & 1) : (int)rb * R + u;
}

// VEC: K % 16 == 0 and 16-byte aligned rows
template <bool VEC, int S>
__global__ void __launch_bounds__(256)
qc_frag_rows_kernel(const uint8_t* __restrict__ in, uint8_t* __restrict__ out, int N, int K, int steps, int nseg,
                    int grp, bool paired) {
    const int ng = frag_groups(N);
    int r, s;
    conv_place(blockIdx.x * 256u + threadIdx.x, steps * 2, S, paired, r, s);
    if (r >= ng * 32) return;
    const int ib = (int)blockIdx.y, ob = ib / (nseg * grp), sg = ib / grp - ob * nseg;
    const int64_t dst_batch = (int64_t)ob * grp + ib % grp;
    uint4 w = make_uint4(0u, 0u, 0u, 0u);
    if (r < N) {
        const uint8_t* row = in + ((int64_t)ib * N + r) * K;
        if constexpr (VEC) {
            if (s * 16 < K) w = *reinterpret_cast<const uint4*>(row + s * 16);
        } else {
            w = row_segment(row, s * 16, K);
        }
    }
    put_frag(w,
             out + ((dst_batch * ng + frag_group(r, paired)) * (int64_t)(steps * nseg) + sg * steps + (s >> 1)) * kFragBytes,
             frag_lane(r, paired) + 32 * (s & 1));
}

// The rows of many problems: workgroup b converts up to kConvThreads segments of one problem.
__global__ void __launch_bounds__(256)
qc_frag_rows_multi_kernel(const PipeProblem* __restrict__ probs, const ConvBlock* __restrict__ blocks) {
    const ConvBlock cb = blocks[blockIdx.x];
    const PipeProblem p = probs[cb.prob];
    const int ng = frag_groups(p.N), segs = p.steps * 2, S = segs % 8 == 0 ? 8 : 4;
    const bool vec = p.K % 16 == 0 && (reinterpret_cast<uintptr_t>(p.A) & 15u) == 0;
    for (uint32_t i = threadIdx.x; i < (uint32_t)kConvThreads; i += 256u) {
        int r, s;
        conv_place(cb.first + i, segs, S, p.nt, r, s);
        if (r >= ng * 32) return;
        uint4 w = make_uint4(0u, 0u, 0u, 0u);
        if (r < p.N) {
            const uint8_t* row = p.A + (int64_t)r * p.K;
            if (vec) {
                if (s * 16 < p.K) w = *reinterpret_cast<const uint4*>(row + s * 16);
            } else if (p.K >= 16) {
                w = row_segment(row, s * 16, p.K);
            } else if (s == 0) {
                uint32_t d[4] = {0u, 0u, 0u, 0u};
                for (int k = 0; k < p.K; ++k) d[k >> 2] |= (uint32_t)row[k] << (8 * (k & 3));
                w = make_uint4(d[0], d[1], d[2], d[3]);
            }
        }
        put_frag(w, p.rows + ((int64_t)frag_group(r, p.nt) * p.steps + (s >> 1)) * kFragBytes,
                 frag_lane(r, p.nt) + 32 * (s & 1));
    }
}

// GGP bytes [batch][K][N] (low nibble Re, high Im, two's complement) -> fragment rows.  A thread
// converts 16 samples of four rows; in a wave 16 lanes run along the rows (64-byte reads of
// each sample's run, 1-kilobyte runs of a group's operands) and 4 along the samples.
// ALIGNED: N % 4 == 0 and 4-byte aligned input.
template <bool ALIGNED>
__global__ void __launch_bounds__(256)
ggp_frag_rows_kernel(const uint8_t* __restrict__ in, uint8_t* __restrict__ out, int N, int K, int steps, int batches) {
    const int tid = threadIdx.x, ng = frag_groups(N);
    const int r0 = ((int)blockIdx.y * 64 + (tid & 15) + 16 * (tid >> 6)) * 4;
    const int s = (int)blockIdx.x * 4 + ((tid >> 4) & 3);  // whole stages: s < 2 steps
    if (r0 >= ng * 32) return;
    for (int b = blockIdx.z; b < batches; b += gridDim.z) {
        const uint8_t* src = in + (int64_t)b * K * N + r0;
        uint32_t d[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int k = s * 16 + e;
            uint32_t v = 0u;
            if (k < K && r0 < N) {
                const uint8_t* run = src + (int64_t)k * N;
                if (ALIGNED) {
                    v = *reinterpret_cast<const uint32_t*>(run);
                } else {
#pragma unroll
                    for (int a = 0; a < 4; ++a)
                        if (r0 + a < N) v |= (uint32_t)run[a] << (8 * a);
                }
            }
            d[e] = v;
        }
        uint32_t t[4][4];  // [sample quad][row]
#pragma unroll
        for (int g = 0; g < 4; ++g) transpose4x4_bytes(d[4 * g], d[4 * g + 1], d[4 * g + 2], d[4 * g + 3], t[g]);
        uint8_t* dst = out + (((int64_t)b * ng + (r0 >> 5)) * steps + (s >> 1)) * kFragBytes;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            uint32_t re[4], im[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                re[g] = ggp_nib4_codes(t[g][a] & 0x0F0F0F0Fu);
                im[g] = ggp_nib4_codes((t[g][a] >> 4) & 0x0F0F0F0Fu);
            }
            put_codes(re, im, dst, ((r0 + a) & 31) + 32 * (s & 1));
        }
    }
}

template <typename OutT>
void launch_ggp(const HerkPlainArgs& a, int fmt, int steps, int tiles, hipStream_t stream) {
    const dim3 grid((unsigned)((int64_t)tiles * a.batch)), block(P_THREADS);
    if (fmt == OUT_UPPER_PACKED)
        hipLaunchKernelGGL((herk_pipe_kernel<OutT, false, OUT_UPPER_PACKED>), grid, block, 0, stream, a, steps, tiles);
    else
        hipLaunchKernelGGL((herk_pipe_kernel<OutT, false, OUT_HERM_FULL>), grid, block, 0, stream, a, steps, tiles);
}

}  // namespace

bool pipe_supported(int N, int K, int nseg) {
    return N > 0 && K >= 16 && nseg >= 1 && (int64_t)K * nseg <= 0x7FFFFFFF - 64 * (int64_t)nseg &&
           frag_rows_bytes(N, K, nseg) <= 0x7FFFFFFFll;
}

int pipe_tiles(int N) {
    const int nb = (N + PT - 1) / PT;
    return nb * (nb + 1) / 2;
}

int pipe_wg_per_cu() { return P_WG_PER_CU; }

// Plain stores let the L2 join the partial lines at the ends of the runs, and fill it with
// output in place of operand rows: they pay where the launch writes more than it multiplies,
// the longer the longer the output's rows.  us, plain / non-temporal (paired rows), buffers in turn:
//   FP32, K =      128         256         384         512
//   512 x 400   115 / 134   147 / 146   179 / 156   213 / 181
//   1664 x 100  269 / 321   293 / 327   386 / 333   452 / 341
//   4000 x 12   190 / 237   192 / 239   218 / 239   261 / 240
//   FP16
//   512 x 400    70 / 86     95 / 100   127 / 118   170 / 156
//   1664 x 100  156 / 200   220 / 202   274 / 216   322 / 244
//   4000 x 12    94 / 147   125 / 152   152 / 152   172 / 154
bool pipe_nontemporal(int N, int samples, bool out_fp16) { return samples > (!out_fp16 && N >= 3000 ? 448 : 320); }

hipError_t launch_qc_frag_rows_multi(const PipeProblem* probs, const ConvBlock* blocks, int nblocks, hipStream_t s) {
    if (nblocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(qc_frag_rows_multi_kernel, dim3((unsigned)nblocks), dim3(256), 0, s, probs, blocks);
    return hipGetLastError();
}

hipError_t launch_herk_pipe_grouped(const PipeProblem* probs, const GroupItemDev* tiles, int ntiles, bool out_fp16,
                                    hipStream_t s) {
    if (ntiles <= 0) return hipSuccess;
    if (out_fp16)
        hipLaunchKernelGGL(herk_pipe_grouped_kernel<_Float16>, dim3((unsigned)ntiles), dim3(P_THREADS), 0, s, probs, tiles);
    else
        hipLaunchKernelGGL(herk_pipe_grouped_kernel<float>, dim3((unsigned)ntiles), dim3(P_THREADS), 0, s, probs, tiles);
    return hipGetLastError();
}

hipError_t launch_qc_frag_rows(const uint8_t* in, uint8_t* out, int N, int K, int batches, int nseg, int seg_group,
                               bool paired, hipStream_t stream) {
    if (N <= 0 || batches <= 0) return hipSuccess;
    if (!pipe_supported(N, K, nseg) || batches > 65535) return hipErrorInvalidValue;
    const int steps = frag_steps(K), segs = steps * 2, rows = frag_groups(N) * 32;
    const bool vec = K % 16 == 0 && (reinterpret_cast<uintptr_t>(in) & 15u) == 0;
    const dim3 grid((unsigned)(((int64_t)rows * segs + 255) / 256), (unsigned)batches), block(256);
    // 8 segments per wave where a row's segments allow it (whole stages have 4)
    if (segs % 8 == 0) {
        if (vec)
            hipLaunchKernelGGL((qc_frag_rows_kernel<true, 8>), grid, block, 0, stream, in, out, N, K, steps, nseg,
                               seg_group, paired);
        else
            hipLaunchKernelGGL((qc_frag_rows_kernel<false, 8>), grid, block, 0, stream, in, out, N, K, steps, nseg,
                               seg_group, paired);
    } else {
        if (vec)
            hipLaunchKernelGGL((qc_frag_rows_kernel<true, 4>), grid, block, 0, stream, in, out, N, K, steps, nseg,
                               seg_group, paired);
        else
            hipLaunchKernelGGL((qc_frag_rows_kernel<false, 4>), grid, block, 0, stream, in, out, N, K, steps, nseg,
                               seg_group, paired);
    }
    return hipGetLastError();
}

hipError_t launch_herk_pipe_grid(const HerkPlainArgs& a, hipStream_t stream) {
    if (a.N <= 0 || a.batch <= 0) return hipSuccess;
    const int tiles = pipe_tiles(a.N);
    const int64_t blocks = (int64_t)tiles * a.batch;
    if (blocks > 0x7FFFFFFF || !pipe_supported(a.N, a.K, a.nseg) || !a.uv_m || !a.freq_hz || a.Ng <= 0)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL((herk_pipe_kernel<float, false, OUT_GRID>), dim3((unsigned)blocks), dim3(P_THREADS), 0, stream, a,
                       frag_steps(a.K) * a.nseg, tiles);
    return hipGetLastError();
}

hipError_t launch_herk_pipe(const HerkPlainArgs& a, bool out_fp16, hipStream_t stream) {
    if (a.N <= 0 || a.batch <= 0) return hipSuccess;
    const int tiles = pipe_tiles(a.N);
    const int64_t blocks = (int64_t)tiles * a.batch;
    if (blocks > 0x7FFFFFFF || !pipe_supported(a.N, a.K, a.nseg)) return hipErrorInvalidValue;
    const int steps = frag_steps(a.K) * a.nseg;
    const dim3 grid((unsigned)blocks), block(P_THREADS);
    const bool nt = pipe_nontemporal(a.N, a.K * a.nseg, out_fp16);
    if (out_fp16) {
        if (nt)
            hipLaunchKernelGGL((herk_pipe_kernel<_Float16, true>), grid, block, 0, stream, a, steps, tiles);
        else
            hipLaunchKernelGGL((herk_pipe_kernel<_Float16, false>), grid, block, 0, stream, a, steps, tiles);
    } else {
        if (nt)
            hipLaunchKernelGGL((herk_pipe_kernel<float, true>), grid, block, 0, stream, a, steps, tiles);
        else
            hipLaunchKernelGGL((herk_pipe_kernel<float, false>), grid, block, 0, stream, a, steps, tiles);
    }
    return hipGetLastError();
}

hipError_t launch_ggp_frag_rows(const uint8_t* in, uint8_t* out, int N, int K, int batches, hipStream_t stream) {
    if (N <= 0 || K <= 0 || batches <= 0) return hipSuccess;
    const int steps = frag_steps(K);
    const dim3 grid((unsigned)(steps / 2), (unsigned)((N + 255) / 256), (unsigned)(batches < 65535 ? batches : 65535));
    if (N % 4 == 0 && (reinterpret_cast<uintptr_t>(in) & 3u) == 0)
        hipLaunchKernelGGL(ggp_frag_rows_kernel<true>, grid, dim3(256), 0, stream, in, out, N, K, steps, batches);
    else
        hipLaunchKernelGGL(ggp_frag_rows_kernel<false>, grid, dim3(256), 0, stream, in, out, N, K, steps, batches);
    return hipGetLastError();
}

hipError_t launch_herk_pipe_ggp(const HerkPlainArgs& a, int fmt, bool out_fp64, hipStream_t stream) {
    if (a.N <= 0 || a.batch <= 0) return hipSuccess;
    const int tiles = pipe_tiles(a.N), steps = frag_steps(a.K);
    if ((int64_t)tiles * a.batch > 0x7FFFFFFF || !pipe_supported(a.N, a.K)) return hipErrorInvalidValue;
    if (out_fp64) launch_ggp<double>(a, fmt, steps, tiles, stream);
    else launch_ggp<float>(a, fmt, steps, tiles, stream);
    return hipGetLastError();
}

}  // namespace ftdx
