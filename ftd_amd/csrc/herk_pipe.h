// herk_pipe.h -- host-side launch interface of the pipelined HERK (internal).
//
// The HERK of QC voltages over E3M2 fragment rows: every QC value is exact in E3M2, and
// the matrix cores take 6-bit operands at twice the FP8 rate.  Layout of the rows of one
// batch: [group of 32 rows][step of 32 samples][1536 bytes], the operand of one 32x32x64
// MFMA in lane order.  Lane l holds row l % 32, samples 16 (l / 32) .. + 15 of the step: 16
// six-bit Re codes then 16 Im codes (code k at bits 6k), six dwords, the first four of all
// lanes at 16 l, the last two at 1024 + 8 l.  So a wave copies whole kilobytes from memory
// to LDS and reads its operands from there without bank conflicts, 48 bytes per 32 samples.
// Rows past N and samples past K are zero.  "Paired" rows: of each 64 rows the even ones are one
// group and the odd ones the next, so that a lane's outputs in the two column groups of its
// wave are neighbours in memory.
#pragma once
#include "herk_fp8.h"

namespace ftdx {

constexpr int kFragBytes = 1536;

// Row groups of N rows (whole blocks of 64); row r's group, and its lane in it.
__host__ __device__ inline int frag_groups(int N) { return (N + 63) / 64 * 2; }
__host__ __device__ inline int frag_group(int r, bool paired) { return paired ? (r >> 6) * 2 + (r & 1) : r >> 5; }
__host__ __device__ inline int frag_lane(int r, bool paired) { return paired ? (r & 63) >> 1 : r & 31; }

// 32-sample steps of a row of K samples (whole 64-sample stages).
inline int frag_steps(int K) { return (K + 63) / 64 * 2; }
// Bytes of one batch's fragment rows (nseg segments of K samples per row).
inline int64_t frag_rows_bytes(int N, int K, int nseg = 1) {
    return (int64_t)frag_groups(N) * frag_steps(K) * nseg * kFragBytes;
}

// Whether the pipelined HERK takes this problem: 16-byte row loads (K >= 16) and one
// batch's fragment rows within a 32-bit buffer offset.
bool pipe_supported(int N, int K, int nseg = 1);

// QC rows [batches][N][K] (any K >= 16, any alignment) -> fragment rows.  Input batch
// (ob * nseg + s) * seg_group + i becomes segment s of output batch ob * seg_group + i.
hipError_t launch_qc_frag_rows(const uint8_t* in, uint8_t* out, int N, int K, int batches, int nseg, int seg_group,
                               bool paired, hipStream_t stream);

// The HERK over fragment rows: a.A the rows, a.a_bstride their bytes per batch, a.K the
// samples of one segment (a.nseg of them); packed lower triangle as launch_herk_int4_plain.
// The rows are paired where pipe_nontemporal(a.N, a.K * a.nseg, out_fp16).
hipError_t launch_herk_pipe(const HerkPlainArgs& a, bool out_fp16, hipStream_t stream);

// GGP bytes [batches][K][N], any alignment -> fragment rows; the HERK over them with the GGP
// layouts of launch_herk_ggp (OUT_UPPER_PACKED or OUT_HERM_FULL, FP32 or FP64), alpha 1, beta 0.
hipError_t launch_ggp_frag_rows(const uint8_t* in, uint8_t* out, int N, int K, int batches, hipStream_t stream);
hipError_t launch_herk_pipe_ggp(const HerkPlainArgs& a, int fmt, bool out_fp64, hipStream_t stream);

// The HERK over fragment rows whose epilogue grids (OUT_GRID), as launch_herk_grid.
hipError_t launch_herk_pipe_grid(const HerkPlainArgs& a, hipStream_t stream);

// Tiles per batch and resident workgroups per CU of the launch above.
int pipe_tiles(int N);
int pipe_wg_per_cu();

// Whether the stores of the launch above are non-temporal (samples: of all segments).
bool pipe_nontemporal(int N, int samples, bool out_fp16);

// ---- many problems of different sizes ----
struct PipeProblem {
    const uint8_t* A;  // QC rows [N][K], any K >= 0 and alignment
    uint8_t* rows;     // their fragment rows, 16-byte aligned
    void* C;
    int N, K, steps;   // steps: max(frag_steps(K), 2)
    int nt;            // pipe_nontemporal: non-temporal stores, paired rows
    float alpha, beta;
};
// Segments from `first` of problem `prob`: 32 frag_groups(N) * 2 steps of them in all.
constexpr int kConvThreads = 2048;
struct ConvBlock {
    int prob;
    uint32_t first;  // a multiple of kConvThreads
};
// All arrays in device memory.  tiles[b]: problem and tile (0 .. pipe_tiles(N) - 1) of
// workgroup b, prob < 0 for none; workgroup b runs on XCD b mod 8.
hipError_t launch_qc_frag_rows_multi(const PipeProblem* probs, const ConvBlock* blocks, int nblocks, hipStream_t stream);
hipError_t launch_herk_pipe_grouped(const PipeProblem* probs, const GroupItemDev* tiles, int ntiles, bool out_fp16,
                                    hipStream_t stream);

}  // namespace ftdx
