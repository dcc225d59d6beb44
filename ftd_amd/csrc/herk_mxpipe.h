// herk_mxpipe.h -- host-side launch interface of the pipelined block-scaled HERK (internal).
//
// MX operand fragments of one batch: [group of 32 rows][stage of two 32-sample blocks][block 0,
// block 1, scales].  A block is the operand of one scaled 32x32x64 MFMA in lane order: lane l holds
// the Re (l < 32) or Im codes of row l % 32, E3M2 as in herk_pipe.h (1536 bytes), E2M1 four
// dwords at 16 l (1024 bytes).  Scales: 128 bytes, lane l's E8M0 bytes of the two blocks at 2 l.
#pragma once
#include "herk_fp8.h"
#include "herk_mx.h"

namespace ftdx {

constexpr int mxfrag_bytes(int fmt) { return fmt == MX_FP4_E2M1 ? 1024 : 1536; }

// Bytes of one batch's fragments.
inline int64_t mxfrag_rows_bytes(int N, int K, int fmt) {
    return (int64_t)((N + 31) / 32) * (((int64_t)K + 63) / 64) * (2 * mxfrag_bytes(fmt) + 128);
}

// Whether one batch's fragments fit a 32-bit buffer offset.
inline bool mxpipe_supported(int N, int K, int fmt) {
    return N > 0 && K > 0 && K <= 0x7FFFFFFF - 64 && mxfrag_rows_bytes(N, K, fmt) <= 0x7FFFFFFFll;
}

// X [batches][N][K] QC bytes or FP16 pairs (as launch_mx_quantize) -> fragments.
hipError_t launch_mx_frag_rows(const void* X, int input, int fmt, int rounding, uint8_t* out, int N, int K,
                               int batches, hipStream_t stream);

// The HERK over fragments: a.A, a.a_bstride bytes per batch; packed lower triangle.
hipError_t launch_herk_mxpipe(const HerkPlainArgs& a, int fmt, bool out_fp16, hipStream_t stream);

}  // namespace ftdx
