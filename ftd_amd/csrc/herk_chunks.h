// herk_chunks.h -- how many batches one conversion pass and the multiply after it take (internal; no
// HIP call, so the host tests build it with g++).
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <algorithm>

#include "herk_pipe.h"

namespace ftdx {

// Pre-cast paths (FP16 input, ForceBaseline, E3M2 operands) convert and multiply a chunk
// of batches at a time: the chunk's operand rows (at most kPrecastChunkBytes) are then
// still in the memory-side cache when its tiles read them, and the scratch holds one
// chunk.  Among chunk sizes up to that cap, the one whose launches leave the fewest idle
// workgroup slots in their last rounds (plus a small cost per launch) wins.
constexpr size_t kPrecastChunkBytes = size_t(320) << 20;

// batches of `per` scratch bytes each that fit one chunk
inline int chunk_cap_bytes(size_t per, int batch, size_t limit = kPrecastChunkBytes) {
    const size_t cap = per > 0 ? limit / per : (size_t)batch;
    return (int)std::max<size_t>(1, std::min<size_t>(cap, (size_t)std::max(batch, 1)));
}

// Among the chunks of 1 .. cmax batches (at least 1) the cheapest by the rule above, launches of
// `tiles` workgroups per batch on `slots` workgroup slots.
inline int pick_chunk_of(int64_t slots, int64_t tiles, int batch, int cmax) {
    cmax = std::max(cmax, 1);
    if (cmax >= batch) return std::max(batch, 1);
    double best = 1e30;
    int pick = cmax;
    for (int c = cmax; c >= 1; --c) {
        int64_t idle = 0;
        for (int b0 = 0; b0 < batch; b0 += c) {
            const int64_t t = tiles * std::min(c, batch - b0);
            idle += (t + slots - 1) / slots * slots - t;
        }
        const double cost = (double)idle / (double)slots + 0.1 * ((batch + c - 1) / c);
        if (cost < best) {
            best = cost;
            pick = c;
        }
    }
    return pick;
}

// Chunks of batches as on the pre-cast paths, for the same reason; at most 160 MB, so that a
// chunk's rows and its output share the 256 MB memory-side cache and the next chunk's rows
// overwrite them there, and at most 80 MB where that makes two chunks of what would be one.  us
// for 160 / 80 / 48 MB, buffers in turn: 4096 x 96, K = 2048 4116 / 4253 / 4405; 1024 x 200, K = 2048
// 744 / 891 / 892; 1152 x 66, K = 1024 (117 MB in all) 196 / 180 / 202; 700 x 60, K = 2000, FP16
// (130 MB) 141 / 137 / 152; 1024 x 64, K = 1024 (101 MB) 150 / 147 / 171.
// A launch's input batches are a grid's y dimension: 0 where the nseg segments of one batch alone
// are more than that, and the call takes the fused tile, which loops over them.
constexpr size_t kFragChunkBytes = size_t(160) << 20;

inline int frag_chunk_cap(int N, int K, int nseg, int batch) {
    const size_t per = (size_t)frag_rows_bytes(N, K, nseg);
    const size_t limit = per * (size_t)std::max(batch, 1) <= kFragChunkBytes ? kFragChunkBytes / 2 : kFragChunkBytes;
    return std::min(chunk_cap_bytes(per, batch, limit), 65535 / std::max(nseg, 1));
}

// Repeated on the same buffers, as the autotuner runs it, the conversion finds inputs of up to 100 MB in
// the memory-side cache; a program whose buffers change pays for them what 0.45 bytes per sample take at
// 5 TB/s.  us more with three sets of buffers in turn: 512 x 100, K = 1024 (52 MB) 4.6, 1024 x 64, K = 1024
// (67 MB) 5.9; 1024 x 64, K = 2048 (134 MB) -0.2, 1024 x 128 (268 MB) -2.4, 4096 x 96 (805 MB) -2.5.
inline double pipe_cold_ms(int64_t samples) { return samples <= 100000000 ? (double)samples * 0.45 / 5e9 : 0.0; }

}  // namespace ftdx
