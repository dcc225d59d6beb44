// herk_direct.h -- host-side launch interface of the direct HERK for small problems (internal).
#pragma once
#include "herk_fp8.h"

namespace ftdx {

// QC rows [batch][N][K] of any K >= 16 and any alignment; one input batch per output batch.
bool direct_supported(int N, int K, int batch);
int direct_tiles(int N);  // 32 x 32 tiles per batch
hipError_t launch_herk_direct(const HerkPlainArgs& a, bool out_fp16, hipStream_t stream);

}  // namespace ftdx
