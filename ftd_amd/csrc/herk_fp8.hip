// herk_fp8.hip -- dispatch of the HERK and GEMM launches to the tile configurations
// (kernels in herk_launch.h, compiled per configuration from herk_cfg.hip).
#include "herk_launch.h"

namespace ftdx {

#define FTDX_EXTERN_CFG(C)                                                                          \
    extern template hipError_t launch_plain_cfg<C>(const HerkPlainArgs&, bool, int, hipStream_t);    \
    extern template hipError_t launch_gemm_cfg<C>(const GemmArgs&, int, bool, int, hipStream_t);     \
    extern template hipError_t launch_grid_cfg<C>(const HerkPlainArgs&, int, hipStream_t);           \
    extern template hipError_t launch_ggp_cfg<C>(const HerkPlainArgs&, int, bool, int, hipStream_t); \
    extern template hipError_t launch_grouped_cfg<C>(const GroupProblemDev*, const GroupItemDev*,    \
                                                     const int*, int, bool, bool, hipStream_t);
FTDX_EXTERN_CFG(Cfg0)
FTDX_EXTERN_CFG(Cfg1)
FTDX_EXTERN_CFG(Cfg2)
FTDX_EXTERN_CFG(Cfg3)
FTDX_EXTERN_CFG(Cfg4)
FTDX_EXTERN_CFG(Cfg5)
#undef FTDX_EXTERN_CFG

namespace {

// Calls f(CfgN{}) for tile configuration id `cfg`; hipErrorInvalidValue for unknown ids.
template <typename F>
hipError_t with_cfg(int cfg, F&& f) {
    switch (cfg) {
        case TILE_128x128_K64: return f(Cfg0{});
        case TILE_128x128_K128: return f(Cfg1{});
        case TILE_64x64_K64: return f(Cfg2{});
        case TILE_256x128_K64: return f(Cfg3{});
        case TILE_128x128_K64_P2: return f(Cfg4{});
        case TILE_256x128_K64_P2: return f(Cfg5{});
        default: return hipErrorInvalidValue;
    }
}

template <typename F>
int cfg_value(int cfg, F&& f, int fallback) {
    int v = fallback;
    (void)with_cfg(cfg, [&](auto c) {
        v = f(c);
        return hipSuccess;
    });
    return v;
}

hipError_t launch_gemm_beam_cfg0(const GemmArgs& a, bool out_u8, int xcd_remap, hipStream_t stream) {
    using Cfg = Cfg0;
    if (a.beam_nt <= 0 || 64 % a.beam_nt != 0 || a.M != (a.beam_samples + 63) / 64 * Cfg::TM)
        return hipErrorInvalidValue;
    const int64_t tiles_m = a.M / Cfg::TM, tiles_n = (a.N + Cfg::TN - 1) / Cfg::TN;
    const int64_t blocks = tiles_m * tiles_n * a.batch;
    if (blocks > 0x7FFFFFFF) return hipErrorInvalidValue;
    if (blocks == 0) return hipSuccess;
    dim3 grid((unsigned)blocks), block(Cfg::THREADS);
    const int tm = (int)tiles_m, tiles = (int)(tiles_m * tiles_n);
    if (out_u8)
        hipLaunchKernelGGL((gemm_fp8_kernel<Cfg, uint8_t, OUT_GEMM_BEAM>), grid, block, 0, stream, a, tm,
                           tiles, xcd_remap);
    else
        hipLaunchKernelGGL((gemm_fp8_kernel<Cfg, float, OUT_GEMM_BEAM>), grid, block, 0, stream, a, tm,
                           tiles, xcd_remap);
    return hipGetLastError();
}

}  // namespace

int tile_config_rows(int cfg) {
    return cfg_value(cfg, [](auto c) { return decltype(c)::TM; }, 0);
}

int tile_config_cols(int cfg) {
    return cfg_value(cfg, [](auto c) { return decltype(c)::TN; }, 0);
}

int tile_config_wg_per_cu(int cfg) {
    return cfg_value(cfg, [](auto c) { return decltype(c)::WG_PER_CU; }, 1);
}

int herk_tiles(int cfg, int N) { return tri_tiles(N, tile_config_rows(cfg), tile_config_cols(cfg)); }

bool mx4d_dense_ok(int cfg, int N, int64_t lda) {
    return cfg_value(
               cfg,
               [&](auto c) {
                   using Cfg = decltype(c);
                   return (TileRunner<Cfg>::MX4D_OK && TileRunner<Cfg>::DMA_OK && N > 0 && N % Cfg::TM == 0 &&
                           N % Cfg::TN == 0 && lda > 0 && lda % 16 == 0 && (int64_t)N * lda <= 0xFFFFFFFFll)
                              ? 1
                              : 0;
               },
               0) != 0;
}

hipError_t launch_herk_int4_plain(const HerkPlainArgs& a, int cfg, bool out_fp16, int xcd_remap,
                                  hipStream_t stream) {
    if (a.N <= 0 || a.batch <= 0) return hipSuccess;
    return with_cfg(cfg, [&](auto c) {
        return launch_plain_cfg<decltype(c)>(a, out_fp16, xcd_remap, stream);
    });
}

hipError_t launch_herk_ggp(const HerkPlainArgs& a, int cfg, int fmt, bool out_fp64, int xcd_remap,
                           hipStream_t stream) {
    if (a.N <= 0 || a.batch <= 0) return hipSuccess;
    return with_cfg(cfg, [&](auto c) {
        return launch_ggp_cfg<decltype(c)>(a, fmt, out_fp64, xcd_remap, stream);
    });
}

hipError_t launch_herk_grid(const HerkPlainArgs& a, int cfg, int xcd_remap, hipStream_t stream) {
    if (a.N <= 0 || a.batch <= 0) return hipSuccess;
    return with_cfg(cfg, [&](auto c) { return launch_grid_cfg<decltype(c)>(a, xcd_remap, stream); });
}

hipError_t launch_gemm_beam(const GemmArgs& a, bool out_u8, int xcd_remap, hipStream_t stream) {
    return launch_gemm_beam_cfg0(a, out_u8, xcd_remap, stream);
}

hipError_t launch_gemm_fp8(const GemmArgs& a, int cfg, int fmt, bool out_fp16, int xcd_remap,
                           hipStream_t stream) {
    if (a.M <= 0 || a.N <= 0 || a.batch <= 0) return hipSuccess;
    return with_cfg(cfg, [&](auto c) {
        return launch_gemm_cfg<decltype(c)>(a, fmt, out_fp16, xcd_remap, stream);
    });
}

hipError_t launch_herk_int4_grouped(const GroupProblemDev* probs, const GroupItemDev* items,
                                    const int* wg_begin, int num_wg, int cfg, bool out_fp16, bool all_vec,
                                    hipStream_t stream) {
    if (num_wg <= 0) return hipSuccess;
    return with_cfg(cfg, [&](auto c) {
        return launch_grouped_cfg<decltype(c)>(probs, items, wg_begin, num_wg, out_fp16, all_vec, stream);
    });
}

}  // namespace ftdx
