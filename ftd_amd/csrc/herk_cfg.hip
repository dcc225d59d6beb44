// herk_cfg.hip -- the kernels of one tile configuration (-DFTDX_CFG=Cfg<id>, see herk_launch.h).
#include "herk_launch.h"

namespace ftdx {

template hipError_t launch_plain_cfg<FTDX_CFG>(const HerkPlainArgs&, bool, int, hipStream_t);
template hipError_t launch_gemm_cfg<FTDX_CFG>(const GemmArgs&, int, bool, int, hipStream_t);
template hipError_t launch_grid_cfg<FTDX_CFG>(const HerkPlainArgs&, int, hipStream_t);
template hipError_t launch_ggp_cfg<FTDX_CFG>(const HerkPlainArgs&, int, bool, int, hipStream_t);
template hipError_t launch_grouped_cfg<FTDX_CFG>(const GroupProblemDev*, const GroupItemDev*, const int*, int, bool,
                                                 bool, hipStream_t);

}  // namespace ftdx
