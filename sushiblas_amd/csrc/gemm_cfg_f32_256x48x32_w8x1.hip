// gemm_cfg_f32_256x48x32_w8x1.hip -- instantiates the fp32 split tile
// (gemm_split.hpp): 8 waves of 32x48: the 256x64 tile computing its first 48
// columns.  The name is the plan's (kCfg).
#include "launch_split_impl.hpp"

namespace sbx {
template hipError_t launch_split<256, 64, 8, 1, 2, 2, 48>(const GemmArgs<float>&, bool, bool, int, hipStream_t);
}  // namespace sbx
