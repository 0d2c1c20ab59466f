// gemm_cfg_f32_48x256x32_w1x8.hip -- instantiates the fp32 split tile
// (gemm_split.hpp): 8 waves of 48x32: the 64x256 tile computing its first 48
// rows.  The name is the plan's (kCfg).
#include "launch_split_impl.hpp"

namespace sbx {
template hipError_t launch_split<64, 256, 1, 8, 2, 2, 256, 48>(const GemmArgs<float>&, bool, bool, int, hipStream_t);
}  // namespace sbx
