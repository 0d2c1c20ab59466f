// gemm_cfg_f32_256x256x32_w4x2.hip -- instantiates the fp32 split tile
// (gemm_split.hpp): 8 waves of 32x256, one workgroup per CU.  The name is the
// plan's (kCfg).
#include "launch_split_impl.hpp"

namespace sbx {
template hipError_t launch_split<256, 256, 8, 1, 1, 2>(const GemmArgs<float>&, bool, bool, int, hipStream_t);
}  // namespace sbx
