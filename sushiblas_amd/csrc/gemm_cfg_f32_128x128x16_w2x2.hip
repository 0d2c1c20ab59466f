// gemm_cfg_f32_128x128x16_w2x2.hip -- instantiates the fp32 split tile
// (gemm_split.hpp): 4 waves of 32x128, two workgroups per CU.  The name is the
// plan's (kCfg).
#include "launch_split_impl.hpp"

namespace sbx {
template hipError_t launch_split<128, 128, 4, 1, 2, 2>(const GemmArgs<float>&, bool, bool, int, hipStream_t);
}  // namespace sbx
