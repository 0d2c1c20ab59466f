// gemm_cfg_f32_128x128x16_w2x2_o3.hip -- instantiates the fp32 split tile
// (gemm_split.hpp): 4 waves of 32x128, at most 168 VGPRs: three workgroups per
// CU (768 tiles in one round on 256 CUs).  The name is the plan's (kCfg).
#include "launch_split_impl.hpp"

namespace sbx {
template hipError_t launch_split<128, 128, 4, 1, 1, 3>(const GemmArgs<float>&, bool, bool, int, hipStream_t);
}  // namespace sbx
