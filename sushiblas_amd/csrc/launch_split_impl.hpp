// launch_split_impl.hpp -- definition of launch_split (see launch.hpp), for the
// gemm_cfg_*.hip translation units that instantiate a tile of gemm_split.hpp.
#pragma once

#include "gemm_split.hpp"
#include "launch_mfma_impl.hpp"

namespace sbx {

template <int BM, int BN, int WM, int WN, int PF, int WPE, int BNC, int BMC>
hipError_t launch_split(const GemmArgs<float>& a, bool a_kc, bool b_kc, int batch, hipStream_t stream)
{
    const dim3 grid((unsigned)(a.num_full + (a.tiles - a.num_full) * a.split), 1, (unsigned)batch);
    const dim3 block(WM * WN * 64);
    // the variants of launch_mfma: k-tail masking, and the non-temporal
    // operand of the tall and wide tiles
    const bool tail = (a_kc || b_kc) && a.K % 4 != 0;
    constexpr int kStream = BN <= 64 ? 1 : (BM <= 64 ? 2 : 0);
    const bool streamed = kStream != 0 && a.stream_op == kStream;
#define SBX_LAUNCH(AK, BKC, TAIL)                                                          \
    do {                                                                                   \
        if (streamed)                                                                      \
            gemm_split_kernel<BM, BN, WM, WN, AK, BKC, TAIL, PF, WPE, kStream, BNC, BMC>   \
                <<<grid, block, 0, stream>>>(a);                                           \
        else                                                                               \
            gemm_split_kernel<BM, BN, WM, WN, AK, BKC, TAIL, PF, WPE, 0, BNC, BMC>         \
                <<<grid, block, 0, stream>>>(a);                                           \
    } while (0)
    if (a_kc && b_kc) {
        if (tail) SBX_LAUNCH(true, true, true);
        else SBX_LAUNCH(true, true, false);
    } else if (a_kc) {
        if (tail) SBX_LAUNCH(true, false, true);
        else SBX_LAUNCH(true, false, false);
    } else if (b_kc) {
        if (tail) SBX_LAUNCH(false, true, true);
        else SBX_LAUNCH(false, true, false);
    } else {
        SBX_LAUNCH(false, false, false);
    }
#undef SBX_LAUNCH
    return launch_reduce<float, BM, BN>(a, batch, stream);
}

}  // namespace sbx
