// conv_split_gather.hip - the split-bf16 conv kernels of one B loader (SplitGather<false>).
#include "conv_split.h"

namespace spinn {

int launch_conv_split_gather(const ConvSplitArgs &a, int bm, int groups, int split, const SkSched *sk, int sk_grid,
                      hipStream_t st) {
    return bm == 128 ? launch_conv_split_act<128, SplitGather<false>>(a, groups, split, sk, sk_grid, st)
                     : launch_conv_split_act<64, SplitGather<false>>(a, groups, split, sk, sk_grid, st);
}

} // namespace spinn
