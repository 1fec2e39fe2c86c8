// conv_split_pw2.hip - the split-bf16 conv kernels of one B loader (SplitPw2).
#include "conv_split.h"

namespace spinn {

int launch_conv_split_pw2(const ConvSplitArgs &a, int bm, int groups, int split, const SkSched *sk, int sk_grid,
                      hipStream_t st) {
    return bm == 128 ? launch_conv_split_act<128, SplitPw2>(a, groups, split, sk, sk_grid, st)
                     : launch_conv_split_act<64, SplitPw2>(a, groups, split, sk, sk_grid, st);
}

} // namespace spinn
