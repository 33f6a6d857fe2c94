// Wide forward, head dim 128.
#include "htree_fwd_wide.h"

namespace htree {
template void launch_fwd_wide_d<128>(int dtype, const FwdArgs& a, dim3 grid, hipStream_t st, bool sel);
}  // namespace htree
