// Backward instances: head_dim 128, binary16 and bfloat16 (stats, dK/dV and dQ kernels).
#include "fa_bwd_kernel.h"

namespace fa {
template void launch_bwd<128, false, false>(const BwdArgs&, const BwdSplit&, int, bool, hipStream_t);
template void launch_bwd<128, true, false>(const BwdArgs&, const BwdSplit&, int, bool, hipStream_t);
}  // namespace fa
