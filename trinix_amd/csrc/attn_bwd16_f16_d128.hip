// Backward kernels for f16, head_dim 128 (one translation unit per
// instantiation keeps compile times parallel).
#include "attn_bwd16.h"

namespace trinix {
TRINIX_ATTN_BWD16_LAUNCHER(launch_dkdv16_f16_d128, F16, 128, kDkdv)
TRINIX_ATTN_BWD16_LAUNCHER(launch_dq16_f16_d128, F16, 128, kDq)
}  // namespace trinix
