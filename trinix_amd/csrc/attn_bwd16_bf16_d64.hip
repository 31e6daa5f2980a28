// Backward kernels for bf16, head_dim 64 (one translation unit per
// instantiation keeps compile times parallel).
#include "attn_bwd16.h"

namespace trinix {
TRINIX_ATTN_BWD16_LAUNCHER(launch_dkdv16_bf16_d64, BF16, 64, kDkdv)
TRINIX_ATTN_BWD16_LAUNCHER(launch_dq16_bf16_d64, BF16, 64, kDq)
}  // namespace trinix
