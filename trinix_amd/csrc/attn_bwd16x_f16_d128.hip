// dK/dV kernels for f16, head_dim 128, in pieces or with narrow rows (one
// translation unit per instantiation keeps compile times parallel).
#include "attn_bwd16.h"

namespace trinix {
TRINIX_ATTN_BWD16_LAUNCHER(launch_dkdv16x_f16_d128, F16, 128, kDkdvExt)
}  // namespace trinix
