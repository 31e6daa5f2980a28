// bf16 backward kernels at head_dim 256.
#include "attn_bwd_generic.h"

namespace trinix {

hipError_t launch_bwd_generic_bf16(const BwdParams& p, const BwdPlan& plan, hipStream_t st) {
  using O = Ops16<BF16, 256>;
  const hipError_t e = plan.kv_ks == 2 ? launch_generic_dkdv<O, 1, 2, 2>(p, st) : launch_generic_dkdv<O, 1, 2, 1>(p, st);
  if (e != hipSuccess) return e;
  return plan.dq_ks == 2 ? launch_generic_dq<O, 1, 1, 2>(p, st) : launch_generic_dq<O, 1, 1, 1>(p, st);
}

}  // namespace trinix
