// fp32 backward kernels, head_dim 64, 128 and 256.
#include "attn_bwd_generic.h"

namespace trinix {

hipError_t launch_bwd_generic_f32(const BwdParams& p, int D, const BwdPlan& plan, hipStream_t st) {
  hipError_t e;
  switch (D) {
    case 64:
      e = plan.kv_ks == 2 ? launch_generic_dkdv<Ops32<64>, 2, 1, 2>(p, st) : launch_generic_dkdv<Ops32<64>, 2, 1, 1>(p, st);
      if (e != hipSuccess) return e;
      return plan.dq_ks == 2 ? launch_generic_dq<Ops32<64>, 2, 1, 2>(p, st) : launch_generic_dq<Ops32<64>, 2, 1, 1>(p, st);
    case 128:
      e = plan.kv_ks == 2 ? launch_generic_dkdv<Ops32<128>, 1, 1, 2>(p, st) : launch_generic_dkdv<Ops32<128>, 1, 1, 1>(p, st);
      if (e != hipSuccess) return e;
      return plan.dq_ks == 2 ? launch_generic_dq<Ops32<128>, 1, 1, 2>(p, st) : launch_generic_dq<Ops32<128>, 1, 1, 1>(p, st);
    case 256:  // K and V rows and 64 columns of dK and dV fill the registers
      e = launch_generic_dkdv<Ops32<256>, 1, 4, 1>(p, st);
      return e != hipSuccess ? e : launch_generic_dq<Ops32<256>, 1, 2, 1>(p, st);
  }
  return hipErrorNotSupported;
}

}  // namespace trinix
