// trinix_pad_heads: zero-pads the rows of up to three (B, S, H, D) 16-bit
// tensors (q, k and v) to a kernel head_dim in one launch.  HBM-bound (2 bytes
// read per element, 2 written per padded element), and for the small tensors
// it usually serves bound by the launch.  A training step at B=3 S=777/1111
// H=10 D=80 fp16 spent 45 us on torch's four fills and five copies (and took
// the full host path); with this launch, dout padded by the delta pass and out,
// dq, dk and dv at their own width it went from 228 to 149 us (this kernel 11;
// the unit's indexes in 32-bit divisions: 10.8 against 11.5, nothing in the step).
#include "common.h"
#include "trinix_attn.h"

namespace trinix {

struct PadParams {
  const uint16_t* x[3];
  uint16_t* out[3];
  int64_t sb[3], ss[3], sh[3], units[3];  // element strides; 16-byte units of out
  int S[3], H[3];
  int vec[3];  // 16-byte loads
  int D, UPR;  // elements read, 16-byte units written per row
};

// One 16-byte unit (8 elements) of one output row per thread.
__global__ __launch_bounds__(256) void pad_heads_kernel(const PadParams p) {
  const int n = blockIdx.y;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= p.units[n]) return;
  const PadUnit pu = pad_unit(t, p.UPR, p.H[n], p.S[n]);
  const uint16_t* x = p.x[n] + pu.b * p.sb[n] + pu.s * p.ss[n] + pu.h * p.sh[n] + pu.u * 8;
  const int live = p.D - pu.u * 8;  // elements of the unit that exist
  u32x4_t w = {};
  if (p.vec[n]) {
    if (live > 0) w = *(const u32x4_t*)x;
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < live) w[e / 2] |= (uint32_t)x[e] << (16 * (e & 1));
  }
  *(u32x4_t*)(p.out[n] + t * 8) = w;
}

}  // namespace trinix

using namespace trinix;

extern "C" int trinix_pad_heads(int32_t n, const void* const* x, const int64_t* x_stride, void* const* out,
                                const int64_t* sizes, int64_t head_dim, int64_t out_dim, int32_t dtype, void* stream) {
  if (!x || !x_stride || !out || !sizes) return TRINIX_ERR_NULL_POINTER;
  if (dtype != TRINIX_BF16 && dtype != TRINIX_F16) return TRINIX_ERR_BAD_DTYPE;
  if (n < 1 || n > 3) return TRINIX_ERR_BAD_ARGUMENT;
  if (head_dim <= 0 || out_dim < head_dim || out_dim % 8 != 0 || out_dim > 1024) return TRINIX_ERR_BAD_HEAD_DIM;
  PadParams p{};
  p.D = (int)head_dim;
  p.UPR = (int)(out_dim / 8);
  int64_t most = 0;
  for (int k = 0; k < n; ++k) {
    const int64_t *st = x_stride + 4 * k, *sz = sizes + 3 * k;
    if (!x[k] || !out[k]) return TRINIX_ERR_NULL_POINTER;
    if (sz[0] <= 0 || sz[1] <= 0 || sz[2] <= 0 || sz[0] >= (1ll << 30) || sz[1] >= (1ll << 30) || sz[2] >= (1ll << 30))
      return TRINIX_ERR_BAD_SHAPE;
    // no more rows than a grid's units, before their product is formed
    if (sz[0] * sz[1] > (1ll << 39) / sz[2]) return TRINIX_ERR_BAD_SHAPE;
    if (st[3] != 1 || ((uintptr_t)x[k] & 1) || ((uintptr_t)out[k] & 15)) return TRINIX_ERR_BAD_STRIDE;
    p.x[k] = (const uint16_t*)x[k];
    p.out[k] = (uint16_t*)out[k];
    p.sb[k] = st[0];
    p.ss[k] = st[1];
    p.sh[k] = st[2];
    p.S[k] = (int)sz[1];
    p.H[k] = (int)sz[2];
    p.units[k] = sz[0] * sz[1] * sz[2] * p.UPR;
    // a whole unit of a row is read at once: rows of whole, aligned units
    p.vec[k] = head_dim % 8 == 0 && ((uintptr_t)x[k] & 15) == 0 && st[0] % 8 == 0 && st[1] % 8 == 0 && st[2] % 8 == 0;
    most = p.units[k] > most ? p.units[k] : most;
  }
  const int64_t blocks = (most + 255) / 256;
  if (blocks >= (1ll << 31)) return TRINIX_ERR_BAD_SHAPE;
  const hipError_t err =
      launch_kernel(&pad_heads_kernel, dim3((unsigned)blocks, (unsigned)n), dim3(256), 0, (hipStream_t)stream, p);
  return err == hipSuccess ? TRINIX_OK : TRINIX_ERR_LAUNCH;
}
