// Host entry points of the attention library (C ABI).
//
// trinix_attn_fwd validates the arguments, picks a tile configuration for
// (dtype, head_dim, problem size), the feature flags (ALiBi, mask, dropout)
// and launches the bf16/fp16 MFMA kernel (attn_kernel16.h, instantiated per
// (dtype, head_dim) in attn16_*.hip) or the fp32 kernel (attn_fwd_f32.hip).
#include <atomic>
#include <cstring>

#include "attn_params.h"
#include "host_plan.h"

using namespace trinix;

extern "C" {

int trinix_abi_version(void) { return TRINIX_ATTN_ABI_VERSION; }

const char* trinix_status_string(int status) {
  switch (status) {
    case TRINIX_OK: return "ok";
    case TRINIX_ERR_NULL_POINTER: return "a required pointer is NULL";
    case TRINIX_ERR_BAD_DTYPE: return "unsupported dtype";
    case TRINIX_ERR_BAD_HEAD_DIM: return "unsupported head_dim (forward and backward kernels are built for 64, 128 and 256; split-KV for 64 and 128)";
    case TRINIX_ERR_BAD_SHAPE: return "invalid or inconsistent sizes";
    case TRINIX_ERR_BAD_STRIDE: return "unsupported strides or alignment (head_dim stride must be 1, 16-byte aligned rows, 16-bit K/V key-row stride below 2^22 elements)";
    case TRINIX_ERR_BAD_ARGUMENT: return "invalid argument";
    case TRINIX_ERR_NO_DEVICE: return "no gfx950 device available";
    case TRINIX_ERR_LAUNCH: return "kernel launch failed";
    case TRINIX_ERR_SCRATCH_TOO_SMALL: return "the call needs more scratch than the library's static buffer holds (TRINIX_SPLITKV_SCRATCH_BYTES); use the entry point that takes a workspace";
    default: return "unknown status";
  }
}

int trinix_attn_is_available(void) {
  // The architecture of each device is read once and kept (0 = not read yet,
  // 1 = not gfx950, 2 = gfx950); later calls cost one hipGetDevice.
  static std::atomic<int> arch_ok[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return 0;
  if (dev < 64) {
    const int known = arch_ok[dev].load(std::memory_order_relaxed);
    if (known) return known == 2 ? 1 : 0;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return 0;
  const int ok = strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 1 : 0;
  if (dev < 64) arch_ok[dev].store(ok ? 2 : 1, std::memory_order_relaxed);
  return ok;
}

int trinix_attn_tile_config(int64_t head_dim, int32_t dtype, trinix_tile_cfg* out) {
  if (!out) return TRINIX_ERR_NULL_POINTER;
  if (head_dim != 64 && head_dim != 128 && head_dim != 256) return TRINIX_ERR_BAD_HEAD_DIM;
  if (dtype == TRINIX_BF16 || dtype == TRINIX_F16) {
    const Cfg16 c = pick_cfg16(head_dim, 1 << 20, 1, 1 << 20, true, true);  // large-problem choice
    out->block_m = 32 * c.nw / c.ks;
    out->block_n = c.bn;
    out->block_d = (int32_t)head_dim;
    out->waves = c.nw;
    out->lds_bytes = (int32_t)(2 * 2 * c.ks * c.bn * head_dim * 2);
  } else if (dtype == TRINIX_F32) {
    out->block_m = 32 * kWavesF32;
    out->block_n = 32;
    out->block_d = (int32_t)head_dim;
    out->waves = kWavesF32;
    out->lds_bytes = (int32_t)(2 * 2 * 32 * head_dim * 4);
  } else {
    return TRINIX_ERR_BAD_DTYPE;
  }
  return TRINIX_OK;
}

int trinix_attn_fwd(const trinix_attn_fwd_args* a, void* stream) {
  return trinix_attn_fwd_narrow(a, a ? a->head_dim : 0, stream);
}

int trinix_attn_fwd_narrow(const trinix_attn_fwd_args* a, int64_t d_out, void* stream) {
  const int vrc = validate_fwd_args(a);
  if (vrc != TRINIX_OK) return vrc;
  const int nrc = check_narrow(a->dtype, a->head_dim, d_out);
  if (nrc != TRINIX_OK) return nrc;
  if (d_out < a->head_dim && (a->q_norm_weight || a->rope_cos)) return TRINIX_ERR_BAD_ARGUMENT;  // over head_dim columns

  FwdParams p{};  // value-initialised: fields a configuration does not use are zero
  p.q = (const uint16_t*)a->q;
  p.k = (const uint16_t*)a->k;
  p.v = (const uint16_t*)a->v;
  p.o = (uint16_t*)a->out;
  p.lse = a->lse;
  p.q_sb = a->q_stride[0]; p.q_ss = a->q_stride[1]; p.q_sh = a->q_stride[2];
  p.k_sb = a->k_stride[0]; p.k_ss = a->k_stride[1]; p.k_sh = a->k_stride[2];
  p.v_sb = a->v_stride[0]; p.v_ss = a->v_stride[1]; p.v_sh = a->v_stride[2];
  p.o_sb = a->out_stride[0]; p.o_ss = a->out_stride[1]; p.o_sh = a->out_stride[2];
  p.B = (int)a->batch;
  p.Sq = (int)a->seqlen_q;
  p.Sk = (int)a->seqlen_k;
  p.Hq = (int)a->nheads_q;
  p.Hkv = (int)a->nheads_kv;
  p.G = p.Hq / p.Hkv;
  const bool f32 = a->dtype == TRINIX_F32;
  FwdPlan plan;
  const int prc = plan_fwd(a, &plan);
  if (prc != TRINIX_OK) return prc;
  const Cfg16 cfg = plan.cfg;
  p.num_mblk = plan.num_mblk;
  for (int k = 0; k < plan.n_items; ++k) p.row_items[k] = plan.row_items[k];
  p.total_work = (int)plan.total_work;
  p.scale_log2 = a->softmax_scale * kLog2e;
  p.causal = a->causal ? 1 : 0;
  p.has_window = a->has_window ? 1 : 0;
  p.wl = clamp_window(a->window_left);
  p.wr = clamp_window(a->window_right);
  p.alibi = a->alibi_slopes;
  p.al_sb = a->alibi_stride[0];
  p.al_sh = a->alibi_stride[1];
  p.mask = a->mask;
  p.mask_dtype = a->mask_dtype;
  p.mk_sb = a->mask_stride[0]; p.mk_sh = a->mask_stride[1]; p.mk_si = a->mask_stride[2]; p.mk_sj = a->mask_stride[3];
  p.bmap = a->mask_blockmap;
  p.bm_sb = a->blockmap_stride[0];
  p.bm_sh = a->blockmap_stride[1];
  p.bm_cols = (int)((a->seqlen_k + 63) / 64);
  p.use_dropout = a->dropout_p > 0.f ? 1 : 0;
  {
    // dropped when the key's 16-bit Philox field < floor(p * 2^16)
    const double th = (double)a->dropout_p * 65536.0;
    p.drop_thresh = th >= 65535.0 ? 65535u : (uint32_t)th;
    p.drop_scale = a->dropout_p > 0.f ? 1.f / (1.f - a->dropout_p) : 1.f;
  }
  p.seed_lo = (uint32_t)a->dropout_seed;
  p.seed_hi = (uint32_t)(a->dropout_seed >> 32);
  p.off_lo = (uint32_t)a->dropout_offset;
  p.off_hi = (uint32_t)(a->dropout_offset >> 32);
  p.drop_state = a->dropout_state;
  p.rope_cos = (const uint16_t*)a->rope_cos;
  p.rope_sin = (const uint16_t*)a->rope_sin;
  p.rope_stride = a->rope_stride;
  p.qn_w = (const uint16_t*)a->q_norm_weight;
  p.qn_eps = a->q_norm_eps;
  p.qn_out = (uint16_t*)a->q_norm_out;
  p.keep_map = (uint32_t*)a->dropout_keep_map;
  p.d_out = (int)d_out;
  p.km_nbi = keep_map_nbi(a->seqlen_q);
  p.km_nbj = keep_map_nbj(a->seqlen_k);

  hipStream_t st = (hipStream_t)stream;
  hipError_t err;
  if (f32) {
    p.rows16 = rows_aligned16(a->k, a->k_stride) && rows_aligned16(a->v, a->v_stride);
    err = launch_attn_f32(p, (int)a->head_dim, plan.f32_ks, st);
  } else {
    const int feat = (p.alibi ? kFeatAlibi : 0) | (p.mask ? kFeatMask : 0) | (p.use_dropout ? kFeatDropout : 0) |
                     (p.qn_w ? kFeatQNorm : 0) | (p.use_dropout && p.keep_map ? kFeatKeepMap : 0);
    const bool bf = a->dtype == TRINIX_BF16;
    if (a->head_dim == 64)
      err = bf ? launch_attn16_bf16_d64(p, cfg, feat, st) : launch_attn16_f16_d64(p, cfg, feat, st);
    else if (a->head_dim == 128)
      err = bf ? launch_attn16_bf16_d128(p, cfg, feat, st) : launch_attn16_f16_d128(p, cfg, feat, st);
    else
      err = bf ? launch_attn16_bf16_d256(p, cfg, feat, st) : launch_attn16_f16_d256(p, cfg, feat, st);
    if (err == hipErrorNotSupported) return TRINIX_ERR_BAD_ARGUMENT;  // tile config not built
  }
  return err == hipSuccess ? TRINIX_OK : TRINIX_ERR_LAUNCH;
}

}  // extern "C"
