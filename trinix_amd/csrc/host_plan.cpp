// Host-only argument checks and launch planning (declared in host_plan.h):
// plain C++, no HIP.  Every function only reads its arguments and returns a
// status, a plan or a tile shape.
#include "host_plan.h"

#ifndef __host__  // plain C++: index_map.h's attributes are empty
#define __host__
#define __device__
#endif
#include "index_map.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>

namespace trinix {
namespace {

bool aligned16(const void* ptr) { return ((uintptr_t)ptr & 15) == 0; }

int check_tensor(const void* ptr, const int64_t st[4], int esize) {
  if (!ptr) return TRINIX_ERR_NULL_POINTER;
  if (st[3] != 1) return TRINIX_ERR_BAD_STRIDE;
  if (esize == 2) {
    // 16-byte vector loads of 8 consecutive head_dim elements per row
    if (!aligned16(ptr)) return TRINIX_ERR_BAD_STRIDE;
    for (int a = 0; a < 3; ++a)
      if (st[a] % 8 != 0) return TRINIX_ERR_BAD_STRIDE;
  } else if (((uintptr_t)ptr & 3) != 0) {
    return TRINIX_ERR_BAD_STRIDE;
  }
  return TRINIX_OK;
}

// fp32 BSHD tensor: head_dim stride 1, 4-byte aligned, any other stride (the
// kernels copy rows 16 bytes a lane where rows_aligned16 allows, else 4).
int check32(const void* ptr, const int64_t st[4]) {
  if (!ptr) return TRINIX_ERR_NULL_POINTER;
  if (st[3] != 1 || ((uintptr_t)ptr & 3) != 0) return TRINIX_ERR_BAD_STRIDE;
  return TRINIX_OK;
}

// 16-bit BSHD tensor: head_dim stride 1, 16-byte aligned rows, and a row
// stride the 32-bit in-tile offsets can address (tiles of up to 128 rows).
int check16(const void* ptr, const int64_t st[4]) {
  if (!ptr) return TRINIX_ERR_NULL_POINTER;
  if (st[3] != 1 || !aligned16(ptr)) return TRINIX_ERR_BAD_STRIDE;
  for (int a = 0; a < 3; ++a)
    if (st[a] % 8 != 0) return TRINIX_ERR_BAD_STRIDE;
  if (st[1] < 0 || st[1] >= kMaxKvRowStride) return TRINIX_ERR_BAD_STRIDE;
  return TRINIX_OK;
}

}  // namespace

// Tile configuration of the 16-bit kernel: 4 wavefronts x 32 query rows,
// 64-key tiles, 2 wavefronts per SIMD (1 for head_dim 256).  A small grid at
// head_dim 64 -- no more 128-row workgroups than CUs -- splits each 32-row
// group's keys between two wavefronts (ks = 2, 64 rows per workgroup): twice
// the workgroups, half the longest chain of tiles, at twice the K/V copies
// per flop.  Measured at head_dim 64, bf16: 128 workgroups at S = 4096..16384
// +50..62%, 64 workgroups at S = 1024 +2%, 384 workgroups (S = 1024) -3%.
// Head_dim 128 without a mask or dropout takes 8 wavefronts x 32 rows and
// 128-key tiles (one workgroup of 256 rows per CU, 128 KiB of LDS): half the
// barriers and tile bookkeeping per flop, once the grid holds enough 256-row
// workgroups -- 512 with causal / window bands (whose rows differ in length),
// 256 without.  Measured at bf16, graph-timed kernel: causal 512 workgroups
// +8%, 1024 +1.5..3% (C3), 2048 +2.7%, C4 +2..2.4%; full rows 256 workgroups
// +8%; below those counts it loses (causal 256 workgroups -9%, 128 -20%).
// TRINIX_ATTN_CFG="nw,occ,bn[,ks]" overrides the choice (tuning only; a
// configuration that is not built is rejected with TRINIX_ERR_BAD_ARGUMENT).
constexpr int64_t kSmallGrid = 256;  // CUs of an MI355X
// Enough 256-row workgroups for the wide shape: 512 with a causal / window
// band, 256 without (batch * hq * row blocks, without overflow: each factor
// < 2^31 here, and the product is formed only below 2^9 * 2^22).
static bool wide_grid(int64_t batch, int64_t hq, int64_t sq, bool banded) {
  const int64_t need = banded ? 2 * kSmallGrid : kSmallGrid;
  return batch * hq >= need || batch * hq * ((sq + 255) / 256) >= need;
}
// The key split of head_dim 128 and 256 (plain features): 64-row workgroups
// whose wavefront pairs take alternate 32-key tiles, where 128-row workgroups
// leave CUs idle or one wavefront per SIMD, and the longest row block's
// `chain` of 64-key tiles is worth halving against the merge.  Head_dim 128
// runs two workgroups per CU (64 KiB of LDS), head_dim 256 one.  Measured, bf16,
// graph-timed kernel, speedup by the split (grids of bh x row blocks):
//   up to 128 workgroups, D=128: full rows chain 6 1.10..1.13, 16 1.18, 48 1.24;
//     causal chain 8 1.09, 10 1.13, 20 1.19; D=256 48 x 11 31.3 | 27.0 us, 128 x 32
//     76.7 | 60.0; it loses at chain 2 and 3 (7.7 | 8.0, 8.4 | 8.8 us) and at D=256
//     above (192 x 8 27.8 | 31.8, 192 x 32 75.2 | 81.5)
//   129..256, D=128, full rows (and windows, whose rows are even too): up to 224
//     workgroups chain 6..10 0.96..0.98, 12 0.99..1.00, 14 1.00..1.01, 20 1.02..1.05,
//     48 1.03..1.12; 240 0.97..1.02 and 256 0.96..1.01 at any chain
//   129..256, D=128, causal: with the head groups dealt evenly to the XCDs, and so
//     dispatched longest rows first (fwd_item), chain 10 1.05, 16 1.09, 32 1.07;
//     otherwise 10 0.96..1.02, 11 0.91..0.94, 12 0.96, 16 0.98..1.01, 18
//     1.01..1.09, 32 1.07
//   beyond: 384 x 16 27.9 | 30.2 us, 512 x 32 49.9 | 52.0
static bool key_split(const trinix_attn_fwd_args* a) {
  const int64_t D = a->head_dim, bh = a->batch * a->nheads_q;
  if (D < 128 || bh > kSmallGrid) return false;
  // keys the longest 128-row block sees, in 64-key tiles
  int64_t keys = a->causal ? std::min(a->seqlen_q, a->seqlen_k) : a->seqlen_k;
  if (a->has_window) {
    const int64_t right = a->causal ? 0 : std::max<int64_t>(0, clamp_window(a->window_right));
    keys = std::min(keys, std::max<int64_t>(0, clamp_window(a->window_left)) + right + 128);
  }
  const int64_t chain = (keys + 63) / 64, wgs = bh * ((a->seqlen_q + 127) / 128);
  if (wgs <= kSmallGrid / 2) return chain >= 4;
  if (D != 128 || wgs > kSmallGrid) return false;
  if (a->causal && !a->has_window) return chain >= (a->batch * a->nheads_kv % kXcds == 0 ? 10 : 18);
  return chain >= 14 && wgs <= kSmallGrid * 7 / 8;
}
Cfg16 pick_cfg16(int64_t head_dim, int64_t batch, int64_t hq, int64_t sq, bool banded, bool plain,
                 bool split_ok, bool split_keys) {
  Cfg16 c{4, head_dim == 256 ? 1 : 2, 64, 1};
  // batch * hq * row blocks, without overflow (each factor < 2^31 here)
  if (head_dim == 64 && batch * hq <= kSmallGrid && batch * hq * ((sq + 127) / 128) <= kSmallGrid) c.ks = 2;
  else if (head_dim == 64 && split_ok && batch * hq <= 2 * kSmallGrid &&
           batch * hq * ((sq + 127) / 128) <= 2 * kSmallGrid)
    c.ks = 0;
  // the wide shape where it applies: 256 (batch, q-head) pairs of at most 128
  // full rows, 2048 keys 48.3 us wide, 55.1 with the key split
  if (head_dim == 128 && plain && wide_grid(batch, hq, sq, banded)) c = Cfg16{8, 2, 128, 1};
  else if (split_keys) c = Cfg16{4, c.occ, 32, 2};
  if (const char* env = getenv("TRINIX_ATTN_CFG")) {
    int nw = 0, occ = 0, bn = 0, ks = 1;
    // ks 1 or 2: wavefronts per 32-row group; 0: the per-item split
    if (sscanf(env, "%d,%d,%d,%d", &nw, &occ, &bn, &ks) >= 3 && nw > 0 && ks >= 0 && ks <= 2 &&
        (ks == 0 || nw % ks == 0))
      c = Cfg16{nw, occ, bn, ks};
  }
  return c;
}

// Per-item key split for causal grids of up to two rounds of 128-row
// workgroups at head_dim 64 (C2: 384): the longest row blocks' chains of
// tiles set the kernel time there, so the longest blocks run as two 64-row
// items with two wavefronts per 32-row group (half the chain each), the
// others as one item.  Blocks are split longest first while the grid stays
// within one round of resident workgroups (two per CU: 2 * 256 for all
// (batch, q-head) pairs), since a workgroup of a second round pays its
// start-up and epilogue again after the first round.
int plan_split_rows(int64_t sq, int64_t sk, int64_t heads, int rows, int bn, uint8_t* items, int max) {
  const int64_t nb = (sq + rows - 1) / rows;
  if (nb <= 0 || nb > 63 || heads <= 0) return 0;  // row block in 6 bits
  auto tiles = [&](int64_t rb) {
    const int64_t keys = std::min(sk, (rb + 1) * rows);  // causal: row i sees keys j <= i
    return (keys + bn - 1) / bn;
  };
  const int64_t max_t = tiles(nb - 1);
  const int64_t budget = std::min<int64_t>(max, std::max<int64_t>(nb, 2 * kSmallGrid / heads));
  struct Item { int64_t chain; int rb, split, half; };
  Item list[2 * 64];
  int n = 0;
  int64_t count = nb;  // items so far: one per block, one more per split block
  for (int64_t rb = nb - 1; rb >= 0; --rb) {
    const int64_t t = tiles(rb);
    if (2 * t > max_t + 1 && count + 1 <= budget) {
      ++count;
      for (int h = 0; h < 2; ++h) list[n++] = Item{(t + 1) / 2, (int)rb, 1, h};
    } else {
      list[n++] = Item{t, (int)rb, 0, 0};
    }
  }
  if (n > max) return 0;
  std::stable_sort(list, list + n, [](const Item& a, const Item& b) { return a.chain > b.chain; });
  for (int k = 0; k < n; ++k) items[k] = (uint8_t)((list[k].rb << 2) | (list[k].split << 1) | list[k].half);
  return n;
}

// The dQ backward kernel takes the same wide shape (8 wavefronts x 32 rows,
// 128-key tiles) under the same rule, at head_dim 128 without a mask
// (dropout included).  Measured at C3 (bf16): forward + backward 2.297 ->
// 2.284 ms, dQ ~2% faster, gradients bit-identical.
// TRINIX_BWD_DQ_WIDE=0 / 1 overrides the grid rule (tuning and tests; the
// wide shape is still only taken where it is built).
bool pick_dq_wide(int64_t head_dim, int64_t batch, int64_t hq, int64_t sq, bool banded, bool masked) {
  if (head_dim != 128 || masked) return false;
  if (const char* env = getenv("TRINIX_BWD_DQ_WIDE")) {
    if (env[0] == '0') return false;
    if (env[0] == '1') return true;
  }
  return wide_grid(batch, hq, sq, banded);
}

// The kernels address a mask row with 32-bit element offsets (load_mask4):
// a key stride in [0, 2^31 / Sk).  A mask broadcast over keys has stride 0.
static bool mask_key_stride_ok(int64_t sj, int64_t sk) {
  return sj >= 0 && (sk <= 1 || sj <= ((1ll << 31) - 1) / (sk - 1));  // (sk - 1) * sj < 2^31, no overflow
}

// Every mask stride is a non-negative element count (0 = broadcast); the
// batch, head and row parts of an address are formed in 64 bits.  The dK/dV
// kernel reads the 32 rows of a query sub-tile at 32-bit offsets r * si from
// the sub-tile's first row (r < 32, and r <= Sq - 1).
static bool mask_strides_ok(const int64_t st[4], int64_t sq, int64_t sk) {
  if (st[0] < 0 || st[1] < 0 || st[2] < 0) return false;
  const int64_t rows = sq - 1 < 31 ? sq - 1 : 31;
  if (rows > 0 && st[2] > ((1ll << 31) - 1) / rows) return false;
  return mask_key_stride_ok(st[3], sk);
}

// A dropout keep map goes with dropout, the 16-bit kernels at head_dim 64
// or 128 (the MFMA backward that reads it), and a 16-byte aligned buffer.
static bool keep_map_ok(const void* map, float dropout_p, int32_t dtype, int64_t head_dim) {
  return dropout_p > 0.f && (dtype == TRINIX_BF16 || dtype == TRINIX_F16) && (head_dim == 64 || head_dim == 128) &&
         aligned16(map);
}

int validate_fwd_args(const trinix_attn_fwd_args* a) {
  if (!a) return TRINIX_ERR_NULL_POINTER;
  const int esize = a->dtype == TRINIX_F32 ? 4 : 2;
  if (a->dtype != TRINIX_F32 && a->dtype != TRINIX_F16 && a->dtype != TRINIX_BF16) return TRINIX_ERR_BAD_DTYPE;
  if (a->head_dim != 64 && a->head_dim != 128 && a->head_dim != 256) return TRINIX_ERR_BAD_HEAD_DIM;
  if (a->batch <= 0 || a->seqlen_q <= 0 || a->seqlen_k <= 0 || a->nheads_q <= 0 || a->nheads_kv <= 0)
    return TRINIX_ERR_BAD_SHAPE;
  if (a->nheads_q % a->nheads_kv != 0) return TRINIX_ERR_BAD_SHAPE;
  if (a->seqlen_q >= (1ll << 30) || a->seqlen_k >= (1ll << 30) || a->batch >= (1 << 20) || a->nheads_q >= (1 << 20))
    return TRINIX_ERR_BAD_SHAPE;
  int rc;
  if ((rc = check_tensor(a->q, a->q_stride, esize))) return rc;
  if ((rc = check_tensor(a->k, a->k_stride, esize))) return rc;
  if ((rc = check_tensor(a->v, a->v_stride, esize))) return rc;
  // 16-bit kernels address a K/V tile (up to 128 key rows) as one base plus
  // per-lane 32-bit byte offsets: the key-row stride must be in [0, 2^22).
  if (esize == 2 && (a->k_stride[1] < 0 || a->k_stride[1] >= kMaxKvRowStride || a->v_stride[1] < 0 ||
                     a->v_stride[1] >= kMaxKvRowStride))
    return TRINIX_ERR_BAD_STRIDE;
  if ((rc = check_tensor(a->out, a->out_stride, esize))) return rc;
  if (a->mask && a->mask_dtype != TRINIX_F32 && a->mask_dtype != TRINIX_F16 && a->mask_dtype != TRINIX_BF16 &&
      a->mask_dtype != TRINIX_U8)
    return TRINIX_ERR_BAD_DTYPE;
  if (a->mask_blockmap && !a->mask) return TRINIX_ERR_BAD_ARGUMENT;
  if (a->mask && !mask_strides_ok(a->mask_stride, a->seqlen_q, a->seqlen_k)) return TRINIX_ERR_BAD_STRIDE;
  if (!(a->dropout_p >= 0.f && a->dropout_p < 1.f)) return TRINIX_ERR_BAD_ARGUMENT;
  if (a->dropout_state && ((uintptr_t)a->dropout_state & 7)) return TRINIX_ERR_BAD_ARGUMENT;
  if ((a->rope_cos == nullptr) != (a->rope_sin == nullptr)) return TRINIX_ERR_NULL_POINTER;
  if (a->rope_cos && esize == 2 &&
      (!aligned16(a->rope_cos) || !aligned16(a->rope_sin) || a->rope_stride % 8 != 0))
    return TRINIX_ERR_BAD_STRIDE;
  if (a->q_norm_out && (!a->q_norm_weight || !aligned16(a->q_norm_out))) return TRINIX_ERR_BAD_ARGUMENT;
  if (a->dropout_keep_map && !keep_map_ok(a->dropout_keep_map, a->dropout_p, a->dtype, a->head_dim))
    return TRINIX_ERR_BAD_ARGUMENT;
  if (a->q_norm_weight) {
    if (esize != 2) return TRINIX_ERR_BAD_DTYPE;
    if (a->mask || a->dropout_p > 0.f) return TRINIX_ERR_BAD_ARGUMENT;
    if (!aligned16(a->q_norm_weight)) return TRINIX_ERR_BAD_STRIDE;
    if (!(a->q_norm_eps >= 0.f)) return TRINIX_ERR_BAD_ARGUMENT;
  }

  return TRINIX_OK;
}

int validate_bwd_args(const trinix_attn_bwd_args* a) {
  if (!a) return TRINIX_ERR_NULL_POINTER;
  if (a->dtype != TRINIX_F16 && a->dtype != TRINIX_BF16 && a->dtype != TRINIX_F32) return TRINIX_ERR_BAD_DTYPE;
  if (a->head_dim != 64 && a->head_dim != 128 && a->head_dim != 256) return TRINIX_ERR_BAD_HEAD_DIM;
  if (!(a->dropout_p >= 0.f && a->dropout_p < 1.f)) return TRINIX_ERR_BAD_ARGUMENT;
  if (a->dropout_state && ((uintptr_t)a->dropout_state & 7)) return TRINIX_ERR_BAD_ARGUMENT;
  if (a->dropout_keep_map && !keep_map_ok(a->dropout_keep_map, a->dropout_p, a->dtype, a->head_dim))
    return TRINIX_ERR_BAD_ARGUMENT;
  if (a->batch <= 0 || a->seqlen_q <= 0 || a->seqlen_k <= 0 || a->nheads_q <= 0 || a->nheads_kv <= 0 ||
      a->nheads_q % a->nheads_kv != 0)
    return TRINIX_ERR_BAD_SHAPE;
  if (a->seqlen_q >= (1ll << 30) || a->seqlen_k >= (1ll << 30) || a->batch >= (1 << 20) || a->nheads_q >= (1 << 20))
    return TRINIX_ERR_BAD_SHAPE;
  if (!a->lse || !a->delta) return TRINIX_ERR_NULL_POINTER;
  int rc;
  auto check = a->dtype == TRINIX_F32 ? check32 : check16;
  if ((rc = check(a->q, a->q_stride)) || (rc = check(a->k, a->k_stride)) || (rc = check(a->v, a->v_stride)) ||
      (rc = check(a->out, a->out_stride)) || (rc = check(a->dout, a->dout_stride)) ||
      (rc = check(a->dq, a->dq_stride)) || (rc = check(a->dk, a->dk_stride)) || (rc = check(a->dv, a->dv_stride)))
    return rc;
  if (a->mask && a->mask_dtype != TRINIX_F32 && a->mask_dtype != TRINIX_F16 && a->mask_dtype != TRINIX_BF16 &&
      a->mask_dtype != TRINIX_U8)
    return TRINIX_ERR_BAD_DTYPE;
  if (a->mask_blockmap && !a->mask) return TRINIX_ERR_BAD_ARGUMENT;
  if (a->mask && !mask_strides_ok(a->mask_stride, a->seqlen_q, a->seqlen_k)) return TRINIX_ERR_BAD_STRIDE;
  return TRINIX_OK;
}

int check_narrow(int32_t dtype, int64_t head_dim, int64_t d_out) {
  if (d_out == head_dim) return TRINIX_OK;
  const bool ok = (dtype == TRINIX_BF16 || dtype == TRINIX_F16) && (head_dim == 64 || head_dim == 128) && d_out > 0 &&
                  d_out < head_dim && d_out % 8 == 0;
  return ok ? TRINIX_OK : TRINIX_ERR_BAD_HEAD_DIM;
}

int64_t clamp_window(int64_t w) {
  const int64_t lim = 1ll << 30;
  return w < -lim ? -lim : (w > lim ? lim : w);
}

// Two wavefronts per 32 keys or rows (half the chain of tiles, twice the
// workgroups, but twice the tile copies per product and a merge through LDS)
// in the fp32 and head_dim 256 kernels; `wgs` workgroups of one wavefront per 32.
// Rows of even length: where halves of a workgroup, each 4..10% dearer, take
// fewer rounds of the CUs.  Measured, us, one | two (fp32 S=1024, the backward's
// other kernel at its best):
//   D=64 forward 96 workgroups 96 | 59, 384 158 | 132, 512 161 | 165, 768 230 | 237, 896
//     300 | 277, 1024 301 | 316; dK/dV + dQ 384 480 | 398, 512 488 | 505, 896 937 | 866,
//     4096 3678 | 3868
//   D=128 forward 128 162 | 97, 192 164 | 178, 384 317 | 268, 512 323 | 350; backward 192
//     495 | 526, 384 967 | 793, 512 983 | 1046
//   D=256 bf16 dK/dV (two workgroups a block) 128 147 | 125, 256 160 | 175, 384 228 | 220,
//     512 419 | 469; dQ 64 147 | 130, 128 160 | 143, 192 228 | 246
// Causal rows, whose blocks differ in length, longest first: up to `limit`.
//   D=64 forward 512 128 | 109, 896 170 | 163, 1024 184 | 182, 1536 259 | 260, 2048 333 |
//     343, 4096 647 | 682; dK/dV 512 424 | 389, 1024 728 | 717, 1536 987 | 1007, 4096 2464 |
//     2528; dQ 1024 728 | 634, 4096 2464 | 2319, 5120 3055 | 2859 (half the
//     diagonal's waste: at any count)
//   D=128 forward 256 163 | 107, 384 166 | 165, 512 192 | 201; dK/dV 384 597 | 592, 512 738 |
//     754; dQ 384 597 | 549, 1024 1374 | 1293, 1280 1666 | 1617
//   D=256 bf16 dK/dV 256 381 | 300, 512 285 | 316; dQ 256 285 | 266, 512 445 | 478; fp16 dQ
//     (two workgroups a block) 256 157 | 150, 512 325 | 350
//   and of at most 256 rows as even ones: dQ D=64 S=256 4096 894 | 944, D=128 512 266 | 285
static bool two_per_group(int64_t head_dim, bool even, int64_t wgs, int64_t limit) {
  if (!even) return wgs <= limit;
  const double dearer = head_dim == 64 ? 1.04 : head_dim == 128 ? 1.08 : 1.1;
  return dearer * (double)((2 * wgs + kSmallGrid - 1) / kSmallGrid) < 2.0 * (double)((wgs + kSmallGrid - 1) / kSmallGrid);
}
// Whether the blocks of a problem are of (nearly) one length.
static bool even_rows(int32_t causal, int32_t has_window, int64_t sq) { return !causal || has_window || sq <= 256; }

int plan_fwd(const trinix_attn_fwd_args* a, FwdPlan* pl) {
  const bool f32 = a->dtype == TRINIX_F32;
  const bool plain = !a->mask && !(a->dropout_p > 0.f);
  const bool split_ok = plain && a->causal && !a->has_window && !a->q_norm_weight;
  Cfg16 cfg = pick_cfg16(a->head_dim, a->batch, a->nheads_q, a->seqlen_q, a->causal || a->has_window, plain,
                         split_ok, plain && key_split(a));
  if (a->q_norm_weight && a->head_dim == 64) cfg.ks = 1;  // where the fused q RMSNorm is built without the key split
  pl->n_items = 0;
  pl->num_mblk = 0;
  pl->f32_ks = 1;
  if (f32 && a->head_dim <= 128) {
    pl->f32_ks = two_per_group(a->head_dim, even_rows(a->causal, a->has_window, a->seqlen_q),
                               a->batch * a->nheads_q * ((a->seqlen_q + 127) / 128), a->head_dim == 64 ? 1024 : 384)
                     ? 2 : 1;
    if (const char* env = getenv("TRINIX_F32_KS"))  // tuning and tests
      if (env[0] == '1' || env[0] == '2') pl->f32_ks = env[0] - '0';
  }
  if (cfg.ks == 0) {  // per-item key split: the item table, or no split
    const int n = split_ok ? plan_split_rows(a->seqlen_q, a->seqlen_k, a->batch * a->nheads_q, 32 * cfg.nw, cfg.bn,
                                             pl->row_items, kMaxRowItems) : 0;
    if (n > (a->seqlen_q + 32 * cfg.nw - 1) / (32 * cfg.nw)) {
      pl->num_mblk = n;
      pl->n_items = n;
    } else {
      cfg.ks = 1;  // no block split (or no plan): the plain shape, without the per-item decode
    }
  }
  if (f32 || cfg.ks != 0) {
    const int bm = f32 ? 32 * kWavesF32 / pl->f32_ks : 32 * cfg.nw / cfg.ks;
    pl->num_mblk = (int)((a->seqlen_q + bm - 1) / bm);
  }
  pl->cfg = cfg;
  pl->total_work = a->batch * a->nheads_q * pl->num_mblk;
  if (pl->total_work >= (1ll << 31)) return TRINIX_ERR_BAD_SHAPE;
  return TRINIX_OK;
}

// dK/dV of the 16-bit kernels in pieces: where whole key blocks leave the
// 256 CUs (one workgroup each) with a long chain and idle neighbours -- few
// (batch, KV head) pairs, a causal band, or a last round nearly empty -- the
// blocks' items are cut into pieces of at most T that fill one or two rounds.
// Costs are in items (64 query rows of one q-head; 1.7 us at D = 128, 1.0 at
// D = 64, two wavefronts per SIMD busy): the longest chain or the share of a
// CU, against T per round plus the partials' write and read (about 4 TB/s) and
// one more launch (7 us).  Taken when it saves a tenth (figures beside
// attn_bwd_dkdv, attn_bwd16.h: forward + backward 342 -> 214 us at B=2 S=2048
// 16/4 heads; pieces lose 3..30% where whole blocks fill the chip).
static void plan_bwd_pieces(const trinix_attn_bwd_args* a, BwdPlan* pl) {
  constexpr int BK = 128, BQ = 64;
  constexpr int64_t slots = kSmallGrid;
  const int D = (int)a->head_dim, G = (int)(a->nheads_q / a->nheads_kv), nk = pl->num_kblk;
  const int64_t groups = a->batch * a->nheads_kv;
  if (nk > kMaxSplitKblk || groups * nk > 4 * slots) return;
  int dlo, dhi, items[kMaxSplitKblk], longest = 0;
  band_offsets(a->causal != 0, a->has_window != 0, clamp_window(a->window_left), clamp_window(a->window_right), dlo, dhi);
  int64_t total = 0;
  for (int k = 0; k < nk; ++k) {
    items[k] = bwd_kv_items(k, BK, G, (int)a->seqlen_q, (int)a->seqlen_k, dlo, dhi, BQ);
    longest = std::max(longest, items[k]);
    total += items[k];
  }
  if (longest < 2) return;
  const double item_us = D == 128 ? 1.7 : 1.0, piece_us = 2.0 * BK * D * 2 * 4 / 4e6;
  const double share = (double)total * groups / slots;
  // nearly equal blocks run in rounds; unequal ones, longest first, pack well
  double whole = std::max((double)longest, 1.1 * share);
  if (longest * (double)nk <= 1.15 * total) whole = (double)longest * ((groups * nk + slots - 1) / slots);
  double best = 0.9 * whole;
  for (int rounds = 1; rounds <= 2; ++rounds) {
    int T = std::max(1, (int)(share / rounds));
    for (; T < longest; T += std::max(1, T / 16)) {
      int64_t pieces = 0, partial = 0;
      for (int k = 0; k < nk; ++k) {
        const int np = bwd_pieces(items[k], T);
        pieces += np;
        partial += np > 1 ? np : 0;
      }
      if (pieces * groups > slots * rounds) continue;
      const double cost = (double)T * rounds + (7.0 + partial * groups * piece_us) / item_us;
      if (cost < best) {
        best = cost;
        pl->kv_T = T;
        pl->kv_P = (int)pieces;
      }
      break;
    }
  }
  if (pl->kv_T) pl->ws_bytes = groups * pl->kv_P * 2 * BK * (int64_t)D * 4;
}

// Workgroups of a launch of `blocks` per (batch, head), or -1 where no grid
// holds them (2^31); batch, heads < 2^20, 0 < blocks < 2^32.
static int64_t grid_of(int64_t batch, int64_t heads, int64_t blocks) {
  const int64_t bh = batch * heads;
  return bh < (1ll << 31) && bh * blocks < (1ll << 31) ? bh * blocks : -1;
}

int plan_bwd(const trinix_attn_bwd_args* a, BwdPlan* pl, bool split) {
  const bool f32 = a->dtype == TRINIX_F32;
  const int64_t D = a->head_dim;
  pl->generic = f32 || D == 256;
  pl->dq_wide = !pl->generic && pick_dq_wide(D, a->batch, a->nheads_q, a->seqlen_q, a->causal || a->has_window,
                                             a->mask != nullptr);
  pl->dq_ks = pl->kv_ks = pl->dq_hs = pl->kv_hs = 1;
  // Every grid is bounded before a plan is chosen from its size.  The fp32 and
  // head_dim 256 calls take what blocks of 32 rows and keys, and 4 rows of the
  // delta pass, can cover; the others 128 keys, 128 or 256 rows, and the
  // 2048 / D rows of a delta workgroup.
  const int64_t bq = pl->generic ? 32 : (pl->dq_wide ? 256 : 128), bk0 = pl->generic ? 32 : 128;
  const int64_t bd = pl->generic ? 4 : 2048 / D;
  if (grid_of(a->batch, a->nheads_q, (a->seqlen_q + bq - 1) / bq) < 0 ||
      grid_of(a->batch, a->nheads_kv, (a->seqlen_k + bk0 - 1) / bk0) < 0 ||
      (a->batch * a->nheads_q * a->seqlen_q + bd - 1) / bd >= (1ll << 31))  // < 2^31 * 256 rows here
    return TRINIX_ERR_BAD_SHAPE;
  if (pl->generic) {
    if (D == 256) {  // column splits: the kernels' registers
      pl->kv_hs = f32 ? 4 : 2;
      pl->dq_hs = a->dtype == TRINIX_BF16 ? 1 : 2;
    }
    if (!(f32 && D == 256)) {  // (whose tiles fill the LDS)
      const bool even = even_rows(a->causal, a->has_window, a->seqlen_q);
      const int64_t kv = a->batch * a->nheads_kv * ((a->seqlen_k + 127) / 128) * pl->kv_hs;
      const int64_t dq = a->batch * a->nheads_q * ((a->seqlen_q + 127) / 128) * pl->dq_hs;
      pl->kv_ks = two_per_group(D, even, kv, D == 64 ? 1024 : 384) ? 2 : 1;
      pl->dq_ks = two_per_group(D, even, dq, D == 256 ? 384 : 1ll << 31) ? 2 : 1;
      if (const char* env = getenv("TRINIX_BWD_GENERIC")) {  // "dq_ks,kv_ks" (tuning and tests)
        int ks = 0, kks = 0;
        if (sscanf(env, "%d,%d", &ks, &kks) == 2 && (ks == 1 || ks == 2) && (kks == 1 || kks == 2)) {
          pl->dq_ks = ks;
          pl->kv_ks = kks;
        }
      }
    }
  }
  const int bm = pl->dq_wide ? 256 : 128 / pl->dq_ks, bk = 128 / pl->kv_ks;
  pl->num_kblk = (int)((a->seqlen_k + bk - 1) / bk);
  pl->num_mblk = (int)((a->seqlen_q + bm - 1) / bm);
  if (grid_of(a->batch, a->nheads_q, (int64_t)pl->num_mblk * pl->dq_hs) < 0 ||
      grid_of(a->batch, a->nheads_kv, (int64_t)pl->num_kblk * pl->kv_hs) < 0)
    return TRINIX_ERR_BAD_SHAPE;
  pl->kv_T = pl->kv_P = 0;
  pl->ws_bytes = 0;
  // items of a key block (query tiles of a group's q-heads) count in 31 bits
  const int64_t G = a->nheads_q / a->nheads_kv;
  const bool countable = G * ((a->seqlen_q + 63) / 64) < (1ll << 31);
  if (split && !pl->generic) {
    if (const char* env = getenv("TRINIX_BWD_PIECES")) {  // pieces of at most this many items, 0: whole (tuning and tests)
      const int T = atoi(env);
      if (T > 0 && pl->num_kblk <= kMaxSplitKblk && countable) {
        int dlo, dhi;
        band_offsets(a->causal != 0, a->has_window != 0, clamp_window(a->window_left), clamp_window(a->window_right), dlo,
                     dhi);
        int64_t pieces = 0;
        for (int k = 0; k < pl->num_kblk; ++k)
          pieces += bwd_pieces(bwd_kv_items(k, 128, (int)G, (int)a->seqlen_q, (int)a->seqlen_k, dlo, dhi, 64), T);
        if (grid_of(a->batch, a->nheads_kv, pieces) >= 0 && grid_of(a->batch, a->nheads_kv, 16 * pl->num_kblk) >= 0) {
          pl->kv_T = T;
          pl->kv_P = (int)pieces;
          pl->ws_bytes = a->batch * a->nheads_kv * pieces * 2 * 128 * D * 4;
        }
      }
    } else if (countable) {
      plan_bwd_pieces(a, pl);
    }
  }
  return TRINIX_OK;
}

bool make_split_plan(const trinix_attn_fwd_args* a, SplitPlan* pl) {
  if (a->dtype != TRINIX_BF16 && a->dtype != TRINIX_F16) return false;
  if (a->dropout_p > 0.f || a->rope_cos || a->q_norm_weight) return false;
  if (a->seqlen_q > kDecodeMaxSq) return false;
  if (a->head_dim != 64 && a->head_dim != 128) return false;
  const int64_t Sq = a->seqlen_q, Sk = a->seqlen_k;
  const int64_t G = a->nheads_q / a->nheads_kv;
  const int64_t M = G * Sq;
  const int64_t RG = (M + 15) / 16;
  const int64_t wl = clamp_window(a->window_left), wr = clamp_window(a->window_right);
  // Keys some row i in [0, Sq) may see: lo(i) = max(0, i - wl) is smallest at
  // i = 0, hi(i) = min(Sk - 1, i (causal), i + wr (window)) largest at Sq - 1.
  int64_t klo = a->has_window ? -wl : 0;
  klo = klo < 0 ? 0 : (klo > Sk ? Sk : klo);
  int64_t hi = Sk - 1;
  if (a->causal) hi = hi < Sq - 1 ? hi : Sq - 1;
  if (a->has_window) hi = hi < Sq - 1 + wr ? hi : Sq - 1 + wr;
  int64_t khi = hi + 1;
  khi = khi < 0 ? 0 : (khi > Sk ? Sk : khi);
  if (khi <= klo) return false;  // no visible key: every row is NaN, leave it to trinix_attn_fwd
  const int64_t span = khi - klo;
  const int64_t items = a->batch * a->nheads_kv * RG;
  int64_t target = kDecodeTargetWgs, min_chunk = kDecodeMinChunk;
  if (const char* env = getenv("TRINIX_SPLITKV_CFG")) {  // "target_wgs,min_chunk" (tuning only)
    long long t = 0, c = 0;
    if (sscanf(env, "%lld,%lld", &t, &c) == 2 && t > 0 && c >= 64) {
      target = t;
      min_chunk = c;
    }
  }
  const int64_t max_splits = (span + min_chunk - 1) / min_chunk;
  int64_t n = (target + items - 1) / items;
  n = n < 1 ? 1 : (n > max_splits ? max_splits : n);
  int64_t chunk = (span + n - 1) / n;
  chunk = (chunk + 63) / 64 * 64;
  n = (span + chunk - 1) / chunk;
  if (items * n >= (1ll << 31)) return false;
  pl->n_splits = (int)n;
  pl->chunk = (int)chunk;
  pl->klo = (int)klo;
  pl->khi = (int)khi;
  pl->M = (int)M;
  pl->RG = (int)RG;
  pl->ws_bytes = n > 1 ? a->batch * a->nheads_kv * M * n * (a->head_dim + 1) * 4 : 0;
  return true;
}

// The plan bounds the chunks (and fixes the workspace) at four workgroups per
// CU; a launch runs the count among the planned one and one to four workgroups
// per CU that costs least.  A decode step is bound by HBM, and one workgroup on
// every CU already saturates it: more only add chunks to merge and spread the
// reads.  Cost, in us: the read at 5.5 TB/s, times how unevenly whole workgroups
// fall on the CUs (a workgroup alone on its CU in a partial grid reads up to
// 1 / 0.82 of its share), 6% for more than one per CU and 8% off for
// non-temporal loads; 2 for each round after the first; for the merge 5, its
// rows and the partial sums.  Over 212 grids (3 to 128 sequences, 300 to 8192
// keys, 8 KV heads of D=128, caches cold, graph-timed) the count it takes is
// within 1% of the best one in the mean and 13% at worst, and on the 146 of them
// that were timed with the planned count 10% faster than that, at worst 5%
// slower (B=56 S=3000 136.5 | 130.1).  Head_dim 64 (half the bytes per load)
// follows no such rule: one workgroup per CU where that fills them, the plan's
// count otherwise (B=12 S=3000 16 heads: 1152 workgroups 34.8 us, 768 37.5, 192
// 39.6).
// Measured, bf16, 8 KV heads of D=128 unless noted, us as planned | run: B=16
// S=8192 113.7 | 99.9 (256 workgroups, non-temporal), B=4 S=8000 36.4 | 30.6,
// B=24 S=4000 84.6 | 78.2 (192), B=64 S=2000 104.6 | 98.2 (512, unsplit), B=16
// S=1000 23.4 | 19.1, B=16 S=3000 16 heads of D=64 47.4 | 37.9; short rows, unsplit |
// two chunks: B=48 S=300 21.1 | 25.4, S=500 27.8 | 28.9, S=1000 50.0 | 47.4; B=12
// S=1000 two | eight chunks 17.1 | 20.0.
// Non-temporal K/V loads pay where the workgroups fill the CUs evenly (B=16
// S=8192 107.8 | 99.9 us, B=32 S=8000 193 | 189) and lose where CUs idle in the
// last round (192 workgroups 78.2 | 88.3, 384 90.9 | 94.2, 128 9.8 | 10.1) and at
// head_dim 64 (B=16 S=3000 16 heads 39.6 | 44.2); with several row groups the
// K/V are read again, from L2.  In several rounds of short rows they lose too
// (300 keys, 512, 768 and 1024 workgroups 23.1 | 23.5, 31.6 | 32.7, 39.8 | 42.7;
// 500 keys 55.1 | 55.3, 1000 78.1 | 77.6), in one round they gain (128 items of 300
// keys, two chunks 13.1 | 12.6, 256 13.7 | 13.3).
void decode_run_plan(const trinix_attn_fwd_args* a, SplitPlan* pl, bool* streamed) {
  const int64_t items = a->batch * a->nheads_kv * pl->RG, span = (int64_t)pl->khi - pl->klo;
  auto rounds = [&](int64_t n) { return (items * n + kSmallGrid - 1) / kSmallGrid; };
  auto uneven = [&](int64_t n) { return (double)(rounds(n) * kSmallGrid) / (double)(items * n); };
  auto run = [&](int64_t n, int64_t* chunk) {  // chunks of whole 64 keys, as planned
    *chunk = ((span + n - 1) / n + 63) / 64 * 64;
    return (span + *chunk - 1) / *chunk;
  };
  auto non_temporal = [&](int64_t n) {
    return a->head_dim == 128 && pl->RG == 1 && uneven(n) <= 1.07 && (rounds(n) == 1 || span >= 512);
  };
  auto cost = [&](int64_t n) {
    const double read_us = 4.0 * items * span * a->head_dim / 5.5e6, rows = (double)(a->batch * a->nheads_kv) * pl->M;
    const double share = rounds(n) > 1 ? 1.06 * uneven(n) : std::max(1.0, 0.82 * uneven(n));
    return read_us * share * (non_temporal(n) ? 0.92 : 1.0) + 2.0 * (rounds(n) - 1) +
           (n > 1 ? 5.0 + rows / 400 + rows * n / 3000 : 0.0);
  };
  // several row groups and long rows in more than one round run as planned (16
  // sequences of 16 queries, S=8192 325 us in two chunks | 342 unsplit)
  const bool as_planned = pl->RG > 1 && items > kSmallGrid && span > 3000;
  if (pl->n_splits > 1 && !as_planned && !getenv("TRINIX_SPLITKV_CFG")) {
    int64_t best_n = pl->n_splits, chunk;
    for (int k = 1; k <= 4; ++k) {
      int64_t n = std::min<int64_t>(pl->n_splits, kSmallGrid * k / items);
      if (n < 1) continue;
      n = run(n, &chunk);
      if (a->head_dim == 64) {
        if (k == 1 && uneven(n) <= 1.07) best_n = n;
        break;
      }
      if (cost(n) < cost(best_n)) best_n = n;
    }
    pl->n_splits = (int)run(best_n, &chunk);
    pl->chunk = (int)chunk;
  }
  *streamed = non_temporal(pl->n_splits);
}

}  // namespace trinix
