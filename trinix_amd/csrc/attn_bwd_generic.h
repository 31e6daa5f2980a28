// Backward kernels of fp32 (head_dim 64, 128 and 256) and of bf16 / fp16 at
// head_dim 256 (attn_ops.h).  P and dZ enter their products at fp32 precision in
// fp32, as two 16-bit terms in the others: 16 significant bits in bf16, about 21
// in fp16 (P with a quantum of 2^-35), where one term alone (attn_bwd16.h) has 8 or
// 11 and an fp32 product 24.  Over 28 calls at head_dim 256 (S = 225..2048, both types) the
// error of dq, dk and dv against 64 bits is 0.996 to 1.001 of that with 24-bit
// coefficients (0.9992 in the mean): the output's own rounding, 1.7e-3 to 1.9e-3 in
// bf16 and 2.1e-4 to 2.4e-4 in fp16.
// No counterpart in the reference (its Triton attention returns a detached
// output, trinix/kernels/attention_kernel.py:497-517); the gradients are
// those of the eager path (trinix/layers/attention/base.py:347-400):
//   P = exp(z - lse), Pd = P * keep / (1 - p), z = scale*q k^T + bias + mask,
//   dV = Pd^T dO,  dZ = P * (keep * (dO V^T) / (1 - p) - delta),
//   dK = scale * dZ^T Q,  dQ = scale * dZ K,  delta = rowsum(dO * O).
// As in attn_bwd16.h, delta comes multiplied by 1 - p and the 1 / (1 - p) of
// Pd and dZ is applied once per output element.
//
//   bwd_dkdv_generic  a workgroup of 4 wavefronts per (batch, KV head, 128
//                     keys); a wavefront owns 32 keys (K and V rows in
//                     registers) and walks the 32-row tiles of Q and dO of
//                     every q-head of the group: S, dP, P and dZ in
//                     registers, dV += Pd^T dO, dK += dZ^T Q;
//   bwd_dq_generic    a workgroup of 4 wavefronts per (batch, q-head) and
//                     128 query rows (Q and dO rows in registers), over
//                     32-key tiles of K and V: dQ += dZ K.  With KS = 2 it
//                     owns 64 rows, two wavefronts per 32 rows taking
//                     alternate tiles, summed through LDS at the end.
// KS = 2 in dK/dV likewise: 64 keys, two wavefronts per 32 keys taking
// alternate tiles.  Tiles go global -> LDS asynchronously into two slots, one
// barrier per step; no atomics (deterministic).
//
// What bounds them.  fp32: the matrix cores, a 32x32 block at D = 64 taking
// 128 (dK/dV) and 96 (dQ) v_mfma_f32_32x32x2f32 of 64 cycles; these share the
// vector ALU's cycles (SQ_VALU_MFMA_COEXEC_CYCLES is 0), so what is left to
// gain is the ALU work beside them (3 instructions per MFMA).  Head_dim 256:
// one wavefront per SIMD, whose ALU work and operand reads are mostly exposed
// (MFMA busy 25-30%); dK and dV of 32 keys with their K and V rows leave no
// room for a second, so their columns go over HS workgroups.
// Measured, forward + backward: fp32 B=4 S=1024 12 heads D=64 causal 2077 us
// with one wavefront per 32x32 tile and four barriers (dK/dV 949, dQ 837), now
// 344 (141, 136); bf16 B=2 S=2048 8/4 heads D=256 causal 5900 us on fp32
// products (3402, 2304), now 334 (195, 97).
// ALiBi and mask are wave-uniform branches; dropout is a template flag.
#pragma once
#include "attn_bwd16.h"
#include "attn_ops.h"

namespace trinix {

// Sums of a pair of wavefronts (kp = 0, 1 of group `grp`, two groups): the
// second hands its accumulators, times f, to the first through LDS bytes
// of shared memory, which then holds acc * f of both.  Every wavefront of the workgroup
// calls it.
template <int LDS, int NDB>
__device__ inline void merge_pair(f32x16_t (&acc)[NDB], float f, float* lds, int grp, int kp, int lane) {
  constexpr int HB = NDB > 4 ? 4 : NDB;  // blocks per exchange: 4 KiB each and group
  static_assert(NDB % HB == 0 && 2 * HB * 4096 <= LDS, "exchange");
  float* x = lds + grp * HB * 16 * 64 + lane;
#pragma unroll
  for (int h = 0; h < NDB; h += HB) {
    __syncthreads();
    if (kp == 1) {
#pragma unroll
      for (int db = 0; db < HB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) x[(db * 16 + v) * 64] = acc[h + db][v] * f;
    }
    __syncthreads();
    if (kp == 0) {
#pragma unroll
      for (int db = 0; db < HB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[h + db][v] = __builtin_fmaf(acc[h + db][v], f, x[(db * 16 + v) * 64]);
    }
  }
}

template <class O, int OCC, int HS, int KS, bool DROP>
__global__ __launch_bounds__(256, OCC) void bwd_dkdv_generic(const BwdParams p) {
  using Store = typename O::Store;
  constexpr int NW = 4, BK = NW * 32 / KS, D = O::kD, DB = O::DB / HS;
  constexpr int TILE = kTileRows * D * (int)sizeof(Store);
  // tiles of a step (KS items), two slots
  __shared__ __attribute__((aligned(1024))) char lds_q[2][KS * TILE];
  __shared__ __attribute__((aligned(1024))) char lds_o[2][KS * TILE];
  __shared__ __attribute__((aligned(128))) float lds_l[2][KS * kTileRows];
  __shared__ __attribute__((aligned(128))) float lds_d[2][KS * kTileRows];

  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // HS workgroups share a key block, each summing D / HS of the columns
  const KvItem wi = bwd_kv_item((int)blockIdx.x / HS, p.B, p.Hkv, p.num_kblk, p.causal != 0);  // (index_map.h)
  const int hkv = wi.hkv, b = wi.b, kb0 = wi.kblk * BK, db0 = ((int)blockIdx.x % HS) * DB;
  const int kgrp = wave / KS, kp = wave % KS;
  const int j0 = kb0 + kgrp * 32, j = j0 + (lane & 31), jc = min(j, p.Sk - 1);
  const Band band(p);
  const bool wide = p.rows16 != 0;
  DropKey dkey{};
  if constexpr (DROP) dkey = drop_key(p);

  int qt_lo, qt_hi;
  bwd_query_tiles(kb0, BK, p.Sq, p.Sk, band.dlo, band.dhi, kTileRows, qt_lo, qt_hi);
  const int nqt = qt_hi - qt_lo;
  const int n_items = nqt > 0 ? p.G * nqt : 0;  // item = (q-head of the group, query tile)

  const O ops(lane, db0);
  const typename O::Frag kf = O::load_frag((const Store*)p.k + b * p.k_sb + hkv * p.k_sh + (int64_t)jc * p.k_ss, g);
  const typename O::Frag vf = O::load_frag((const Store*)p.v + b * p.v_sb + hkv * p.v_sh + (int64_t)jc * p.v_ss, g);
  f32x16_t dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dk[db] = dv[db] = (f32x16_t){};
  ZScale<O> zs;

  // lse (times log2 e) and delta of the next item's rows, loaded with its
  // copies and written to LDS at the end of the step.  A row with no allowed
  // key has lse -inf and every score -inf: the finite floor keeps
  // exp2(score - lse2) at 0 instead of exp2(-inf + inf) = NaN.
  const TileCopy<O, NW> copy_q(p.q_ss, wave, lane), copy_o(p.do_ss, wave, lane);
  float lse_next = 0.f, del_next = 0.f;
  auto load_step = [&](int it, int slot) __attribute__((always_inline)) {  // items it .. it + KS - 1
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      if (it + u >= n_items) break;
      const int hq = hkv * p.G + (it + u) / nqt, i0 = (qt_lo + (it + u) % nqt) * kTileRows;
      copy_q((const Store*)p.q + b * p.q_sb + hq * p.q_sh, i0, p.Sq, lds_q[slot] + u * TILE, wide);
      copy_o((const Store*)p.dout + b * p.do_sb + hq * p.do_sh, i0, p.Sq, lds_o[slot] + u * TILE, wide);
      if (tid / kTileRows == u) {
        const int64_t ro = ((int64_t)b * p.Hq + hq) * p.Sq + min(i0 + tid % kTileRows, p.Sq - 1);
        lse_next = p.lse[ro];
        del_next = p.delta[ro];
      }
    }
  };
  auto write_rows = [&](int slot) __attribute__((always_inline)) {
    if (tid < KS * kTileRows) {
      lds_l[slot][tid] = fmaxf(lse_next * kLog2e, -0.5f * FLT_MAX) - O::kPShift;
      lds_d[slot][tid] = del_next;
    }
  };

  auto block = [&](int it, int slot) __attribute__((always_inline)) {
    const int hq = hkv * p.G + it / nqt, i0 = (qt_lo + it % nqt) * kTileRows;
    const char *q_lds = lds_q[slot] + kp * TILE, *o_lds = lds_o[slot] + kp * TILE;
    const float *l_lds = &lds_l[slot][kp * kTileRows], *d_lds = &lds_d[slot][kp * kTileRows];
    const BlockCode code = block_code(p, band, b, hq, i0, j0);
    if (!code.live) return;
    // S and dV first, then dP and dK: one block's scores and one product's
    // operands live at a time
    const f32x16_t s = ops.scores(q_lds, kf);
    float x[16];
#pragma unroll
    for (int vq = 0; vq < 4; ++vq) {
      const f32x4_t l4 = *(const f32x4_t*)(l_lds + vq * 8 + g * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[vq * 4 + e] = __builtin_fmaf(s[vq * 4 + e], p.scale_log2, -l4[e]);
    }
    if (p.alibi) {
      const float slope_l2 = -p.alibi[b * p.al_sb + hq * p.al_sh] * kLog2e;
      const float fj = (float)(j - (i0 + g * 4));
#pragma unroll
      for (int v = 0; v < 16; ++v) x[v] = __builtin_fmaf(fabsf(fj - (float)((v >> 2) * 8 + (v & 3))), slope_l2, x[v]);
    }
    if (code.mask) {
      // the block's rows sit at 32-bit offsets r * mk_si from its first (r <
      // 32, host-bounded); rows past Sq read the last row and are masked below
      const int esz = p.mask_dtype == TRINIX_F32 ? 4 : (p.mask_dtype == TRINIX_U8 ? 1 : 2);
      const char* m0 = (const char*)p.mask +
                       (b * p.mk_sb + hq * p.mk_sh + (int64_t)jc * p.mk_sj + (int64_t)i0 * p.mk_si) * esz;
      const int rlast = min(31, p.Sq - 1 - i0);
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        float mv[4];
        load_mask4(m0, p.mask_dtype, vq * 8 + g * 4, p.mk_si, rlast, mv);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[vq * 4 + e] += mv[e] * kLog2e;
      }
    }
    if (!code.full) {
      // rows the lane's key may see, formed here (not held across the loop)
      int jo = j;
      asm volatile("" : "+v"(jo));
      const Span qspan = jo < p.Sk ? Span(max((int64_t)0, (int64_t)jo - band.dhi), min((int64_t)p.Sq - 1, (int64_t)jo - band.dlo))
                                   : Span(1, 0);
#pragma unroll
      for (int v = 0; v < 16; ++v) x[v] = qspan.ok(i0 + (v >> 2) * 8 + g * 4 + (v & 3)) ? x[v] : -INFINITY;
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) x[v] = __builtin_amdgcn_exp2f(x[v]);
    uint32_t km = 0;
    if constexpr (DROP) {
      km = keep_bits_of_key(dkey, b * p.Hq + hq, j, i0 + g * 4);
      float pd[16];
#pragma unroll
      for (int v = 0; v < 16; ++v) pd[v] = __uint_as_float(__float_as_uint(x[v]) & keep_word(km, v));
      ops.accum(dv, o_lds, pd);
    } else {
      ops.accum(dv, o_lds, x);
    }
    f32x16_t dp = ops.scores(o_lds, vf);
    if constexpr (DROP) {
#pragma unroll
      for (int v = 0; v < 16; ++v) dp[v] = __uint_as_float(__float_as_uint(dp[v]) & keep_word(km, v));
    }
#pragma unroll
    for (int vq = 0; vq < 4; ++vq) {
      const f32x4_t d4 = *(const f32x4_t*)(d_lds + vq * 8 + g * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[vq * 4 + e] *= dp[vq * 4 + e] - d4[e];
    }
    zs.apply(x, dk);
    ops.accum(dk, q_lds, x);
  };

  // A step computes items it .. it + KS - 1 (wavefront kp of a key group the
  // kp-th) from one slot while the next ones land in the other; the barrier
  // at its top is where its items have landed and every wavefront has left
  // the other slot.
  if (n_items > 0) {
    load_step(0, 0);
    write_rows(0);
  }
  auto step = [&](auto slot_c, int it) __attribute__((always_inline)) {
    constexpr int SL = decltype(slot_c)::value;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (it + KS < n_items) load_step(it + KS, 1 - SL);
    if (it + kp < n_items) block(it + kp, SL);
    if (it + KS < n_items) write_rows(1 - SL);
  };
  for (int it = 0; it < n_items; it += 2 * KS) {
    step(std::integral_constant<int, 0>{}, it);
    if (it + KS < n_items) step(std::integral_constant<int, 1>{}, it + KS);
  }

  const float ds = DROP ? p.drop_scale : 1.f;
  float fv = ds * exp2f(-O::kPShift), fk = p.scale * fv * zs.undo();
  if constexpr (KS == 2) {
    merge_pair<2 * KS * TILE>(dv, fv, (float*)&lds_q[0][0], kgrp, kp, lane);
    merge_pair<2 * KS * TILE>(dk, fk, (float*)&lds_q[0][0], kgrp, kp, lane);
    if (kp == 1) return;
    fv = fk = 1.f;
  }
  if (j < p.Sk) {
    Store* krow = (Store*)p.dk + b * p.dk_sb + hkv * p.dk_sh + (int64_t)j * p.dk_ss;
    Store* vrow = (Store*)p.dv + b * p.dv_sb + hkv * p.dv_sh + (int64_t)j * p.dv_ss;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        const int d0 = (db0 + db) * 32 + vq * 8 + g * 4;
        O::store4(vrow, d0, dv[db][vq * 4] * fv, dv[db][vq * 4 + 1] * fv, dv[db][vq * 4 + 2] * fv, dv[db][vq * 4 + 3] * fv);
        O::store4(krow, d0, dk[db][vq * 4] * fk, dk[db][vq * 4 + 1] * fk, dk[db][vq * 4 + 2] * fk, dk[db][vq * 4 + 3] * fk);
      }
  }
}

template <class O, int OCC, int HS, int KS, bool DROP>
__global__ __launch_bounds__(256, OCC) void bwd_dq_generic(const BwdParams p) {
  using Store = typename O::Store;
  constexpr int NW = 4, BM = NW * 32 / KS, D = O::kD, DB = O::DB / HS;
  constexpr int TILE = kTileRows * D * (int)sizeof(Store);
  // tiles of a step (KS of them), two slots
  __shared__ __attribute__((aligned(1024))) char lds_k[2][KS * TILE];
  __shared__ __attribute__((aligned(1024))) char lds_v[2][KS * TILE];

  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rgrp = wave / KS, kp = wave % KS;
  const DqItem wi = bwd_dq_item((int)blockIdx.x / HS, p.B, p.Hq, p.Hkv, p.G, p.num_mblk, p.causal != 0, BM);
  const int hkv = wi.hkv, b = wi.b, m0 = wi.m0, hq = hkv * p.G + wi.gq, db0 = ((int)blockIdx.x % HS) * DB;
  const int iw0 = m0 + rgrp * 32, i = iw0 + r, ic = min(i, p.Sq - 1);
  const Band band(p);
  const bool wide = p.rows16 != 0;
  DropKey dkey{};
  if constexpr (DROP) dkey = drop_key(p);

  const O ops(lane, db0);
  const typename O::Frag qf = O::load_frag((const Store*)p.q + b * p.q_sb + hq * p.q_sh + (int64_t)ic * p.q_ss, g);
  const typename O::Frag of = O::load_frag((const Store*)p.dout + b * p.do_sb + hq * p.do_sh + (int64_t)ic * p.do_ss, g);
  const int64_t vo = ((int64_t)b * p.Hq + hq) * p.Sq + ic;
  // (finite floor: see bwd_dkdv_generic)
  const float lse2 = fmaxf(p.lse[vo] * kLog2e, -0.5f * FLT_MAX), dlt = p.delta[vo];
  const float slope_l2 = p.alibi ? -p.alibi[b * p.al_sb + hq * p.al_sh] * kLog2e : 0.f;
  const int esz = p.mask_dtype == TRINIX_F32 ? 4 : (p.mask_dtype == TRINIX_U8 ? 1 : 2);
  const char* mrow = p.mask ? (const char*)p.mask + (b * p.mk_sb + hq * p.mk_sh + (int64_t)ic * p.mk_si) * esz : nullptr;
  f32x16_t acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = (f32x16_t){};
  ZScale<O> zs;

  int t_lo, t_hi;
  bwd_key_tiles(m0, BM, p.Sq, p.Sk, band.dlo, band.dhi, kTileRows, t_lo, t_hi);
  const Store* kbase = (const Store*)p.k + b * p.k_sb + hkv * p.k_sh;
  const Store* vbase = (const Store*)p.v + b * p.v_sb + hkv * p.v_sh;
  const TileCopy<O, NW> copy_k(p.k_ss, wave, lane), copy_v(p.v_ss, wave, lane);
  auto load = [&](int t, int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < KS; ++u)
      if (t + u < t_hi) {
        copy_k(kbase, (t + u) * kTileRows, p.Sk, lds_k[slot] + u * TILE, wide);
        copy_v(vbase, (t + u) * kTileRows, p.Sk, lds_v[slot] + u * TILE, wide);
      }
  };

  auto block = [&](int t, int slot) __attribute__((always_inline)) {
    const int n0 = t * kTileRows;
    const BlockCode code = block_code(p, band, b, hq, iw0, n0);
    if (!code.live) return;
    const char* kt = lds_k[slot] + kp * TILE;
    const f32x16_t s = ops.scores(kt, qf);
    f32x16_t dp = ops.scores(lds_v[slot] + kp * TILE, of);
    float x[16];
    const float fi = (float)(i - n0 - 4 * g);
#pragma unroll
    for (int v = 0; v < 16; ++v) x[v] = __builtin_fmaf(s[v], p.scale_log2, -lse2);
    if (p.alibi) {
#pragma unroll
      for (int v = 0; v < 16; ++v) x[v] = __builtin_fmaf(fabsf(fi - (float)((v >> 2) * 8 + (v & 3))), slope_l2, x[v]);
    }
    if (code.mask) {
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        float mv[4];
        load_mask4(mrow, p.mask_dtype, n0 + vq * 8 + g * 4, p.mk_sj, p.Sk - 1, mv);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[vq * 4 + e] += mv[e] * kLog2e;
      }
    }
    if (!code.full) {
      // keys the lane's row may see (see bwd_dkdv_generic)
      int io = i;
      asm volatile("" : "+v"(io));
      const Span kspan = io < p.Sq ? Span(max((int64_t)0, (int64_t)io + band.dlo), min((int64_t)p.Sk - 1, (int64_t)io + band.dhi))
                                   : Span(1, 0);
#pragma unroll
      for (int v = 0; v < 16; ++v) x[v] = kspan.ok(n0 + (v >> 2) * 8 + g * 4 + (v & 3)) ? x[v] : -INFINITY;
    }
    if constexpr (DROP) {
#pragma unroll
      for (int vp = 0; vp < 2; ++vp) {  // 8-key groups vq = 2vp, 2vp + 1: one call per lane pair
        uint32_t wq[2][2];
        philox_pair_words((uint32_t)((n0 + vp * 16) >> 3), (uint32_t)i, (uint32_t)(b * p.Hq + hq), dkey.off_lo, dkey.k0,
                          dkey.k1, g, wq[0], wq[1]);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int v = (vp * 2 + h) * 4 + e;
            dp[v] = keep_field(wq[h][e >> 1], e & 1, dkey.thresh) ? dp[v] : 0.f;
          }
      }
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) x[v] = __builtin_amdgcn_exp2f(x[v]) * (dp[v] - dlt);
    zs.apply(x, acc);
    ops.accum(acc, kt, x);
  };

  if (t_lo < t_hi) load(t_lo, 0);
  auto step = [&](auto slot_c, int t) __attribute__((always_inline)) {
    constexpr int SL = decltype(slot_c)::value;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t + KS < t_hi) load(t + KS, 1 - SL);
    if (t + kp < t_hi) block(t + kp, SL);
  };
  for (int t = t_lo; t < t_hi; t += 2 * KS) {
    step(std::integral_constant<int, 0>{}, t);
    if (t + KS < t_hi) step(std::integral_constant<int, 1>{}, t + KS);
  }

  float f = p.scale * (DROP ? p.drop_scale : 1.f) * zs.undo();
  if constexpr (KS == 2) {
    merge_pair<2 * KS * TILE>(acc, f, (float*)&lds_k[0][0], rgrp, kp, lane);
    if (kp == 1) return;
    f = 1.f;
  }
  if (i < p.Sq) {
    Store* row = (Store*)p.dq + b * p.dq_sb + hq * p.dq_sh + (int64_t)i * p.dq_ss;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        const int d0 = (db0 + db) * 32 + vq * 8 + g * 4;
        O::store4(row, d0, acc[db][vq * 4] * f, acc[db][vq * 4 + 1] * f, acc[db][vq * 4 + 2] * f, acc[db][vq * 4 + 3] * f);
      }
  }
}

// Blocks of 128 / KS keys or rows (p.num_kblk, p.num_mblk), KS wavefronts per
// 32 of them, their columns over HS workgroups.
template <class O, int OCC, int HS, int KS>
hipError_t launch_generic_dkdv(const BwdParams& p, hipStream_t st) {
  const dim3 grid((unsigned)(p.B * p.Hkv * p.num_kblk * HS));
  if (p.use_dropout) return launch_kernel(&bwd_dkdv_generic<O, OCC, HS, KS, true>, grid, dim3(256), 0, st, p);
  return launch_kernel(&bwd_dkdv_generic<O, OCC, HS, KS, false>, grid, dim3(256), 0, st, p);
}
template <class O, int OCC, int HS, int KS>
hipError_t launch_generic_dq(const BwdParams& p, hipStream_t st) {
  const dim3 grid((unsigned)(p.B * p.Hq * p.num_mblk * HS));
  if (p.use_dropout) return launch_kernel(&bwd_dq_generic<O, OCC, HS, KS, true>, grid, dim3(256), 0, st, p);
  return launch_kernel(&bwd_dq_generic<O, OCC, HS, KS, false>, grid, dim3(256), 0, st, p);
}

// Both gradient kernels of one dtype (attn_bwd_generic_*.hip); plan: plan_bwd's.
hipError_t launch_bwd_generic_f32(const BwdParams& p, int D, const BwdPlan& plan, hipStream_t st);
hipError_t launch_bwd_generic_bf16(const BwdParams& p, const BwdPlan& plan, hipStream_t st);
hipError_t launch_bwd_generic_f16(const BwdParams& p, const BwdPlan& plan, hipStream_t st);

}  // namespace trinix
