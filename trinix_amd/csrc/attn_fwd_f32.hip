// fp32 attention forward: v_mfma_f32_32x32x2f32 (exact fp32 products, fp32
// sums).  Semantics of the 16-bit kernel (attn_kernel16.h; reference
// trinix/kernels/attention_kernel.py:123-216, :341-416).
//
// A workgroup of 4 wavefronts owns 128 query rows of one (batch, q-head), 32
// per wavefront with their Q rows in registers, or (KS = 2) 64 rows with two
// wavefronts per 32 taking alternate key tiles, merged through LDS at the
// end.  Tiles of 32 keys go global -> LDS asynchronously into two slots, one
// barrier per step; S^T = K Q^T with each lane owning one query row, and
// O^T += V^T P^T straight from the score registers (attn_ops.h Ops32).
// Bound by the matrix cores: a 32x32 block takes D MFMAs of 64 cycles, which
// share the vector ALU's cycles (67% MFMA busy at D = 64).  B=4 S=1024 12 heads
// D=64 causal: 258 us with tiles staged through registers behind two barriers,
// now 79.
#include "attn_ops.h"

namespace trinix {
namespace {

// the lane's Q row, rotated (RoPE) with eager PyTorch's separate roundings
template <int D>
__device__ inline void rotate_frag(typename Ops32<D>::Frag& f, const float* cosr, const float* sinr, int g) {
#pragma clang fp contract(off)
  const auto c = Ops32<D / 2>::load_frag(cosr, g), s = Ops32<D / 2>::load_frag(sinr, g);
#pragma unroll
  for (int t = 0; t < D / 16; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x1 = f.r[t][e], x2 = f.r[t + D / 16][e];
      f.r[t][e] = x1 * c.r[t][e] - x2 * s.r[t][e];
      f.r[t + D / 16][e] = x2 * c.r[t][e] + x1 * s.r[t][e];
    }
}

}  // namespace

template <int D, int KS, int OCC>
__global__ __launch_bounds__(256, OCC) void attn_fwd_f32(const FwdParams p) {
  using O = Ops32<D>;
  constexpr int NW = kWavesF32, BM = NW * 32 / KS, DB = D / 32, TILE = kTileRows * D * 4;
  __shared__ __attribute__((aligned(1024))) char lds_k[2][KS * TILE];
  __shared__ __attribute__((aligned(1024))) char lds_v[2][KS * TILE];

  const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rgrp = wave / KS, kp = wave % KS;
  const FwdItem wi = fwd_item((int)blockIdx.x, p.B, p.Hkv, p.G, p.num_mblk, p.total_work, p.causal != 0, p.has_window != 0);
  const int hkv = wi.hkv, b = wi.b, hq = hkv * p.G + wi.gq;
  const int m0 = (p.causal ? p.num_mblk - 1 - wi.mi : wi.mi) * BM;  // causal: longest rows first
  const int iw0 = m0 + rgrp * 32, i = iw0 + r, ic = min(i, p.Sq - 1);
  const Band band(p);
  const Span kspan = i < p.Sq ? Span(max((int64_t)0, (int64_t)i + band.dlo), min((int64_t)p.Sk - 1, (int64_t)i + band.dhi))
                              : Span(1, 0);
  const bool wide = p.rows16 != 0;
  DropKey dkey{};
  if (p.use_dropout) dkey = drop_key(p);

  const O ops(lane, 0);
  typename O::Frag qf = O::load_frag((const float*)p.q + b * p.q_sb + hq * p.q_sh + (int64_t)ic * p.q_ss, g);
  if (p.rope_cos)
    rotate_frag<D>(qf, (const float*)p.rope_cos + (int64_t)ic * p.rope_stride,
                   (const float*)p.rope_sin + (int64_t)ic * p.rope_stride, g);
  const float slope_l2 = p.alibi ? -p.alibi[b * p.al_sb + hq * p.al_sh] * kLog2e : 0.f;
  const int esz = p.mask_dtype == TRINIX_F32 ? 4 : (p.mask_dtype == TRINIX_U8 ? 1 : 2);
  const char* mrow = p.mask ? (const char*)p.mask + (b * p.mk_sb + hq * p.mk_sh + (int64_t)ic * p.mk_si) * esz : nullptr;
  f32x16_t acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = (f32x16_t){};
  float m_run = -INFINITY, l_run = 0.f;

  int t_lo, t_hi;
  bwd_key_tiles(m0, BM, p.Sq, p.Sk, band.dlo, band.dhi, kTileRows, t_lo, t_hi);
  const float* kbase = (const float*)p.k + b * p.k_sb + hkv * p.k_sh;
  const float* vbase = (const float*)p.v + b * p.v_sb + hkv * p.v_sh;
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
    const f32x16_t s = ops.scores(lds_k[slot] + kp * TILE, qf);
    float x[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) x[v] = s[v] * p.scale_log2;
    if (p.alibi) {
      const float fi = (float)(i - n0 - 4 * g);
#pragma unroll
      for (int v = 0; v < 16; ++v) x[v] = __builtin_fmaf(fabsf(fi - (float)((v >> 2) * 8 + (v & 3))), slope_l2, x[v]);
    }
    if (code.mask) {
#pragma unroll
      for (int vq = 0; vq < 4; ++vq) {
        float mv[4];
        load_mask4(mrow, p.mask_dtype, n0 + vq * 8 + g * 4, p.mk_sj, p.Sk - 1, mv);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[vq * 4 + e] = __builtin_fmaf(mv[e], kLog2e, x[vq * 4 + e]);
      }
    }
    if (!code.full) {
#pragma unroll
      for (int v = 0; v < 16; ++v) x[v] = kspan.ok(n0 + (v >> 2) * 8 + g * 4 + (v & 3)) ? x[v] : -INFINITY;
    }
    float mx = x[0];
#pragma unroll
    for (int v = 1; v < 16; ++v) mx = fmaxf(mx, x[v]);
    mx = xlane_max(mx);
    if (wave_any(mx > m_run)) {
      const float m_new = fmaxf(m_run, mx);
      const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) acc[db] *= alpha;
      m_run = m_new;
    }
    const float m_use = m_run == -INFINITY ? 0.f : m_run;  // all keys so far masked: exp2(-inf - 0) = 0
    // summed within the tile first: a running sum over the keys would round
    // once per key of the row instead of once per tile
    float sum = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      x[v] = __builtin_amdgcn_exp2f(x[v] - m_use);
      sum += x[v];
    }
    l_run += sum;
    if (p.use_dropout) {
#pragma unroll
      for (int vp = 0; vp < 2; ++vp) {  // 8-key groups vq = 2vp, 2vp + 1
        float xa[4], xb[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          xa[e] = x[vp * 8 + e];
          xb[e] = x[vp * 8 + 4 + e];
        }
        dropout_pair(xa, xb, dkey, b * p.Hq + hq, i, n0 + vp * 16, g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          x[vp * 8 + e] = xa[e];
          x[vp * 8 + 4 + e] = xb[e];
        }
      }
    }
    ops.accum(acc, lds_v[slot] + kp * TILE, x);
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

  float l = xlane_sum(l_run);
  if constexpr (KS == 2) {
    // the second wavefront's (max, sum, O) merge into the first's
    constexpr int WORDS = DB * 16 + 2;
    static_assert(2 * WORDS * 64 * 4 <= 2 * KS * TILE, "exchange fits the K tiles");
    float* x = (float*)&lds_k[0][0] + rgrp * WORDS * 64 + lane;
    __syncthreads();
    if (kp == 1) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) x[(db * 16 + v) * 64] = acc[db][v];
      x[DB * 16 * 64] = m_run;
      x[(DB * 16 + 1) * 64] = l;
    }
    __syncthreads();
    if (kp == 1) return;
    const float m1 = x[DB * 16 * 64], l1 = x[(DB * 16 + 1) * 64];
    const float m_new = fmaxf(m_run, m1), m_use = m_new == -INFINITY ? 0.f : m_new;
    const float a0 = __builtin_amdgcn_exp2f(m_run - m_use), a1 = __builtin_amdgcn_exp2f(m1 - m_use);
    l = l * a0 + l1 * a1;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[db][v] = acc[db][v] * a0 + x[(db * 16 + v) * 64] * a1;
    m_run = m_new;
  }
  if (i < p.Sq) {
    float* orow = (float*)p.o + b * p.o_sb + hq * p.o_sh + (int64_t)i * p.o_ss;
    // with dropout, the 1/(1-p) of the kept weights (dropout_pair)
    const float os = p.use_dropout ? p.drop_scale : 1.f;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int vq = 0; vq < 4; ++vq)
        O::store4(orow, db * 32 + vq * 8 + g * 4, acc[db][vq * 4] * os / l, acc[db][vq * 4 + 1] * os / l,
                  acc[db][vq * 4 + 2] * os / l, acc[db][vq * 4 + 3] * os / l);
    if (p.lse && g == 0) p.lse[((int64_t)b * p.Hq + hq) * p.Sq + i] = (m_run + log2f(l)) * kLn2;
  }
}

hipError_t launch_attn_f32(const FwdParams& p, int head_dim, int ks, hipStream_t st) {
  const dim3 grid((unsigned)p.total_work), block(kWavesF32 * 64);
  switch (head_dim) {
    case 64:
      return ks == 2 ? launch_kernel(&attn_fwd_f32<64, 2, 2>, grid, block, 0, st, p)
                     : launch_kernel(&attn_fwd_f32<64, 1, 2>, grid, block, 0, st, p);
    case 128:
      return ks == 2 ? launch_kernel(&attn_fwd_f32<128, 2, 1>, grid, block, 0, st, p)
                     : launch_kernel(&attn_fwd_f32<128, 1, 1>, grid, block, 0, st, p);
    case 256: return launch_kernel(&attn_fwd_f32<256, 1, 1>, grid, block, 0, st, p);
  }
  return hipErrorNotSupported;
}

}  // namespace trinix
