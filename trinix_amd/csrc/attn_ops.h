// Operand policies of the attention kernels whose coefficients (P, dZ) enter
// their products with more bits than a 16-bit operand has: what a tile of 32
// rows looks like in LDS, how a wavefront forms a 32x32 block of row products
// from it, and how it adds tile^T * coefficients to its accumulators.
//
// Common shape: a wavefront owns 32 columns (keys in dK/dV, query rows in dQ
// and the forward); lane l holds column l % 32, whose own rows (K and V, or Q
// and dO) are a Frag in registers.  A tile holds 32 rows of the other side in
// LDS, 16-byte units XOR-swizzled within the row, filled by asynchronous
// copies.  With g = l / 32 and element v = 0..15:
//   scores(tile, frag)   element v: row (v/4)*8 + 4g + v%4 of the tile times
//                        the lane's column;
//   accum(acc, tile, x)  acc[k], k < NDB (row d = (db0 + k)*32 + (v/4)*8 + 4g +
//                        v%4, column l % 32) += sum over tile rows of
//                        tile[row][d] * x, for the NDB of the D/32 head_dim
//                        blocks from db0 (a multiple of NDB).
//
//   Ops32  fp32 operands on v_mfma_f32_32x32x2f32 (exact products, fp32 sums);
//          the coefficients keep all 24 bits; an operand element is 4 bytes,
//          so neither product needs a transposed copy and P / dZ never leave
//          the registers.
//   Ops16  16-bit operands on v_mfma_f32_32x32x16; the coefficients enter as
//          two 16-bit terms x = hi + lo, hi = round(x), lo = round(x - hi): 16
//          (bf16) or 21 (fp16) significant bits, two MFMAs per operand read.
#pragma once
#include <type_traits>

#include "attn_params.h"
#include "lds_tile.h"

namespace trinix {

constexpr int kTileRows = 32;

// LDS operand reads of a row-major, D-wide 16-bit tile swizzled with swz_kt.
// Row read: row l % 32, head_dim chunk ds (16 elements).  Transpose read:
// rows t and t + 8 of k-step kk, head_dim block db.  The swizzle touches the
// low four bits of a row's 16-byte unit index, so an address is a per-lane
// base XOR an immediate below 256 bytes, plus a multiple of 256 bytes.
template <int D>
struct Tile16Reader {
  uint32_t row_lane, tr0, tr1;
  __device__ Tile16Reader(int lane, int db0) {
    const int r = lane & 31, g = lane >> 5;
    row_lane = (uint32_t)(r * D * 2 + 16 * (g ^ swz_kt<D>(r)));
    const int tr_G = lane >> 4, tr_s = lane & 15, tr_g = tr_G >> 1, tr_dh = tr_G & 1;
    const int row0 = tr_g * 4 + (tr_s >> 2), row1 = row0 + 8;
    const int c = tr_dh * 2 + ((tr_s & 3) >> 1), half = (tr_s & 1) * 4;
    tr0 = (uint32_t)((row0 * D + (c ^ swz_kt<D>(row0)) * 8 + half) * 2) + (uint32_t)(db0 << 6);
    tr1 = (uint32_t)((row1 * D + (c ^ swz_kt<D>(row1)) * 8 + half) * 2) + (uint32_t)(db0 << 6);
  }
  __device__ static const char* at(const char* tile, uint32_t x, int byte) {
    return tile + (byte & ~255) + (x ^ (uint32_t)(byte & 255));
  }
  __device__ u32x4_t row(const char* tile, int ds) const { return *(const u32x4_t*)at(tile, row_lane, ds << 5); }
  __device__ u32x4_t tr(const char* tile, int db, int kk) const {
    const char* base = tile + kk * 16 * D * 2;
    const s16x4_t lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)at(base, tr0, db << 6));
    const s16x4_t hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)at(base, tr1, db << 6));
    const u32x2_t l2 = __builtin_bit_cast(u32x2_t, lo4), h2 = __builtin_bit_cast(u32x2_t, hi4);
    return (u32x4_t){l2[0], l2[1], h2[0], h2[1]};
  }
};

template <class E, int D>
struct Ops16 {
  using Store = uint16_t;
  static constexpr int kD = D, DS = D / 16, DB = D / 32;
  // Held at 2^kPShift: fp16 terms have a fixed quantum of 2^-24, so P (at
  // most 1) is held times 2^11, and dZ at a power of two of its own (Scale).
  static constexpr bool kScaled = std::is_same<E, F16>::value;
  static constexpr float kPShift = kScaled ? 11.f : 0.f;
  struct Frag {
    u32x4_t r[DS];
  };
  Tile16Reader<D> rd;
  __device__ Ops16(int lane, int db0) : rd(lane, db0) {}  // db0: a multiple of 4 (256-byte steps)

  __device__ static Frag load_frag(const Store* row, int g) {
    Frag f;
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) f.r[ds] = *(const u32x4_t*)(row + ds * 16 + g * 8);
    return f;
  }
  // 16-byte unit of tile row `row` held at LDS unit `u`
  __device__ static int swz(int u, int row) { return u ^ swz_kt<D>(row); }

  // Operand reads run PF MFMAs ahead, pinned with sched_group_barrier
  // (0x100 LDS read, 0x008 MFMA).
  __device__ f32x16_t scores(const char* tile, const Frag& f) const {
    constexpr int PF = 4;
    f32x16_t s = {};
    u32x4_t a[DS];
#pragma unroll
    for (int k = 0; k < PF; ++k) a[k] = rd.row(tile, k);
#pragma unroll
    for (int k = 0; k < DS; ++k) {
      if (k + PF < DS) a[k + PF] = rd.row(tile, k + PF);
      s = E::mfma(a[k], f.r[k], s);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, PF, 0);
#pragma unroll
    for (int k = 0; k < DS; ++k) {
      if (k + PF < DS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    return s;
  }
  template <int NDB>
  __device__ void accum(f32x16_t (&acc)[NDB], const char* tile, const float (&x)[16]) const {
    constexpr int PF = 3, NM = 2 * NDB;
    u32x4_t b[2][2];  // [term][k-step]
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float x0 = x[kk * 8 + 2 * w], x1 = x[kk * 8 + 2 * w + 1];
        const uint32_t h = E::pack(x0, x1);
        b[0][kk][w] = h;
        b[1][kk][w] = E::pack(x0 - E::lo(h), x1 - E::hi(h));
      }
    u32x4_t a[NM];
#pragma unroll
    for (int m = 0; m < PF; ++m) a[m] = rd.tr(tile, m / 2, m % 2);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      if (m + PF < NM) a[m + PF] = rd.tr(tile, (m + PF) / 2, (m + PF) % 2);
      acc[m / 2] = E::mfma(a[m], b[1][m % 2], acc[m / 2]);
      acc[m / 2] = E::mfma(a[m], b[0][m % 2], acc[m / 2]);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 2 * PF, 0);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      if (m + PF < NM) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
    }
  }
  // four consecutive head_dim elements of an output row
  __device__ static void store4(Store* row, int d, float a, float b, float c, float e) {
    *(u32x2_t*)(row + d) = (u32x2_t){E::pack(a, b), E::pack(c, e)};
  }
};

template <int D>
struct Ops32 {
  using Store = float;
  static constexpr int kD = D, DB = D / 32, DT = D / 8;
  static constexpr bool kScaled = false;
  static constexpr float kPShift = 0.f;
  struct Frag {
    f32x4_t r[DT];  // element e of r[t]: d = 8t + 4g + e
  };
  uint32_t row_lane, col_lane;
  __device__ Ops32(int lane, int db0) {
    const int r = lane & 31, g = lane >> 5;
    row_lane = (uint32_t)(r * D * 4 + 16 * (g ^ (r & 15)));
    col_lane = (uint32_t)(4 * g * D * 4 + 16 * ((r >> 2) ^ (4 * g) ^ (db0 * 8)) + 4 * (r & 3));
  }
  // (head_dim 256 has no registers to hold the results across the loop)
  __device__ static uint32_t at(uint32_t x, uint32_t imm) {
    if constexpr (D == 256) asm volatile("" : "+v"(x));
    return x ^ imm;
  }
  // any 4-byte aligned row
  __device__ static Frag load_frag(const Store* row, int g) {
    typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
    Frag f;
#pragma unroll
    for (int t = 0; t < DT; ++t) f.r[t] = *(const f32x4_any*)(row + t * 8 + g * 4);
    return f;
  }
  __device__ static int swz(int u, int row) { return u ^ swz_f32(row); }

  // The k pairs of MFMA (t, e) are d = 8t + e (lanes 0..31) and 8t + 4 + e.
  __device__ f32x16_t scores(const char* tile, const Frag& f) const {
    constexpr int PF = D == 256 ? 1 : 2;
    f32x16_t s = {};
    f32x4_t a[DT];
    auto read = [&](int t) __attribute__((always_inline)) {
      a[t] = *(const f32x4_t*)(tile + at(row_lane, (uint32_t)(t << 5)));
    };
#pragma unroll
    for (int t = 0; t < PF; ++t) read(t);
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      if (t + PF < DT) read(t + PF);
#pragma unroll
      for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t][e], f.r[t][e], s, 0, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, PF, 0);
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      if (t + PF < DT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
    }
    return s;
  }
  // Coefficient element v is the k pair of tile rows (v/4)*8 + v%4 and + 4.
  template <int NDB>
  __device__ void accum(f32x16_t (&acc)[NDB], const char* tile, const float (&x)[16]) const {
    constexpr int PF = D == 256 ? 3 : 6, NM = 16 * NDB;
    float a[NM];
    auto read = [&](int m) __attribute__((always_inline)) {
      const int v = m / NDB, db = m % NDB, row = (v >> 2) * 8 + (v & 3);  // + 4g (col_lane)
      a[m] = *(const float*)(tile + row * D * 4 + at(col_lane, (uint32_t)(((db * 8) ^ (row & 15)) << 4)));
    };
#pragma unroll
    for (int m = 0; m < PF; ++m) read(m);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      if (m + PF < NM) read(m + PF);
      acc[m % NDB] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[m], x[m / NDB], acc[m % NDB], 0, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, PF, 0);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      if (m + PF < NM) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
  }
  __device__ static void store4(Store* row, int d, float a, float b, float c, float e) {
    row[d] = a;
    row[d + 1] = b;
    row[d + 2] = c;
    row[d + 3] = e;
  }
};

// The power of two that a lane's column of dZ is held at where its terms
// have a fixed quantum (Ops16 at fp16): set by the first nonzero block, and
// lowered together with the accumulators when a block's largest |dZ| would
// pass 2^15.  Both lanes of a column (l, l ^ 32) take the same steps.
template <class O>
struct ZScale {
  float f = 0x1p+120f;
  template <int NDB>
  __device__ void apply(float (&z)[16], f32x16_t (&acc)[NDB]) {
    if constexpr (O::kScaled) {
      float m = 0.f;
#pragma unroll
      for (int v = 0; v < 16; ++v) m = fmaxf(m, fabsf(z[v]));
      const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
      m = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      const bool over = m * f > 32768.f;
      if (__builtin_amdgcn_ballot_w64(over) != 0) {
        const float nf = over ? ldexpf(1.f, 11 - __builtin_amdgcn_frexp_expf(m)) : f;  // m * nf in [2^10, 2^11)
        const float r = nf / f;
        f = nf;
#pragma unroll
        for (int db = 0; db < NDB; ++db) acc[db] *= r;
      }
#pragma unroll
      for (int v = 0; v < 16; ++v) z[v] *= f;
    }
  }
  __device__ float undo() const { return O::kScaled ? 1.f / f : 1.f; }
};

// Asynchronous copy of tile rows [i0, i0 + 32) of a (rows, D) slice (row
// stride ss elements, n rows; rows past the last read the last) to an LDS
// tile, 16 bytes per lane, spread over NW wavefronts.  The lane's offsets
// within a tile are formed once; a tile then costs scalar instructions only
// (fp32 products leave the vector ALU no cycles of its own).  `wide` false:
// fp32 rows that are not 16-byte aligned, or whose stride leaves the 32-bit
// offsets: 4 bytes per lane from 64-bit addresses.
template <class O, int NW>
struct TileCopy {
  using Store = typename O::Store;
  static constexpr int ESZ = (int)sizeof(Store), UPR = O::kD * ESZ / 16, PER = kTileRows * UPR / (64 * NW);
  static_assert(PER >= 1 && kTileRows * UPR % (64 * NW) == 0, "tile shape");
  int64_t ss;
  int wave, lane;
  uint32_t off[PER];
  __device__ TileCopy(int64_t ss_, int wave_, int lane_) : ss(ss_), wave(wave_), lane(lane_) {
#pragma unroll
    for (int l = 0; l < PER; ++l) off[l] = offset(l, kTileRows - 1);
  }
  __device__ uint32_t offset(int l, int last) const {
    const int row = tile_copy_row(wave, PER, l, lane, UPR);
    return tile32_offset(row, last, ss, ESZ, O::swz(((wave * PER + l) * 64 + lane) % UPR, row));
  }
  __device__ void operator()(const Store* base, int i0, int n, char* lds_tile, bool wide) const {
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void_t*)lds_tile;
    if (ESZ == 2 || wide) {
      const uint64_t gb = uniform_ptr(base + (int64_t)i0 * ss);
      if (i0 + kTileRows <= n) {
#pragma unroll
        for (int l = 0; l < PER; ++l) dma_16b_s(off[l], gb, __builtin_amdgcn_readfirstlane(lds0 + (wave * PER + l) * 1024));
      } else {
#pragma unroll 1
        for (int l = 0; l < PER; ++l)
          dma_16b_s(offset(l, n - 1 - i0), gb, __builtin_amdgcn_readfirstlane(lds0 + (wave * PER + l) * 1024));
      }
    } else {
#pragma unroll 1
      for (int l = 0; l < PER * 4; ++l) {
        const int c = wave * PER * 4 + l, word = c * 64 + lane, unit = word / 4, row = unit / UPR;
        dma_4b(base + (int64_t)min(i0 + row, n - 1) * ss + O::swz(unit % UPR, row) * 4 + (word & 3),
               __builtin_amdgcn_readfirstlane(lds0 + c * 256));
      }
    }
  }
};

// The block of query rows [ia, ia + 32) and keys [ja, ja + 32) of one
// (batch, q-head): does it hold allowed pairs (live), are all its pairs
// allowed (full), is its mask read (mask)?
struct BlockCode {
  bool live, full, mask;
};
template <class P>
__device__ inline BlockCode block_code(const P& p, const Band& band, int b, int hq, int ia, int ja) {
  BlockCode c{false, false, false};
  if (ia >= p.Sq || ja >= p.Sk) return c;
  const int ib = min(ia + 31, p.Sq - 1), jb = min(ja + 31, p.Sk - 1);
  if (ja - ib > band.dhi || jb - ia < band.dlo) return c;
  if (p.mask) {
    c.mask = true;
    if (p.bmap) {
      const uint8_t code = p.bmap[b * p.bm_sb + hq * p.bm_sh + (int64_t)(ia / 32) * p.bm_cols + ja / 64];
      if (code == 2) return c;
      c.mask = code != 0;
    }
  }
  c.live = true;
  c.full = ia + 31 < p.Sq && ja + 31 < p.Sk && jb - ia <= band.dhi && ja - ib >= band.dlo;
  return c;
}

}  // namespace trinix
