// CPU driver for the host-side argument checks and launch planning of
// libtrinix_attn.so (trinix_amd/csrc/host_plan.cpp), built by
// tests/test_host_sanitizers.py with AddressSanitizer and
// UndefinedBehaviorSanitizer (every report fatal).  It runs the status-code
// cases of the C ABI's validation, then a seeded fuzz over the whole range of
// every size, stride and window field (int64 extremes included), and checks
// the split-KV plan's invariants on every accepted decode call.  The bounds
// model (bounds_model.h) then walks the kernels' index maps for the
// BASELINE configurations and edge shapes (every work item and row where
// the grid is small enough) and for a share of the accepted fuzz cases.
// Exit status 0 and a final "ok" line mean no sanitizer report and no
// failed check.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>

#include "bounds_model.h"
#include "host_plan.h"

using namespace trinix;

static int failures = 0;
#define CHECK(cond, ...)                                 \
  do {                                                   \
    if (!(cond)) {                                       \
      std::fprintf(stderr, "check failed: " __VA_ARGS__); \
      std::fprintf(stderr, "\n");                        \
      ++failures;                                        \
    }                                                    \
  } while (0)

static uint64_t rng = 0x9E3779B97F4A7C15ull;
static uint64_t next_u64() {  // xorshift64*
  rng ^= rng >> 12;
  rng ^= rng << 25;
  rng ^= rng >> 27;
  return rng * 0x2545F4914F6CDD1Dull;
}
static int64_t pick(const int64_t* vals, int n) { return vals[next_u64() % (uint64_t)n]; }

static const int64_t kEdge[] = {std::numeric_limits<int64_t>::min(), -(1ll << 40), -65536, -1, 0, 1, 2, 3, 7, 8,
                                15, 16, 17, 63, 64, 65, 127, 128, 1000, 4096, 8192, 65535, 1ll << 20, (1ll << 22) - 8,
                                1ll << 22, (1ll << 30) - 1, 1ll << 30, 1ll << 40, std::numeric_limits<int64_t>::max()};
static const int kNEdge = sizeof(kEdge) / sizeof(kEdge[0]);

static int64_t rand_size() {
  switch (next_u64() % 4) {
    case 0: return pick(kEdge, kNEdge);
    case 1: return (int64_t)(next_u64() % 17);
    case 2: return (int64_t)(next_u64() % 100000);
    default: return (int64_t)next_u64();
  }
}

static trinix_attn_fwd_args valid_fwd() {
  trinix_attn_fwd_args a;
  std::memset(&a, 0, sizeof(a));
  a.q = a.k = a.v = a.out = (void*)4096;
  const int64_t st[4] = {8 * 64 * 128, 8 * 128, 128, 1};
  for (int i = 0; i < 4; ++i) a.q_stride[i] = a.k_stride[i] = a.v_stride[i] = a.out_stride[i] = st[i];
  a.batch = 1;
  a.seqlen_q = 64;
  a.seqlen_k = 64;
  a.nheads_q = 8;
  a.nheads_kv = 8;
  a.head_dim = 128;
  a.dtype = TRINIX_BF16;
  a.softmax_scale = 0.088f;
  return a;
}

template <class Args>
static void set_mask(Args& x, int64_t sb, int64_t sh, int64_t si, int64_t sj) {
  x.mask = (const void*)4096;
  x.mask_dtype = TRINIX_F32;
  x.mask_stride[0] = sb;
  x.mask_stride[1] = sh;
  x.mask_stride[2] = si;
  x.mask_stride[3] = sj;
}

static trinix_attn_bwd_args valid_bwd() {
  trinix_attn_bwd_args a;
  std::memset(&a, 0, sizeof(a));
  a.q = a.k = a.v = a.out = a.dout = (void*)4096;
  a.dq = a.dk = a.dv = (void*)8192;
  a.lse = (const float*)4096;
  a.delta = (float*)8192;
  const int64_t st[4] = {8 * 64 * 128, 8 * 128, 128, 1};
  for (int i = 0; i < 4; ++i)
    a.q_stride[i] = a.k_stride[i] = a.v_stride[i] = a.out_stride[i] = a.dout_stride[i] = a.dq_stride[i] =
        a.dk_stride[i] = a.dv_stride[i] = st[i];
  a.batch = 1;
  a.seqlen_q = 64;
  a.seqlen_k = 64;
  a.nheads_q = 8;
  a.nheads_kv = 8;
  a.head_dim = 128;
  a.dtype = TRINIX_BF16;
  a.softmax_scale = 0.088f;
  return a;
}

// Invariants of an accepted split plan: the chunks tile the visible keys,
// the grid fits int32, the workspace matches rows * chunks * (D + 1) floats.
static void check_plan(const trinix_attn_fwd_args& a, const SplitPlan& pl) {
  CHECK(pl.n_splits >= 1 && pl.chunk >= 64 && pl.chunk % 64 == 0, "plan chunking");
  CHECK(pl.klo >= 0 && pl.klo < pl.khi && pl.khi <= a.seqlen_k, "plan key range");
  const int64_t span = (int64_t)pl.khi - pl.klo;
  CHECK((int64_t)pl.n_splits * pl.chunk >= span && (int64_t)(pl.n_splits - 1) * pl.chunk < span, "plan covers");
  const int64_t items = a.batch * a.nheads_kv * pl.RG;
  CHECK(items * pl.n_splits < (1ll << 31), "plan grid");
  const int64_t rows = a.batch * a.nheads_kv * pl.M;
  CHECK(pl.ws_bytes == (pl.n_splits > 1 ? rows * pl.n_splits * (a.head_dim + 1) * 4 : 0), "plan workspace");
}

// Grids of a backward plan, in 128 bits.  The fp32 and head_dim 256 kernels
// refuse what blocks of 32 keys or rows, or of 4 rows in the delta pass,
// cannot cover in one grid; the others what their own blocks cannot.
static void check_bwd_grids(const trinix_attn_bwd_args& a, int rc, const BwdPlan& pl, bool generic) {
  typedef __int128 wide;
  const wide lim = (wide)1 << 31, bq = (wide)a.batch * a.nheads_q, bkv = (wide)a.batch * a.nheads_kv;
  const int64_t delta_rows = a.dtype == TRINIX_F32 ? 1024 / a.head_dim : 2048 / a.head_dim;  // per workgroup
  const wide delta = (bq * a.seqlen_q + delta_rows - 1) / delta_rows;
  const bool fits32 = bkv * ((a.seqlen_k + 31) / 32) < lim && bq * ((a.seqlen_q + 31) / 32) < lim &&
                       (bq * a.seqlen_q + 3) / 4 < lim;
  CHECK(rc == TRINIX_OK || rc == TRINIX_ERR_BAD_SHAPE, "bwd plan status %d", rc);
  // (at most four workgroups of different columns share a block of 128 or 64)
  const bool one_each = bkv * ((a.seqlen_k + 63) / 64) * 4 < lim && bq * ((a.seqlen_q + 63) / 64) * 2 < lim;
  if (generic) CHECK(rc == TRINIX_OK ? fits32 : !fits32 || !one_each, "fp32 / head_dim 256 plan: rc %d", rc);
  if (rc != TRINIX_OK) return;
  CHECK(delta < lim, "delta grid");
  CHECK(bkv * pl.num_kblk * pl.kv_hs < lim && bq * pl.num_mblk * pl.dq_hs < lim, "gradient grids");
  const int bk = 128 / pl.kv_ks, bm = pl.dq_wide ? 256 : 128 / pl.dq_ks;
  CHECK((wide)pl.num_kblk * bk >= a.seqlen_k && (wide)pl.num_mblk * bm >= a.seqlen_q, "blocks cover");
  if (pl.kv_T) CHECK(bkv * pl.kv_P < lim && bkv * pl.num_kblk * 16 < lim, "piece grids");
  CHECK((wide)pl.ws_bytes == (pl.kv_T ? bkv * pl.kv_P * 2 * 128 * a.head_dim * 4 : 0), "piece workspace");
}

int main(int argc, char** argv) {
  int cases = 0;
  // ---- status codes of the forward's validation
  {
    trinix_attn_fwd_args a = valid_fwd();
    CHECK(validate_fwd_args(&a) == TRINIX_OK, "valid fwd");
    CHECK(validate_fwd_args(nullptr) == TRINIX_ERR_NULL_POINTER, "null args");
    struct Case {
      void (*edit)(trinix_attn_fwd_args&);
      int code;
    } table[] = {
        {[](trinix_attn_fwd_args& x) { x.q = nullptr; }, TRINIX_ERR_NULL_POINTER},
        {[](trinix_attn_fwd_args& x) { x.dtype = 7; }, TRINIX_ERR_BAD_DTYPE},
        {[](trinix_attn_fwd_args& x) { x.head_dim = 96; }, TRINIX_ERR_BAD_HEAD_DIM},
        {[](trinix_attn_fwd_args& x) { x.nheads_kv = 3; }, TRINIX_ERR_BAD_SHAPE},
        {[](trinix_attn_fwd_args& x) { x.seqlen_q = 0; }, TRINIX_ERR_BAD_SHAPE},
        {[](trinix_attn_fwd_args& x) { x.batch = std::numeric_limits<int64_t>::max(); }, TRINIX_ERR_BAD_SHAPE},
        {[](trinix_attn_fwd_args& x) { x.nheads_kv = std::numeric_limits<int64_t>::min(); }, TRINIX_ERR_BAD_SHAPE},
        {[](trinix_attn_fwd_args& x) { x.q_stride[3] = 2; }, TRINIX_ERR_BAD_STRIDE},
        {[](trinix_attn_fwd_args& x) { x.k_stride[2] = 130; }, TRINIX_ERR_BAD_STRIDE},
        {[](trinix_attn_fwd_args& x) { x.k_stride[1] = 1ll << 22; }, TRINIX_ERR_BAD_STRIDE},
        {[](trinix_attn_fwd_args& x) { x.v_stride[1] = std::numeric_limits<int64_t>::min(); }, TRINIX_ERR_BAD_STRIDE},
        {[](trinix_attn_fwd_args& x) { x.out = (void*)4100; }, TRINIX_ERR_BAD_STRIDE},
        {[](trinix_attn_fwd_args& x) { x.dropout_p = 1.0f; }, TRINIX_ERR_BAD_ARGUMENT},
        {[](trinix_attn_fwd_args& x) { x.dropout_p = NAN; }, TRINIX_ERR_BAD_ARGUMENT},
        {[](trinix_attn_fwd_args& x) { x.mask_blockmap = (const uint8_t*)4096; }, TRINIX_ERR_BAD_ARGUMENT},
        {[](trinix_attn_fwd_args& x) { x.rope_cos = (void*)4096; }, TRINIX_ERR_NULL_POINTER},
        {[](trinix_attn_fwd_args& x) { x.mask = (void*)4096; x.mask_dtype = 9; }, TRINIX_ERR_BAD_DTYPE},
        {[](trinix_attn_fwd_args& x) { x.q_norm_weight = (void*)4096; x.dropout_p = 0.1f; }, TRINIX_ERR_BAD_ARGUMENT},
        // mask strides: non-negative; a 32-row sub-tile's rows at 32-bit offsets
        {[](trinix_attn_fwd_args& x) { set_mask(x, 0, 0, -64, 1); }, TRINIX_ERR_BAD_STRIDE},
        {[](trinix_attn_fwd_args& x) { set_mask(x, -4096, 0, 64, 1); }, TRINIX_ERR_BAD_STRIDE},
        {[](trinix_attn_fwd_args& x) { set_mask(x, 0, 0, 1ll << 27, 1); }, TRINIX_ERR_BAD_STRIDE},
        {[](trinix_attn_fwd_args& x) { set_mask(x, 0, 0, (1ll << 31) / 31, 1); }, TRINIX_OK},
        {[](trinix_attn_fwd_args& x) { set_mask(x, 0, 0, 64, 1ll << 26); }, TRINIX_ERR_BAD_STRIDE},
        {[](trinix_attn_fwd_args& x) { x.seqlen_q = 1; set_mask(x, 0, 0, 1ll << 40, 1); }, TRINIX_OK},
    };
    for (const Case& c : table) {
      trinix_attn_fwd_args x = valid_fwd();
      c.edit(x);
      const int rc = validate_fwd_args(&x);
      CHECK(rc == c.code, "fwd case %d: got %d, want %d", cases, rc, c.code);
      ++cases;
    }
  }
  // ---- status codes of the backward's validation
  {
    trinix_attn_bwd_args a = valid_bwd();
    CHECK(validate_bwd_args(&a) == TRINIX_OK, "valid bwd");
    a.dtype = TRINIX_F32;
    a.q = (void*)4098;
    CHECK(validate_bwd_args(&a) == TRINIX_ERR_BAD_STRIDE, "bwd fp32 misaligned");
    a = valid_bwd();
    a.delta = nullptr;
    CHECK(validate_bwd_args(&a) == TRINIX_ERR_NULL_POINTER, "bwd delta");
    a = valid_bwd();
    a.dropout_p = -0.5f;
    CHECK(validate_bwd_args(&a) == TRINIX_ERR_BAD_ARGUMENT, "bwd dropout");
    a = valid_bwd();
    a.dk_stride[1] = std::numeric_limits<int64_t>::max();
    CHECK(validate_bwd_args(&a) == TRINIX_ERR_BAD_STRIDE, "bwd stride");
    // the dK/dV kernel reads a mask sub-tile's 32 rows at 32-bit offsets
    // r * row_stride from its first row (64-bit): (Sq = 64) 31 * stride < 2^31
    a = valid_bwd();
    set_mask(a, 0, 0, (1ll << 31) / 31 + 1, 1);
    CHECK(validate_bwd_args(&a) == TRINIX_ERR_BAD_STRIDE, "bwd mask row stride");
    a = valid_bwd();
    set_mask(a, 0, 0, (1ll << 31) / 31, 1);
    CHECK(validate_bwd_args(&a) == TRINIX_OK, "bwd mask row stride at the limit");
    a = valid_bwd();
    set_mask(a, 0, 0, -1, 1);
    CHECK(validate_bwd_args(&a) == TRINIX_ERR_BAD_STRIDE, "bwd negative mask row stride");
    a = valid_bwd();
    a.seqlen_q = a.seqlen_k = 70000;  // a contiguous mask beyond 2^32 elements
    set_mask(a, 0, 0, 70000, 1);
    CHECK(validate_bwd_args(&a) == TRINIX_OK, "bwd contiguous mask of 70000^2");
    cases += 9;
  }
  // ---- the backward plan's grids: a launch has fewer than 2^31 workgroups,
  // whatever the arguments that validation accepts (their products pass 2^63)
  {
    const int64_t big = (1 << 20) - 1, longest = (1ll << 30) - 1;
    const int64_t sizes[][5] = {{big, longest, longest, big, big}, {big, 1, longest, big, 1}, {big, longest, 1, big, big},
                                {1 << 19, longest, longest, 1 << 19, 1 << 19}, {1, longest, longest, big, 1},
                                {1, 1 << 17, 1 << 17, big, 1}, {16, 1 << 24, 1 << 24, 128, 128},
                                {1, 1 << 25, 1 << 25, 256, 256}, {1, longest, longest, 1, 1}};
    for (const auto& z : sizes)
      for (int dtype : {TRINIX_F32, TRINIX_F16, TRINIX_BF16})
        for (int64_t D : {64, 128, 256})
          for (bool split : {false, true}) {
            trinix_attn_bwd_args a = valid_bwd();
            a.batch = z[0], a.seqlen_q = z[1], a.seqlen_k = z[2], a.nheads_q = z[3], a.nheads_kv = z[4];
            a.dtype = dtype, a.head_dim = D;
            CHECK(validate_bwd_args(&a) == TRINIX_OK, "bwd sizes accepted");
            BwdPlan pl;
            const int rc = plan_bwd(&a, &pl, split);
            const bool generic = dtype == TRINIX_F32 || D == 256;
            check_bwd_grids(a, rc, pl, generic);
            ++cases;
          }
  }
  // ---- the forward's shape on small grids at head_dim 128 (figures beside
  // key_split, host_plan.cpp): where the key split of 32-key tiles loses, the
  // shape without it
  {
    struct Case {
      int64_t B, Sq, Sk, Hq, Hkv;
      int causal;
      int64_t window;  // 0: none
      int nw, bn, ks;
    } table[] = {
        {1, 1500, 1500, 8, 8, 0, 0, 4, 32, 2},       // 96 workgroups
        {1, 200, 200, 30, 30, 0, 0, 4, 32, 2},       // 60, chain 4
        {1, 130, 130, 30, 30, 0, 0, 4, 64, 1},       // 60, chain 3
        {1, 1024, 1024, 24, 24, 0, 0, 4, 32, 2},     // 192 of full rows, chain 16
        {1, 768, 768, 24, 24, 0, 0, 4, 64, 1},       // 144, chain 12
        {1, 640, 640, 48, 48, 0, 0, 4, 64, 1},       // 240, chain 10
        {1, 2048, 2048, 16, 16, 0, 0, 4, 64, 1},     // 256: full rows
        {8, 128, 2048, 32, 32, 0, 0, 8, 128, 1},     // 256 pairs of 128 full rows: the wide shape
        {1, 4096, 4096, 8, 8, 1, 512, 4, 64, 1},     // a window's even rows, 256
        {1, 4096, 4096, 6, 6, 1, 1024, 4, 32, 2},    // the same, 192, chain 18
        {1, 640, 640, 48, 48, 1, 0, 4, 32, 2},       // causal, head groups dealt evenly, chain 10
        {1, 700, 700, 28, 28, 1, 0, 4, 64, 1},       // not evenly, chain 11
        {1, 1024, 1024, 30, 30, 1, 0, 4, 64, 1},     // chain 16
        {1, 1200, 1200, 20, 20, 1, 0, 4, 32, 2},     // chain 19
        {1, 1024, 1024, 32, 4, 1, 0, 4, 64, 1},      // four groups of eight q-heads
    };
    for (const Case& c : table) {
      trinix_attn_fwd_args a = valid_fwd();
      a.batch = c.B, a.seqlen_q = c.Sq, a.seqlen_k = c.Sk, a.nheads_q = c.Hq, a.nheads_kv = c.Hkv, a.causal = c.causal;
      a.has_window = c.window > 0, a.window_left = c.window;
      FwdPlan pl;
      CHECK(validate_fwd_args(&a) == TRINIX_OK && plan_fwd(&a, &pl) == TRINIX_OK, "key split case");
      CHECK(pl.cfg.nw == c.nw && pl.cfg.bn == c.bn && pl.cfg.ks == c.ks, "key split case %d: (%d, %d, %d)", cases, pl.cfg.nw,
            pl.cfg.bn, pl.cfg.ks);
      ++cases;
    }
  }
  // ---- the decode launch's chunk count and loads (figures beside
  // decode_run_plan, host_plan.cpp): short rows in several rounds run unsplit
  // and through the caches
  {
    struct Case {
      int64_t B, Sk;
      int n_splits, streamed;
    } table[] = {{16, 8192, 2, 1}, {48, 2048, 2, 1}, {12, 8192, 8, 1}, {24, 8192, 4, 1}, {16, 1000, 2, 1},
                 {32, 300, 1, 1},  {48, 300, 1, 0},  {64, 300, 1, 0},  {96, 300, 1, 0},  {128, 300, 1, 0},
                 {12, 1000, 2, 0}, {128, 1000, 1, 1}};
    for (const Case& c : table) {  // 32 q-heads, 8 KV heads of D = 128: 8 B items, 32 B rows to merge
      trinix_attn_fwd_args a = valid_fwd();
      a.batch = c.B, a.seqlen_q = 1, a.seqlen_k = c.Sk, a.nheads_q = 32, a.nheads_kv = 8;
      SplitPlan pl;
      bool streamed = false;
      CHECK(validate_fwd_args(&a) == TRINIX_OK && make_split_plan(&a, &pl), "decode case");
      decode_run_plan(&a, &pl, &streamed);
      CHECK(pl.n_splits == c.n_splits && streamed == (c.streamed != 0), "decode case %d: %d chunks, streamed %d", cases,
            pl.n_splits, (int)streamed);
      ++cases;
    }
  }
  // ---- wavefronts per 32 rows or keys of the fp32 and head_dim 256 kernels
  // (figures beside two_per_group, host_plan.cpp)
  {
    struct Case {
      int dtype;
      int64_t D, B, S, H;
      int causal, fwd, dkdv, dq;
    } table[] = {
        {TRINIX_F32, 64, 4, 1024, 12, 1, 2, 2, 2},  {TRINIX_F32, 64, 8, 1024, 16, 1, 2, 2, 2},
        {TRINIX_F32, 64, 16, 1024, 16, 1, 1, 1, 2}, {TRINIX_F32, 64, 128, 256, 16, 1, 1, 1, 1},
        {TRINIX_F32, 64, 4, 1024, 12, 0, 2, 2, 2},  {TRINIX_F32, 64, 4, 1024, 16, 0, 1, 1, 1},
        {TRINIX_F32, 64, 7, 1024, 16, 0, 2, 2, 2},  {TRINIX_F32, 64, 32, 1024, 16, 0, 1, 1, 1},
        {TRINIX_F32, 128, 6, 1024, 8, 1, 2, 2, 2},  {TRINIX_F32, 128, 8, 1024, 8, 1, 1, 1, 2},
        {TRINIX_F32, 128, 2, 1024, 8, 0, 2, 2, 2},  {TRINIX_F32, 128, 3, 1024, 8, 0, 1, 1, 1},
        {TRINIX_F32, 128, 6, 1024, 8, 0, 2, 2, 2},  {TRINIX_F32, 256, 1, 1024, 8, 1, 1, 1, 1},
        {TRINIX_BF16, 256, 2, 1024, 8, 1, 1, 2, 2}, {TRINIX_BF16, 256, 2, 2048, 8, 1, 1, 1, 2},
        {TRINIX_BF16, 256, 2, 1024, 8, 0, 1, 1, 2}, {TRINIX_F16, 256, 2, 1024, 8, 0, 1, 1, 1},
        {TRINIX_F16, 256, 2, 1024, 8, 1, 1, 2, 2},  {TRINIX_F16, 256, 2, 2048, 8, 1, 1, 1, 1},
    };
    for (const Case& c : table) {
      trinix_attn_fwd_args f = valid_fwd();
      trinix_attn_bwd_args b = valid_bwd();
      f.batch = b.batch = c.B, f.seqlen_q = f.seqlen_k = b.seqlen_q = b.seqlen_k = c.S;
      f.nheads_q = f.nheads_kv = b.nheads_q = b.nheads_kv = c.H, f.head_dim = b.head_dim = c.D;
      f.dtype = b.dtype = c.dtype, f.causal = b.causal = c.causal;
      FwdPlan fp;
      BwdPlan bp;
      CHECK(validate_fwd_args(&f) == TRINIX_OK && validate_bwd_args(&b) == TRINIX_OK && plan_fwd(&f, &fp) == TRINIX_OK &&
                plan_bwd(&b, &bp) == TRINIX_OK, "wavefronts per group case");
      CHECK(fp.f32_ks == c.fwd && bp.kv_ks == c.dkdv && bp.dq_ks == c.dq, "wavefronts per group case %d: %d, %d, %d", cases,
            fp.f32_ks, bp.kv_ks, bp.dq_ks);
      ++cases;
    }
  }
  // ---- the tuning override TRINIX_ATTN_CFG="nw,occ,bn[,ks]": ks 0 (the
  // per-item split), 1 and 2 are taken, anything else leaves the planner's
  // choice
  {
    auto forced = [](const char* v) {
      setenv("TRINIX_ATTN_CFG", v, 1);
      const Cfg16 c = pick_cfg16(64, 1, 4, 512, true, true, true);
      unsetenv("TRINIX_ATTN_CFG");
      return c;
    };
    const Cfg16 dflt = pick_cfg16(64, 1, 4, 512, true, true, true);
    Cfg16 c = forced("4,2,64,0");
    CHECK(c.nw == 4 && c.occ == 2 && c.bn == 64 && c.ks == 0, "override ks 0");
    c = forced("4,2,64,2");
    CHECK(c.ks == 2, "override ks 2");
    c = forced("8,2,128");
    CHECK(c.nw == 8 && c.bn == 128 && c.ks == 1, "override without ks");
    c = forced("4,2,64,3");
    CHECK(c.nw == dflt.nw && c.bn == dflt.bn && c.ks == dflt.ks, "override ks 3 rejected");
    c = forced("3,2,64,2");
    CHECK(c.nw == dflt.nw && c.ks == dflt.ks, "override nw not a multiple of ks rejected");
    cases += 5;
  }
  // ---- fuzz: every field over its whole range
  int accepted = 0, planned = 0;
  for (int it = 0; it < 200000; ++it) {
    trinix_attn_fwd_args a = valid_fwd();
    a.batch = rand_size();
    a.seqlen_q = next_u64() % 3 ? (int64_t)(next_u64() % 20) : rand_size();
    a.seqlen_k = rand_size();
    a.nheads_kv = next_u64() % 2 ? (int64_t)(1 + next_u64() % 8) : rand_size();
    const bool small_kv = a.nheads_kv > 0 && a.nheads_kv <= (1 << 20);
    a.nheads_q = small_kv && next_u64() % 2 ? a.nheads_kv * (int64_t)(1 + next_u64() % 8) : rand_size();
    if (a.nheads_kv > 0 && a.nheads_q > 0 && a.nheads_q % a.nheads_kv) a.nheads_q = a.nheads_kv;
    a.head_dim = next_u64() % 5 ? (int64_t)(64 << (next_u64() % 3)) : rand_size();
    a.dtype = (int32_t)(next_u64() % 4);
    a.causal = (int32_t)(next_u64() % 2);
    a.has_window = (int32_t)(next_u64() % 2);
    a.window_left = rand_size();
    a.window_right = rand_size();
    for (int i = 0; i < 3; ++i) {
      if (next_u64() % 8 == 0) a.q_stride[i] = rand_size();
      if (next_u64() % 8 == 0) a.k_stride[i] = rand_size();
      if (next_u64() % 8 == 0) a.v_stride[i] = rand_size();
    }
    if (next_u64() % 16 == 0) a.dropout_p = (float)(next_u64() % 1000) / 900.f;
    const int rc = validate_fwd_args(&a);
    if (rc != TRINIX_OK) continue;
    ++accepted;
    const bool plain = !a.mask && a.dropout_p == 0.f;
    const bool split_ok = plain && a.causal && !a.has_window;
    const Cfg16 c = pick_cfg16(a.head_dim, a.batch, a.nheads_q, a.seqlen_q, a.causal || a.has_window, plain,
                               split_ok);
    CHECK((c.nw == 4 && c.bn == 64 && (c.ks == 1 || c.ks == 2)) ||
              (c.nw == 4 && c.bn == 64 && c.ks == 0 && a.head_dim == 64 && split_ok) ||
              (c.nw == 8 && c.bn == 128 && c.ks == 1 && a.head_dim == 128 && plain), "tile config");
    if (c.ks == 0) {
      uint8_t items[kMaxRowItems];
      const int n = plan_split_rows(a.seqlen_q, a.seqlen_k, a.batch * a.nheads_q, 128, 64, items, kMaxRowItems);
      CHECK(n >= 0 && n <= kMaxRowItems, "split items");
      // every 128-row block appears once whole or as both halves
      int seen[64] = {0};
      for (int k = 0; k < n; ++k) seen[items[k] >> 2] += (items[k] & 2) ? 1 : 2;
      const int64_t nb = (a.seqlen_q + 127) / 128;
      for (int64_t rb = 0; n > 0 && rb < nb; ++rb) CHECK(seen[rb] == 2, "split items cover every row block");
    }
    SplitPlan pl;
    if (make_split_plan(&a, &pl)) {
      ++planned;
      check_plan(a, pl);
      CHECK(a.seqlen_q <= kDecodeMaxSq, "plan only for decode shapes");
      CHECK(pl.ws_bytes <= (int64_t)TRINIX_SPLITKV_SCRATCH_BYTES, "default plan fits the static scratch");
      SplitPlan run = pl;
      bool streamed;
      decode_run_plan(&a, &run, &streamed);
      CHECK(run.n_splits >= 1 && run.n_splits <= pl.n_splits && run.ws_bytes == pl.ws_bytes, "run within the plan");
      run.ws_bytes = run.n_splits > 1 ? pl.ws_bytes / pl.n_splits * run.n_splits : 0;
      check_plan(a, run);
    }
  }
  for (int it = 0; it < 50000; ++it) {
    trinix_attn_bwd_args a = valid_bwd();
    a.batch = rand_size();
    a.seqlen_q = rand_size();
    a.seqlen_k = rand_size();
    a.nheads_kv = rand_size();
    a.nheads_q = rand_size();
    a.head_dim = next_u64() % 3 ? (int64_t)(64 << (next_u64() % 3)) : rand_size();
    a.dtype = (int32_t)(next_u64() % 4);
    for (int i = 0; i < 4; ++i)
      if (next_u64() % 4 == 0) a.dk_stride[i] = rand_size();
    if (next_u64() % 2 == 0) set_mask(a, rand_size(), rand_size(), rand_size(), rand_size());
    if (validate_bwd_args(&a) != TRINIX_OK) continue;
    if (a.mask) {
      // what the kernels' mask addressing relies on (see mask_strides_ok)
      for (int i = 0; i < 4; ++i) CHECK(a.mask_stride[i] >= 0, "accepted mask stride >= 0");
      const int64_t rows = a.seqlen_q - 1 < 31 ? a.seqlen_q - 1 : 31;
      CHECK((__int128)rows * a.mask_stride[2] < ((__int128)1 << 31), "sub-tile row offsets fit 31 bits");
      CHECK((__int128)(a.seqlen_k - 1) * a.mask_stride[3] < ((__int128)1 << 31), "key offsets fit 31 bits");
    }
    BwdPlan bp;
    const int prc = plan_bwd(&a, &bp, next_u64() % 2 == 0);
    check_bwd_grids(a, prc, bp, a.dtype == TRINIX_F32 || a.head_dim == 256);
    const bool masked = next_u64() % 2 == 0;
    if (pick_dq_wide(a.head_dim, a.batch, a.nheads_q, a.seqlen_q, a.causal || a.has_window, masked))
      CHECK(a.head_dim == 128 && !masked, "wide dQ only at head_dim 128 without a mask");
  }
  // ---- bounds model: curated shapes (every item and row where small), then
  // a share of the fuzz's accepted argument sets (sampled items)
  bounds::Report BR;
  int modelled = 0;
  long pieced = 0, generic = 0, narrow = 0;
  auto bwd_of = [](const trinix_attn_fwd_args& f) {
    trinix_attn_bwd_args b = valid_bwd();
    b.batch = f.batch, b.seqlen_q = f.seqlen_q, b.seqlen_k = f.seqlen_k, b.nheads_q = f.nheads_q;
    b.nheads_kv = f.nheads_kv, b.head_dim = f.head_dim, b.dtype = f.dtype, b.causal = f.causal;
    b.has_window = f.has_window, b.window_left = f.window_left, b.window_right = f.window_right;
    b.mask = f.mask, b.mask_dtype = f.mask_dtype, b.mask_blockmap = f.mask_blockmap, b.dropout_p = f.dropout_p;
    b.dropout_keep_map = f.dropout_keep_map;
    for (int i = 0; i < 4; ++i) {
      b.q_stride[i] = b.dout_stride[i] = b.out_stride[i] = b.dq_stride[i] = f.q_stride[i];
      b.k_stride[i] = b.dk_stride[i] = f.k_stride[i];
      b.v_stride[i] = b.dv_stride[i] = f.v_stride[i];
      b.mask_stride[i] = f.mask_stride[i];
    }
    return b;
  };
  auto model_pieces = [&](const trinix_attn_bwd_args& b) {
    BwdPlan bp;
    if (validate_bwd_args(&b) != TRINIX_OK || plan_bwd(&b, &bp, true) != TRINIX_OK || !bp.kv_T) return;
    bounds::model_pieces(BR, b, bp);
    ++pieced;
  };
  // `first`: the caller wants to know whether any check fails, not how many
  const bool first = argc > 1 && std::strcmp(argv[1], "first") == 0;
  auto model_one = [&](const trinix_attn_fwd_args& f, int64_t limit) {
    if (validate_fwd_args(&f) != TRINIX_OK || (first && BR.failures)) return;
    FwdPlan fp;
    const bool planned_fwd = plan_fwd(&f, &fp) == TRINIX_OK;
    if (f.dtype == TRINIX_F32) {
      if (planned_fwd) bounds::model_fwd_f32(BR, f, fp, limit);
    } else if (planned_fwd) {
      bounds::model_fwd16(BR, f, fp, limit);
    }
    SplitPlan sp;
    if (make_split_plan(&f, &sp)) {
      bounds::model_decode(BR, f, sp, limit);
      const int64_t slot = sp.ws_bytes / sp.n_splits;
      bool streamed;
      decode_run_plan(&f, &sp, &streamed);
      sp.ws_bytes = sp.n_splits > 1 ? slot * sp.n_splits : 0;
      bounds::model_decode(BR, f, sp, limit);
    }
    if (f.q_norm_weight == nullptr) {
      const trinix_attn_bwd_args b = bwd_of(f);
      BwdPlan bp;
      if (validate_bwd_args(&b) == TRINIX_OK) {
        if (plan_bwd(&b, &bp) == TRINIX_OK) {
          if (bp.generic) bounds::model_bwd_generic(BR, b, bp, limit), ++generic;
          else bounds::model_bwd16(BR, b, bp, limit);
        }
        model_pieces(b);
        if (b.dtype != TRINIX_F32 && b.head_dim <= 128)
          for (int64_t d : {(int64_t)8, b.head_dim / 2 + 8, b.head_dim - 8})
            if (b.batch * b.nheads_q < (1ll << 31)) bounds::model_narrow(BR, b, d), ++narrow;
      }
    }
    ++modelled;
  };
  auto shape = [](int64_t B, int64_t Sq, int64_t Sk, int64_t Hq, int64_t Hkv, int64_t D, int dtype) {
    trinix_attn_fwd_args a = valid_fwd();
    a.batch = B, a.seqlen_q = Sq, a.seqlen_k = Sk, a.nheads_q = Hq, a.nheads_kv = Hkv, a.head_dim = D, a.dtype = dtype;
    const int64_t q[4] = {Sq * Hq * D, Hq * D, D, 1}, kv[4] = {Sk * Hkv * D, Hkv * D, D, 1};
    for (int i = 0; i < 4; ++i) a.q_stride[i] = a.out_stride[i] = q[i], a.k_stride[i] = a.v_stride[i] = kv[i];
    return a;
  };
  {
    const int64_t kAll = 1 << 16;  // list every work item / row up to this many
    std::vector<trinix_attn_fwd_args> cur;
    auto add = [&](trinix_attn_fwd_args a) { cur.push_back(a); };
    trinix_attn_fwd_args a;
    a = shape(4, 1024, 1024, 12, 12, 64, TRINIX_BF16), a.causal = 1, add(a);          // C2
    a = shape(1, 8192, 8192, 32, 8, 128, TRINIX_BF16), a.causal = 1, add(a);          // C3
    a = shape(2, 16384, 16384, 32, 8, 128, TRINIX_BF16), a.causal = 1;                // C4
    a.has_window = 1, a.window_left = 4096, a.window_right = 0, add(a);
    a = shape(8, 2048, 2048, 16, 16, 64, TRINIX_F16);                                 // C5a, mask + block map
    a.mask = (void*)4096, a.mask_dtype = TRINIX_F32, a.mask_blockmap = (const uint8_t*)4096;
    a.mask_stride[0] = a.mask_stride[1] = 0, a.mask_stride[2] = 2048, a.mask_stride[3] = 1, add(a);
    a.nheads_kv = 1, a.k_stride[2] = a.v_stride[2] = 0, add(a);                       // C5b (expanded KV)
    for (int64_t D : {64, 128, 256})
      for (int64_t Sq : {1, 17, 100, 128, 300})
        for (int64_t Sk : {1, 63, 64, 65, 300})
          for (int c = 0; c < 6; ++c) {
            a = shape(2, Sq, Sk, 4, c % 2 ? 1 : 2, D, c % 3 ? TRINIX_BF16 : TRINIX_F16);
            a.causal = c & 1;
            if (c >= 2) a.has_window = 1, a.window_left = c == 4 ? -3 : 40, a.window_right = c == 5 ? (1ll << 62) : 7;
            if (c == 3) a.mask = (void*)4096, a.mask_dtype = TRINIX_BF16, a.mask_blockmap = (const uint8_t*)4096,
                        a.mask_stride[2] = Sk, a.mask_stride[3] = 1;
            if (c == 5) a.dropout_p = 0.25f, a.dropout_keep_map = D <= 128 ? (void*)4096 : nullptr;
            add(a);
          }
    a = shape(4, 1024, 1024, 12, 12, 64, TRINIX_BF16), a.causal = 1;                     // C2, C3 with dropout
    a.dropout_p = 0.1f, a.dropout_keep_map = (void*)4096, add(a);
    a = shape(1, 8192, 8192, 32, 8, 128, TRINIX_BF16), a.causal = 1;
    a.dropout_p = 0.1f, a.dropout_keep_map = (void*)4096, add(a);
    a = shape(3, 300, 77, 6, 2, 64, TRINIX_F16), a.dropout_p = 0.3f, a.dropout_keep_map = (void*)4096, add(a);
    a = shape(1, 40000, 40000, 2, 1, 64, TRINIX_BF16), a.causal = 1, a.has_window = 1;  // long, two-sided window
    a.window_left = 8192, a.window_right = 300, add(a);
    a = shape(3, 9, 70000, 32, 8, 128, TRINIX_BF16), a.causal = 1, add(a);              // decode shapes
    a = shape(16, 1, 8192, 32, 8, 128, TRINIX_BF16), add(a);
    a = shape(1, 5, 777, 8, 2, 64, TRINIX_F16), a.has_window = 1, a.window_left = 100, a.window_right = -2, add(a);
    a = shape(1, 64, 64, 8, 8, 128, TRINIX_BF16), a.has_window = 1;                       // extreme windows
    a.window_left = std::numeric_limits<int64_t>::min(), a.window_right = std::numeric_limits<int64_t>::max(), add(a);
    a.window_left = std::numeric_limits<int64_t>::max(), a.window_right = std::numeric_limits<int64_t>::min(), add(a);
    const int64_t inf = std::numeric_limits<int64_t>::max();
    for (int64_t D : {64, 128, 256})  // fp32: 16-byte and odd row strides, every split
      for (int64_t Sq : {1, 33, 128, 300})
        for (int64_t Sk : {1, 64, 257})
          for (int c = 0; c < 4; ++c) {
            a = shape(2, Sq, Sk, 4, c % 2 ? 1 : 2, D, TRINIX_F32);
            a.causal = c & 1;
            if (c >= 2) a.has_window = 1, a.window_left = 40, a.window_right = c == 3 ? inf : -5;
            if (c == 2) a.k_stride[1] += 1, a.q_stride[1] += 3;
            if (c == 3) a.mask = (void*)4096, a.mask_dtype = TRINIX_F32, a.mask_blockmap = (const uint8_t*)4096,
                        a.mask_stride[2] = Sk, a.mask_stride[3] = 1;
            add(a);
          }
    a = shape(4, 1024, 1024, 12, 12, 64, TRINIX_F32), a.causal = 1, add(a);
    a = shape(64, 1024, 1024, 16, 16, 64, TRINIX_F32), a.causal = 1, add(a);             // one wavefront per 32 rows
    a = shape(2, 700, 700, 4, 4, 128, TRINIX_F32), a.k_stride[1] = a.v_stride[1] = (1ll << 24) - 4, add(a);
    a.k_stride[1] = 1ll << 40, add(a);
    a = shape(2, 2048, 2048, 8, 4, 256, TRINIX_BF16), a.causal = 1, add(a);
    a = shape(16, 300, 300, 8, 8, 256, TRINIX_F16), a.k_stride[1] = (1ll << 22) - 8, add(a);
    a = shape(2, 2048, 2048, 16, 4, 128, TRINIX_BF16), a.causal = 1, add(a);             // dK/dV in pieces
    a = shape(1, 8192, 8192, 16, 4, 128, TRINIX_BF16), a.causal = 1, add(a);
    a = shape(2, 1000, 1000, 16, 4, 64, TRINIX_F16), add(a);
    for (const auto& f : cur) model_one(f, kAll);
    for (const char* both : {"1,1", "1,2", "2,1", "2,2"}) {  // every built split, whatever the plan takes
      setenv("TRINIX_BWD_GENERIC", both, 1);
      setenv("TRINIX_F32_KS", both, 1);
      for (size_t k = 0; k < cur.size(); k += 3)
        if (cur[k].dtype == TRINIX_F32 || cur[k].head_dim == 256) model_one(cur[k], kAll);
      unsetenv("TRINIX_F32_KS");
      unsetenv("TRINIX_BWD_GENERIC");
    }
    for (const char* pieces : {"1", "3", "20"}) {
      setenv("TRINIX_BWD_PIECES", pieces, 1);
      for (size_t k = 0; k < cur.size(); k += 2)
        if (cur[k].seqlen_q <= 2048) model_pieces(bwd_of(cur[k]));
      unsetenv("TRINIX_BWD_PIECES");
    }
    const int64_t pads[][5] = {{1, 1, 1, 1, 64}, {2, 70, 4, 36, 64}, {3, 17, 5, 80, 128}, {1, 9, 2, 63, 64}, {2, 5, 3, 160, 256}};
    for (const auto& z : pads) bounds::model_pad(BR, z[0], z[1], z[2], z[3], z[4], true);
    bounds::model_pad(BR, 1 << 19, 1 << 19, 64, 100, 128, false);
    cases += (int)cur.size();
  }
  {
    // fuzz share: 1 in 40 accepted 16-bit argument sets, sampled items
    bounds::g_sample_ends = 3, bounds::g_sample_inner = 6;
    rng = 0x1234567887654321ull;
    int ran = 0;
    for (int it = 0; it < 400000 && ran < 1500; ++it) {
      trinix_attn_fwd_args a = valid_fwd();
      a.batch = next_u64() % 3 ? (int64_t)(1 + next_u64() % 8) : rand_size();
      a.seqlen_q = next_u64() % 2 ? (int64_t)(1 + next_u64() % 20) : rand_size();
      a.seqlen_k = rand_size();
      a.nheads_kv = (int64_t)(1 + next_u64() % 8);
      a.nheads_q = a.nheads_kv * (int64_t)(1 + next_u64() % 8);
      a.head_dim = (int64_t)(64 << (next_u64() % 3));
      a.dtype = next_u64() % 2 ? TRINIX_BF16 : TRINIX_F16;
      if (next_u64() % 4 == 0) a.dtype = TRINIX_F32;
      a.causal = (int32_t)(next_u64() % 2);
      a.has_window = (int32_t)(next_u64() % 2);
      a.window_left = rand_size();
      a.window_right = rand_size();
      if (next_u64() % 2) a.window_left = (int64_t)(next_u64() % 3000) - 1000;  // small, both signs
      if (next_u64() % 2) a.window_right = (int64_t)(next_u64() % 3000) - 1000;
      const int64_t kvs = next_u64() % 2 ? a.nheads_kv * a.head_dim : (int64_t)(8 * (next_u64() % (1 << 19)));
      a.k_stride[1] = a.v_stride[1] = kvs;
      if (next_u64() % 3 == 0) {
        a.mask = (void*)4096, a.mask_dtype = (int32_t)(next_u64() % 4);
        a.mask_blockmap = next_u64() % 2 ? (const uint8_t*)4096 : nullptr;
        a.mask_stride[0] = rand_size(), a.mask_stride[1] = rand_size();
        a.mask_stride[2] = rand_size(), a.mask_stride[3] = next_u64() % 2 ? 1 : rand_size();
      }
      if (next_u64() % 4 == 0) {
        a.dropout_p = 0.1f;
        if (a.head_dim <= 128 && a.dtype != TRINIX_F32) a.dropout_keep_map = (void*)4096;
      }
      if (validate_fwd_args(&a) != TRINIX_OK) continue;
      model_one(a, 4096);
      ++ran;
    }
    cases += ran;
  }
  CHECK(pieced > 300 && generic > 500 && narrow > 1000, "modelled %ld plans in pieces, %ld generic, %ld narrow", pieced, generic, narrow);
  std::printf("bounds model: %d argument sets, %ld checks, %ld failures\n", modelled, BR.checks, BR.failures);
  failures += (int)BR.failures;
  std::printf("cases %d, fuzz accepted %d, planned %d, failures %d\n", cases, accepted, planned, failures);
  if (failures) return 1;
  std::printf("ok\n");
  return 0;
}
