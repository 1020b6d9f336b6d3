// Projection GEMM entry points (zk_gemm, zk_gemm_nt, zk_gemm_rope,
// zk_gemm_swiglu) and the rule that names a product's tile; the kernels and
// their design are in gemm_kernels.h and gemm_ring.h.  The tiled forms with a
// K-major operand are launched from gemm_kmajor.hip, the small tiles from
// gemm_ring.hip and gemm_ring_kmajor.hip.
#include <type_traits>

#include "gemm_kernels.h"

namespace zk {

// A launch's grid dimension holds fewer than 2^32 threads, a tile has 256 (the
// 512-thread ones run at most one per CU): products of more 64 x 64 tiles stay
// on the general kernel's 128 x 128.
static constexpr int64_t kMaxTiles = int64_t(1) << 24;

// Whether the 256 x 256 pipeline takes a launch: 2-byte type, M and N
// multiples of 256, K a multiple of 128 and at least 256, leading dimensions
// multiples of 8 (16-byte tile rows and stores), and every tile of an operand
// within reach of one buffer resource: 256 rows of an NT operand or 64 rows
// of a K-major one below 2 GiB (lda, ldb below 2^22 / 2^24 elements).
// Pointer alignment is checked by the caller.
static bool tiled_takes(int64_t M, int64_t N, int64_t K, int64_t lda, int a_km, int64_t ldb,
                        int b_km, int64_t ldc, int64_t ldr, int dtype) {
  if (dtype != ZK_BF16 && dtype != ZK_F16) return false;
  if (!(M > 0 && N > 0 && M % gemm::BM == 0 && N % gemm::BN == 0 && K % (2 * gemm::BK) == 0 &&
        K >= 4 * gemm::BK))
    return false;
  if (lda % 8 || ldb % 8 || ldc % 8 || ldr % 8) return false;
  const int64_t lim_a = int64_t(1) << (a_km ? 24 : 22), lim_b = int64_t(1) << (b_km ? 24 : 22);
  return lda < lim_a && ldb < lim_b;
}

// Whether the MFMA kernels whose edges are masked (the RAG form of the 256 x
// 256 pipeline, gemm_ring.h) take a launch: every 8-element run of an operand
// whole and 16-byte aligned -- N a multiple of 8 (stores), K of 8 for an
// operand along K, M of 8 for a K-major A, leading dimensions of 8 -- and
// tiles within one buffer resource (fp32: half the leading dimensions above).
// Pointer alignment is checked by the caller.
static bool masked_takes(int64_t M, int64_t N, int64_t K, int64_t lda, int a_km, int64_t ldb,
                         int b_km, int64_t ldc, int64_t ldr, int dtype) {
  if (M <= 0 || N <= 0 || K <= 0 || N % 8 || (a_km ? M : K) % 8 || (!b_km && K % 8)) return false;
  if (lda % 8 || ldb % 8 || ldc % 8 || ldr % 8 || M >= 0x7fffffffLL) return false;
  const int wide = dtype == ZK_F32 ? 1 : 0;
  const int64_t lim_a = int64_t(1) << ((a_km ? 24 : 22) - wide),
                lim_b = int64_t(1) << ((b_km ? 24 : 22) - wide);
  return lda < lim_a && ldb < lim_b && gemm::tile_count(gemm::k64, M, N) < kMaxTiles;
}

// The tile a 2-byte product runs on: the one with the least estimated time
//   launch + max((full rounds + part) (edge + steps * step), rounds * store),
// rounds of the tiles the CUs hold at once (cap workgroups each), `part` the
// share of a round's time that a partly filled last round takes, `store` what
// storing a round's tiles takes.  Constants
// in us, fitted to 372 products timed on an MI355X in every tile (32 to 4095
// tokens by the widths of the layers and heads from 1536 to 49152, forward,
// input- and weight-gradient layouts, weights not in any cache).  The choice by
// these constants alone was on average 0.3 % and at most 15 % slower than the
// best tile; that was without the 128 x 256 tile and `store`, fitted later to
// products of their own, and without the two terms for weight gradients below,
// which on purpose name a tile that is not the fastest by itself.  Examples, us
// on 256 / 128 / 128x2 / 64 / 64x128 tiles:
//   128 x 2048 x 2048 NT       42 / 26 / 21 / 11.5 / 16      (64)
//   512 x 4096 x 11008 dX     198 / 121 / 100 / 104 / 76     (64x128)
//   2048 x 2048 x 5632 NT     105 / 67 / 57 / 85 / 81        (128x2)
//   1527 x 4096 x 4096 NT      82 / 56 / 80 / 80 / 109       (128)
//   4095 x 4096 x 32000 dX    731 / 1015 / 1323 / 2839 / -   (256)
// The K-split tiles are for grids of at most one workgroup per CU, and not
// built for weight gradients, whose reduction (the tokens) is the short side.
// `half`: the 128 x 256 tile is a candidate too, again for at most one
// workgroup per CU -- products on the grid (its masked form, measured, was 4 to
// 8 % behind 128 x 128 up to K = 4096) without the SwiGLU epilogue, A along K:
//   4096 x 2048 x 8192 NT      99.7, on 128 x 128 tiles 109
//   2048 x 3072 x 16384 dX    177,   on 128 x 128 tiles 201
static gemm::Tile pick_tile(int64_t M, int64_t N, int64_t K, bool a_km, bool b_km, bool half,
                            double* cost = nullptr) {
  struct Cost {
    gemm::Tile t;
    int per_cu;
    double launch, edge, step, part, store = 0;
  };
  // store, and the four steps a 256 x 256 tile always runs: 3848 x 2744 x 24 takes
  // 14 us on 256 x 256 tiles, 9.6 on 128 x 128 and 17 on 64 x 64, where the steps
  // alone make 11, 8 and 7; gate|up of 2048 x 13952 x 64 40 / 26 / 43
  static constexpr Cost kAlongK[] = {{gemm::k256, 1, 0.5, 9.5, 1.29, 0.82},
                                     {gemm::k128x256, 1, 0.5, 5.5, 0.745, 0.72},
                                     {gemm::k128, 2, 4.7, 0.8, 0.926, 0.73, 3.6},
                                     {gemm::k128x2, 1, 0.0, 5.7, 0.59, 0.82},
                                     {gemm::k64, 2, 4.4, 0.0, 0.48, 0.60, 2.3},
                                     {gemm::k64x128, 1, 0.0, 5.1, 0.45, 0.92}};
  static constexpr Cost kKMajor[] = {{gemm::k256, 1, 4.0, 10.4, 1.31, 0.73},
                                     {gemm::k128, 2, 4.0, 3.0, 0.79, 0.59},
                                     {gemm::k64, 2, 2.9, 1.9, 0.36, 0.59}};
  if (a_km && !b_km) return gemm::k128;  // no layer product: one tile is built
  const Cost* c = a_km ? kKMajor : kAlongK;
  const int nc = a_km ? 3 : 6;
  const int64_t cus = device_cus(), steps = (K + gemm::BK - 1) / gemm::BK;
  const int64_t tiles256 = gemm::tile_count(gemm::k256, M, N);
  gemm::Tile best = gemm::k256;
  double best_us = 0;
  for (int i = 0; i < nc; ++i) {
    const int64_t n = gemm::tile_count(c[i].t, M, N), cap = cus * c[i].per_cu;
    const bool is_half = c[i].t == gemm::k128x256;
    if ((is_half || c[i].t == gemm::k128x2 || c[i].t == gemm::k64x128) && n > cus) continue;
    if (is_half && !half) continue;
    const int64_t full = n / cap, rem = n % cap;
    double part = 0;  // two per CU: a lone workgroup runs faster than a pair
    if (rem > 0)
      part = c[i].per_cu == 2 ? (rem <= cus ? c[i].part : 1.0)
                              : c[i].part + (1 - c[i].part) * static_cast<double>(rem) / cap;
    const int64_t run = i == 0 && !a_km && steps < 4 ? 4 : steps;
    double us = (c[i].edge + run * c[i].step) * (full + part);
    const double stores = c[i].store * static_cast<double>(n) / cap;
    us = c[i].launch + (us > stores ? us : stores);
    // a K-major A is a weight gradient, which runs beside the input-gradient
    // chain: the share of the chip it holds counts more than its own time
    // (a stage of 2048-wide layers 4.29 ms this way, 4.37 by time alone; the
    // line between 0.15 and 1 rests on that stage).  Layers of fewer tokens, K,
    // mostly run it in order, where its own time counts: 2048 x 2048 x 48 on 128 x
    // 128 tiles 7.3 us, on 256 x 256, which the share would name, 14.2; x 512 9.5 and
    // 16.9; a 2B layer of 512 tokens 513, with the share 530.
    if (a_km && n < cus && K >= 1024) us *= 0.15 + 0.85 * static_cast<double>(n) / cus;
    // and one of two rounds of 256 x 256 or more stays on those unless a smaller
    // tile is clearly ahead: twice the operand reads and a stream of short
    // workgroups slow the chain beside it.  5120 x 13824 x 2048: 495 us on 128 x
    // 128 tiles and 501 on 256 x 256, but the input gradient beside it takes 429
    // against 290; forward + backward of the 13B layer, 2048 tokens, 3745 / 3680
    // us, of the 14336-wide grouped-query layer, 1527 tokens, 2382 / 2350.  Below
    // two rounds the smaller tile's own time decides (1B grouped-query layer, 1024
    // tokens, 680 against 705 us), as it does more than 8 % ahead (7B, 512 tokens,
    // 908 against 925 with 20 % or no small tiles at all).
    if (a_km && i > 0 && tiles256 >= 2 * cus) us *= 1.08;
    if (i == 0 || us < best_us) {
      best = c[i].t;
      best_us = us;
    }
  }
  if (cost != nullptr) *cost = best_us;
  return best;
}

// Splitting the reduction over workgroups (gemm_split.hip): `parts` ranges of
// split_k on tiles of at most one workgroup per CU, when the estimate of the
// rule above for tiles and parts, plus the partial sums (5 us for the second
// launch, and 8 bytes an output and part, stored by one and read by the other, at
// 3.5 TB/s), is 11 us below that of
// the best single pass: a layer whose products are that short is bound by the
// host, whom the workspace and the second launch cost 7 us (a forward of the
// 2048-wide layer at 128 tokens: 112 us, 121 with its down product split, 22
// against 15 us).  A along K, 2-byte types.  Measured, us, single pass / split:
//     64 x 4096 x 11008 NT     47 /  24     64 x 2688 x 21504 dX    93 /  28
//    256 x 4096 x 22016 dX    122 /  67    512 x 5120 x 13824 NT   130 /  77
//   1024 x 2688 x 21504 dX    168 / 111   2046 x 1536 x 49152 dX   424 / 245
struct Split {
  gemm::Tile tile;
  int parts;  // 0: not split
  int64_t split_k;
};
static Split pick_split(int64_t M, int64_t N, int64_t K, bool on_grid) {
  struct Cost {
    gemm::Tile t;
    double launch, edge, step;
  };
  static constexpr Cost kCost[] = {{gemm::k256, 0.5, 9.5, 1.29},
                                   {gemm::k128x2, 0.0, 5.7, 0.59},
                                   {gemm::k64x128, 0.0, 5.1, 0.45}};
  Split best{gemm::k256, 0, 0};
  const int64_t cus = device_cus(), steps = (K + gemm::BK - 1) / gemm::BK;
  if (K < 1024 || M * N > (int64_t(1) << 24)) return best;
  double best_us = 0;
  pick_tile(M, N, K, false, false, on_grid, &best_us);
  best_us -= 11;
  for (const Cost& c : kCost) {
    const int64_t n = gemm::tile_count(c.t, M, N);
    for (int64_t p = 2; p <= 16 && n * p <= cus && steps / p >= 4; ++p) {
      const int64_t st = (steps + p - 1) / p;
      if ((steps + st - 1) / st != p) continue;  // the last range would be empty
      const double us = c.launch + c.edge + st * c.step + 5.0 + 8e-6 / 3.5 * p * M * N;
      if (us < best_us) {
        best_us = us;
        best = Split{c.t, static_cast<int>(p), st * gemm::BK};
      }
    }
  }
  return best;
}

// Which kernel a launch with 16-byte aligned pointers and no workspace takes.
struct Plan {
  bool on_grid, mfma;  // mfma false: the general kernel
  gemm::Tile tile;
};
static Plan plan_gemm(int64_t M, int64_t N, int64_t K, int64_t lda, int a_km, int64_t ldb, int b_km,
                      int64_t ldc, int64_t ldr, int dtype) {
  Plan p{tiled_takes(M, N, K, lda, a_km, ldb, b_km, ldc, ldr, dtype), false, gemm::k256};
  p.mfma = p.on_grid || masked_takes(M, N, K, lda, a_km, ldb, b_km, ldc, ldr, dtype);
  if (!p.mfma) return p;
  if (dtype == ZK_F32)
    p.tile = gemm::f32_tile(M, N);
  else if (!(a_km && !b_km && p.on_grid))
    p.tile = pick_tile(M, N, K, a_km, b_km, p.on_grid);
  return p;
}
// gate|up with the SwiGLU epilogue: N = 2 F.
static Plan plan_swiglu(int64_t M, int64_t N, int64_t K, int64_t ld_x, int64_t ld_w, int64_t ld_gu,
                        int dtype) {
  Plan p{tiled_takes(M, N, K, ld_x, 0, ld_w, 0, ld_gu, 8, dtype),
         masked_takes(M, N, K, ld_x, 0, ld_w, 0, ld_gu, 8, dtype), gemm::k256};
  if (p.mfma) p.tile = pick_tile(M, N, K, false, false, false);
  return p;
}
// mfma: the product rotates in the epilogue.
static Plan plan_rope(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc,
                      int64_t S, int64_t rot_cols, int64_t head_dim, int64_t n_pos, int dtype) {
  Plan p{tiled_takes(M, N, K, lda, 0, ldb, 0, ldc, 8, dtype), false, gemm::k256};
  if (dtype == ZK_F32 || !masked_takes(M, N, K, lda, 0, ldb, 0, ldc, 8, dtype) ||
      (head_dim != 64 && head_dim != 128) || S >= (int64_t(1) << 30) ||
      n_pos >= (int64_t(1) << 24))
    return p;
  p.tile = pick_tile(M, N, K, false, false, p.on_grid);
  // the 256-wide tile rotates whole 128-column blocks of sequences of at least
  // 128 tokens; a 64-wide one holds heads of 64 only
  if (p.tile == gemm::k256 || p.tile == gemm::k128x256)
    p.mfma = rot_cols % 128 == 0 && S >= 128;
  else
    p.mfma = p.tile != gemm::k64 || head_dim == 64;
  return p;
}
static int tile_id(const Plan& p) {
  if (!p.mfma) return ZK_TILE_GENERAL;
  switch (p.tile) {
    case gemm::k256: return p.on_grid ? ZK_TILE_256 : ZK_TILE_256_MASKED;
    case gemm::k128x256: return ZK_TILE_128X256;
    case gemm::k128: return ZK_TILE_128;
    case gemm::k128x2: return ZK_TILE_128_K2;
    case gemm::k64: return ZK_TILE_64;
    case gemm::k64x128: return ZK_TILE_64X128_K2;
  }
  return ZK_TILE_GENERAL;
}

}  // namespace zk

using namespace zk;

extern "C" int zk_gemm_nt_supported(int64_t M, int64_t N, int64_t K) {
  return M > 0 && N > 0 && M % gemm::BM == 0 && N % gemm::BN == 0 && K % (2 * gemm::BK) == 0 &&
         K >= 4 * gemm::BK;
}

extern "C" int zk_gemm_path(int64_t M, int64_t N, int64_t K, int64_t lda, int a_kmajor,
                            int64_t ldb, int b_kmajor, int64_t ldc, int64_t ldr, int dtype) {
  ZK_REQUIRE(valid_dtype(dtype), ZK_EDTYPE, "zk_gemm_path: bad dtype %d", dtype);
  return tiled_takes(M, N, K, lda, a_kmajor != 0, ldb, b_kmajor != 0, ldc, ldr < 0 ? 8 : ldr,
                     dtype)
             ? ZK_GEMM_TILED
             : ZK_GEMM_GENERAL;
}

extern "C" int zk_gemm_tile(int64_t M, int64_t N, int64_t K, int64_t lda, int a_kmajor, int64_t ldb,
                            int b_kmajor, int64_t ldc, int64_t ldr, int dtype) {
  ZK_REQUIRE(valid_dtype(dtype), ZK_EDTYPE, "zk_gemm_tile: bad dtype %d", dtype);
  return tile_id(plan_gemm(M, N, K, lda, a_kmajor != 0, ldb, b_kmajor != 0, ldc, ldr < 0 ? 8 : ldr,
                           dtype));
}

extern "C" int zk_gemm_swiglu_tile(int64_t M, int64_t F, int64_t K, int64_t ld_x, int64_t ld_w,
                                   int64_t ld_gu, int dtype) {
  ZK_REQUIRE(dtype == ZK_BF16 || dtype == ZK_F16, ZK_EDTYPE,
             "zk_gemm_swiglu_tile: 2-byte dtypes only (got %d)", dtype);
  return tile_id(plan_swiglu(M, 2 * F, K, ld_x, ld_w, ld_gu, dtype));
}

extern "C" int zk_gemm_rope_tile(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb,
                                 int64_t ldc, int64_t S, int64_t rot_cols, int64_t head_dim,
                                 int64_t n_pos, int dtype) {
  ZK_REQUIRE(valid_dtype(dtype), ZK_EDTYPE, "zk_gemm_rope_tile: bad dtype %d", dtype);
  return tile_id(plan_rope(M, N, K, lda, ldb, ldc, S, rot_cols, head_dim, n_pos, dtype));
}

namespace {

// A 2-byte product on tile t; on_grid: tiled_takes.
template <typename T, int EPI, int MB>
void launch_tiled(bool on_grid, const gemm::GemmArgs& ga, hipStream_t s) {
  const gemm::Tile t = MB == 8 ? gemm::k256 : gemm::k128x256;
  const dim3 grid(static_cast<unsigned>(gemm::tile_count(t, ga.M, ga.N)));
  if (on_grid || MB == 4)
    hipLaunchKernelGGL((gemm::gemm_tiled_kernel<T, EPI, false, false, false, MB>), grid, dim3(256),
                       0, s, ga);
  else
    hipLaunchKernelGGL((gemm::gemm_tiled_kernel<T, EPI, false, false, true, 8>), grid, dim3(256),
                       0, s, ga);
}

template <int EPI>
void launch_mfma(bool bf, gemm::Tile t, bool on_grid, int a_km, int b_km, const gemm::GemmArgs& ga,
                 hipStream_t s) {
  const bool half = t == gemm::k128x256;
  if (t != gemm::k256 && !half) {
    gemm::launch_ring(bf, EPI, a_km, b_km, t, ga, s);
    return;
  }
  if (a_km || b_km) {
    gemm::launch_tiled_kmajor(bf, a_km, b_km, !on_grid, half, ga, s);
    return;
  }
  if constexpr (EPI != 1) {
    if (half) {
      if (bf)
        launch_tiled<bf16, EPI, 4>(on_grid, ga, s);
      else
        launch_tiled<f16, EPI, 4>(on_grid, ga, s);
      return;
    }
  }
  if (bf)
    launch_tiled<bf16, EPI, 8>(on_grid, ga, s);
  else
    launch_tiled<f16, EPI, 8>(on_grid, ga, s);
}

template <typename T>
void launch_general(int a_km, int b_km, const gemm::GemmArgs& ga, hipStream_t s) {
  const int64_t nwg = ((ga.M + gemm::GBM - 1) / gemm::GBM) * ((ga.N + gemm::GBM - 1) / gemm::GBM);
  const dim3 grid(static_cast<unsigned>(nwg));
#define ZK_GEN(A, B) \
  hipLaunchKernelGGL((gemm::gemm_gen_kernel<T, A, B>), grid, dim3(256), 0, s, ga)
  if (!a_km && !b_km)
    ZK_GEN(false, false);
  else if (!a_km)
    ZK_GEN(false, true);
  else if (b_km)
    ZK_GEN(true, true);
  else
    ZK_GEN(true, false);
#undef ZK_GEN
}

}  // namespace

extern "C" int64_t zk_gemm_workspace(int64_t M, int64_t N, int64_t K, int64_t lda, int a_kmajor,
                                     int64_t ldb, int b_kmajor, int64_t ldc, int64_t ldr,
                                     int dtype) {
  if (a_kmajor || (dtype != ZK_BF16 && dtype != ZK_F16) ||
      !masked_takes(M, N, K, lda, 0, ldb, b_kmajor != 0, ldc, ldr < 0 ? 8 : ldr, dtype))
    return 0;
  const Split sp = pick_split(
      M, N, K, tiled_takes(M, N, K, lda, 0, ldb, b_kmajor != 0, ldc, ldr < 0 ? 8 : ldr, dtype));
  return sp.parts * M * N * 4;
}

extern "C" int zk_gemm(const void* a, int64_t lda, int a_kmajor, const void* b, int64_t ldb,
                       int b_kmajor, void* c, int64_t ldc, const void* r, int64_t ldr, int64_t M,
                       int64_t N, int64_t K, int dtype, zk_stream_t stream) {
  return zk_gemm_ws(a, lda, a_kmajor, b, ldb, b_kmajor, c, ldc, r, ldr, M, N, K, dtype, nullptr, 0,
                    stream);
}

extern "C" int zk_gemm_ws(const void* a, int64_t lda, int a_kmajor, const void* b, int64_t ldb,
                          int b_kmajor, void* c, int64_t ldc, const void* r, int64_t ldr,
                          int64_t M, int64_t N, int64_t K, int dtype, void* workspace,
                          int64_t workspace_bytes, zk_stream_t stream) {
  ZK_REQUIRE(valid_dtype(dtype), ZK_EDTYPE, "zk_gemm: bad dtype %d", dtype);
  ZK_REQUIRE(M >= 0 && N >= 0 && K >= 0, ZK_EINVAL, "zk_gemm: bad shape");
  const int a_km = a_kmajor != 0, b_km = b_kmajor != 0;
  // an [M, K] operand needs ld >= K, a K-major [K, M] one ld >= M
  ZK_REQUIRE(lda >= (a_km ? M : K) && ldb >= (b_km ? N : K) && ldc >= N &&
                 (r == nullptr || ldr >= N),
             ZK_EINVAL, "zk_gemm: bad leading dimension");
  if (M == 0 || N == 0) return ZK_OK;
  ZK_REQUIRE(c != nullptr && (K == 0 || (a != nullptr && b != nullptr)), ZK_EINVAL,
             "zk_gemm: null pointer");
  const int eb = dtype_bytes(dtype);
  const void* ptrs[] = {a, b, c, r};
  for (const void* p : ptrs)
    ZK_REQUIRE(p == nullptr || aligned(p, eb), ZK_EALIGN,
               "zk_gemm: operands must be aligned to their element size");
  const int64_t rows_a = a_km ? K : M, rows_b = b_km ? K : N;
  // every index the kernels form stays below 2^62
  ZK_REQUIRE(lda < (int64_t(1) << 40) && ldb < (int64_t(1) << 40) && ldc < (int64_t(1) << 40) &&
                 (r == nullptr || ldr < (int64_t(1) << 40)) && rows_a < (int64_t(1) << 40) &&
                 rows_b < (int64_t(1) << 40) && M < (int64_t(1) << 40),
             ZK_EINVAL, "zk_gemm: sizes out of range");
  const Plan pl = plan_gemm(M, N, K, lda, a_km, ldb, b_km, ldc, r ? ldr : 8, dtype);
  bool mfma = pl.mfma;
  for (const void* p : ptrs) mfma = mfma && (p == nullptr || aligned(p, 16));
  const int64_t nwg = ((M + gemm::GBM - 1) / gemm::GBM) * ((N + gemm::GBM - 1) / gemm::GBM);
  ZK_REQUIRE(nwg < 0x7fffffffLL, ZK_EINVAL, "zk_gemm: grid too large");
  gemm::GemmArgs ga{};
  ga.a = a;
  ga.lda = lda;
  ga.b = b;
  ga.ldb = ldb;
  ga.c = c;
  ga.ldc = ldc;
  ga.r = r;
  ga.ldr = ldr;
  ga.M = M;
  ga.N = N;
  ga.K = K;
  hipStream_t s = as_stream(stream);
  if (mfma && !a_km && dtype != ZK_F32 && workspace != nullptr && aligned(workspace, 16)) {
    const Split sp = pick_split(M, N, K, pl.on_grid);
    if (sp.parts > 0 && workspace_bytes >= sp.parts * M * N * 4) {
      gemm::GemmArgs part = ga;
      part.c = workspace;
      part.split_k = sp.split_k;
      gemm::launch_split(dtype == ZK_BF16, b_km, sp.tile, sp.parts, part, s);
      gemm::launch_split_sum(dtype == ZK_BF16, static_cast<const float*>(workspace), sp.parts, ga,
                             s);
      return launch_status("zk_gemm");
    }
  }
  if (mfma && dtype == ZK_F32)
    gemm::launch_ring_f32(a_km, b_km, ga, s);
  else if (mfma)
    launch_mfma<0>(dtype == ZK_BF16, pl.tile, pl.on_grid, a_km, b_km, ga, s);
  else if (dtype == ZK_BF16)
    launch_general<bf16>(a_km, b_km, ga, s);
  else if (dtype == ZK_F16)
    launch_general<f16>(a_km, b_km, ga, s);
  else
    launch_general<float>(a_km, b_km, ga, s);
  return launch_status("zk_gemm");
}

extern "C" int zk_gemm_nt(const void* a, int64_t lda, const void* b, int64_t ldb, void* c,
                          int64_t ldc, const void* r, int64_t ldr, int64_t M, int64_t N,
                          int64_t K, int dtype, zk_stream_t stream) {
  return zk_gemm(a, lda, 0, b, ldb, 0, c, ldc, r, ldr, M, N, K, dtype, stream);
}

// The q|k|v projection with the rotary embedding applied in the GEMM's
// epilogue (EPI 2) when an MFMA kernel takes the launch and its tile holds
// whole heads; otherwise zk_gemm followed by zk_rope on the rotated columns,
// which rounds the same (both run the tile pick_tile names, so the product
// before the rotation is the same too).
extern "C" int zk_gemm_rope(const void* a, int64_t lda, const void* b, int64_t ldb, void* c,
                            int64_t ldc, int64_t M, int64_t N, int64_t K, int64_t S,
                            int64_t rot_cols, int64_t head_dim, const float* cos,
                            const float* sin, int64_t n_pos, const int64_t* positions,
                            int pairing, int dtype, zk_stream_t stream) {
  ZK_REQUIRE(valid_dtype(dtype), ZK_EDTYPE, "zk_gemm_rope: bad dtype %d", dtype);
  ZK_REQUIRE(pairing == ZK_ROPE_HALF || pairing == ZK_ROPE_INTERLEAVED, ZK_EINVAL,
             "zk_gemm_rope: bad pairing %d", pairing);
  ZK_REQUIRE(M >= 0 && N >= 0 && K >= 0 && S > 0 && M % S == 0, ZK_EINVAL,
             "zk_gemm_rope: bad shape (M = %lld rows must be whole sequences of S = %lld)",
             (long long)M, (long long)S);
  ZK_REQUIRE(head_dim > 0 && head_dim % 2 == 0 && rot_cols >= 0 && rot_cols % head_dim == 0 &&
                 rot_cols <= N,
             ZK_EINVAL, "zk_gemm_rope: rotated columns %lld must be whole heads of %lld within N",
             (long long)rot_cols, (long long)head_dim);
  ZK_REQUIRE(cos != nullptr && sin != nullptr && n_pos > 0, ZK_EINVAL,
             "zk_gemm_rope: null or empty rotation table");
  ZK_REQUIRE(positions != nullptr || n_pos >= S, ZK_EINVAL,
             "zk_gemm_rope: table has %lld positions < S = %lld", (long long)n_pos, (long long)S);
  ZK_REQUIRE(lda >= K && ldb >= K && ldc >= N, ZK_EINVAL, "zk_gemm_rope: bad leading dimension");
  ZK_REQUIRE(lda < (int64_t(1) << 40) && ldb < (int64_t(1) << 40) && ldc < (int64_t(1) << 40) &&
                 M < (int64_t(1) << 40) && N < (int64_t(1) << 40),
             ZK_EINVAL, "zk_gemm_rope: sizes out of range");
  if (M == 0 || N == 0) return ZK_OK;
  ZK_REQUIRE(c != nullptr && (K == 0 || (a != nullptr && b != nullptr)), ZK_EINVAL,
             "zk_gemm_rope: null pointer");
  const Plan pl = plan_rope(M, N, K, lda, ldb, ldc, S, rot_cols, head_dim, n_pos, dtype);
  const bool epi = pl.mfma && aligned(a, 16) && aligned(b, 16) && aligned(c, 16) &&
                   aligned(cos, 16) && aligned(sin, 16);
  if (!epi) {
    const int rc = zk_gemm(a, lda, 0, b, ldb, 0, c, ldc, nullptr, 0, M, N, K, dtype, stream);
    if (rc != ZK_OK || rot_cols == 0) return rc;
    // the rotated heads as the "q" heads of a [B, S, H, d] view of c
    return zk_rope(c, S * ldc, ldc, head_dim, nullptr, 0, 0, 0, M / S, S, rot_cols / head_dim,
                   0, head_dim, cos, sin, n_pos, positions, pairing, 0, dtype, stream);
  }
  gemm::GemmArgs ga{};
  ga.a = a;
  ga.lda = lda;
  ga.b = b;
  ga.ldb = ldb;
  ga.c = c;
  ga.ldc = ldc;
  ga.M = M;
  ga.N = N;
  ga.K = K;
  ga.rcos = cos;
  ga.rsin = sin;
  ga.rpos = positions;
  ga.rnpos = n_pos;
  ga.rS = S;
  ga.rcols = rot_cols;
  ga.rhalf = static_cast<int>(head_dim / 2);
  ga.rpair = pairing;
  launch_mfma<2>(dtype == ZK_BF16, pl.tile, pl.on_grid, 0, 0, ga, as_stream(stream));
  return launch_status("zk_gemm_rope");
}

// The gate|up projection with the SwiGLU epilogue (EPI 1): replaces the two
// nn.Linear products and the activation.  K steps are whole (K % 64 == 0).
extern "C" int zk_gemm_swiglu(const void* x, int64_t ld_x, const void* w_gate,
                              const void* w_up, int64_t ld_w, void* g_out, void* u_out,
                              int64_t ld_gu, void* z, int64_t ld_z, void* zt, int64_t ld_zt,
                              int64_t M, int64_t F, int64_t K, int dtype, zk_stream_t stream) {
  ZK_REQUIRE(dtype == ZK_BF16 || dtype == ZK_F16, ZK_EDTYPE,
             "zk_gemm_swiglu: 2-byte dtypes only (got %d)", dtype);
  ZK_REQUIRE(M >= 0 && F >= 0 && K >= 0, ZK_EINVAL, "zk_gemm_swiglu: bad shape");
  ZK_REQUIRE(ld_x >= K && ld_w >= K && ld_gu >= F && ld_z >= F && (zt == nullptr || ld_zt >= M),
             ZK_EINVAL, "zk_gemm_swiglu: bad leading dimension");
  if (M == 0 || F == 0) return ZK_OK;
  ZK_REQUIRE(K > 0 && K % gemm::BK == 0, ZK_EUNSUPPORTED,
             "zk_gemm_swiglu: K must be a positive multiple of %d (got %lld)", gemm::BK,
             (long long)K);
  ZK_REQUIRE(M % 8 == 0 && F % 8 == 0, ZK_EUNSUPPORTED,
             "zk_gemm_swiglu: M and F must be multiples of 8 (got %lld, %lld)", (long long)M,
             (long long)F);
  const int64_t lds[] = {ld_x, ld_w, ld_gu, ld_z, zt ? ld_zt : 8};
  for (int64_t ld : lds)
    ZK_REQUIRE(ld % 8 == 0, ZK_EALIGN, "zk_gemm_swiglu: leading dimensions must be multiples of 8");
  const void* ptrs[] = {x, w_gate, w_up, g_out, u_out, z};
  for (const void* p : ptrs) {
    ZK_REQUIRE(p != nullptr, ZK_EINVAL, "zk_gemm_swiglu: null pointer");
    ZK_REQUIRE(aligned(p, 16), ZK_EALIGN, "zk_gemm_swiglu: operands must be 16-byte aligned");
  }
  ZK_REQUIRE(zt == nullptr || aligned(zt, 16), ZK_EALIGN,
             "zk_gemm_swiglu: operands must be 16-byte aligned");
  ZK_REQUIRE(ld_x < (int64_t(1) << 26) && ld_w < (int64_t(1) << 26), ZK_EUNSUPPORTED,
             "zk_gemm_swiglu: leading dimension out of range");
  ZK_REQUIRE(((M + 127) / 128) * ((F + 63) / 64) < 0x7fffffffLL, ZK_EINVAL,
             "zk_gemm_swiglu: grid too large");
  const Plan pl = plan_swiglu(M, 2 * F, K, ld_x, ld_w, ld_gu, dtype);
  if (!pl.mfma) {
    // rows too far apart for a tile's buffer resource: the two products and the
    // activation as separate launches
    int rc = zk_gemm(x, ld_x, 0, w_gate, ld_w, 0, g_out, ld_gu, nullptr, 0, M, F, K, dtype, stream);
    if (rc != ZK_OK) return rc;
    rc = zk_gemm(x, ld_x, 0, w_up, ld_w, 0, u_out, ld_gu, nullptr, 0, M, F, K, dtype, stream);
    if (rc != ZK_OK) return rc;
    if (zt == nullptr) return zk_swiglu_fwd(g_out, u_out, ld_gu, z, ld_z, M, F, dtype, stream);
    return zk_swiglu_fwd_t(g_out, u_out, ld_gu, z, ld_z, zt, ld_zt, M, F, dtype, stream);
  }
  gemm::GemmArgs ga{};
  ga.a = x;
  ga.lda = ld_x;
  ga.b = w_gate;
  ga.b2 = w_up;
  ga.ldb = ld_w;
  ga.c = g_out;
  ga.c2 = u_out;
  ga.ldc = ld_gu;
  ga.z = z;
  ga.ldz = ld_z;
  ga.zt = zt;
  ga.ldzt = ld_zt;
  ga.M = M;
  ga.N = 2 * F;
  ga.K = K;
  launch_mfma<1>(dtype == ZK_BF16, pl.tile, pl.on_grid, 0, 0, ga, as_stream(stream));
  return launch_status("zk_gemm_swiglu");
}
