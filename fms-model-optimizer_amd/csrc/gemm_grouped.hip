// Grouped (mixture-of-experts) int8 GEMM: one launch over experts of uneven row counts, which only the device
// knows (offsets).
#include "gemm_launch.hpp"

namespace {

// A few dozen rows per expert: the weights bound the launch, and small tiles make the blocks that stream them.
// Two blocks of either fit a compute unit.
struct Tile64 { static constexpr int BM = 64, BN = 64, BK = 128, NST = 4, WGM = 2, WGN = 2; };
struct Tile32 { static constexpr int BM = 32, BN = 128, BK = 128, NST = 4, WGM = 1, WGN = 4; };

// The tile by an estimate of the time: rounds of tiles (the host knows rows and experts, not their split:
// every expert's last tile is taken to be half full) times what a tile takes, a + b per 128 bytes of K as
// measured.  256 x 256 (persistent blocks) where the others are not clearly ahead.
// us, 256 x 256 | 128 x 128, 128-byte stages | 128 x 128, 64-byte stages | 64 x 64 | 32 x 128  (experts, rows, N, K):
//   4, 153, 3840, 1024  19.0 | 9.9 | 9.7 | 6.9 | 7.2         4, 172, 1792, 6912   64.7 | 24.1 | 29.0 | 16.3 | 16.4
//   16, 164, 8192, 1024 39.5 | 35.6 | 27.3 | 30.9 | 24.5     8, 1445, 2560, 1152  26.1 | 20.1 | 14.2 | 19.6 | 17.3
//   8, 1445, 1152, 1280 34.3 | 11.0 | 10.9 | 8.7 | 9.7       4, 1387, 3968, 4096  58.5 | 36.9 | 40.7 | 44.5 | 52.3
//   16, 1336, 1664, 5632 67.6 | 29.3 | 30.3 | 39.1 | 43.2    8, 2652, 4352, 2176  69.1 | 48.2 | 49.4 | 59.7 | 63.6
//   16, 1992, 1280, 11136 106.7 | 54.1 | 61.5 | 58.3 | 72.4  4, 1387, 8192, 3968  61.2 | 64.1 | 67.9 | 85.5 | 102.9
//   8, 4772, 2560, 12672 175 | 234 | 254 | 325 | 377         8, 8192, 4096, 14336 537 | 636 | 724 | 1012 | 1331
// A launch takes a round at least, however few its tiles (taken as half a one, up to a dozen tiles went to 256 x 256; us,
// -> as now: 4, 9, 130, 256 8.8 -> 3.9; 7, 949, 59, 448 24.7 -> 9.0; of 60 such launches all faster, 13.8 -> 6.2 in the mean).
enum GroupedTile { G_BIG, G_MIDK, G_MID, G_64, G_32 };
GroupedTile pick_grouped_tile(int64_t experts, int64_t rows, int64_t N, int64_t K) {
  const double slabs = (double)K / 128;
  auto tiles = [&](int bm, int bn) {
    const double per = std::max(1.0, (double)rows / ((double)experts * bm) + 0.5);
    return (rows < experts ? (double)rows : experts * per) * div_up(N, bn);
  };
  const double t256 = tiles(256, 256) / 256, t128 = tiles(128, 128);
  const double big = 0.5 * (std::max(1.0, std::ceil(t256 - 0.05)) + std::ceil(t256 + 0.05)) * (1.6 * slabs + 9);
  double best = 0.95 * big;
  GroupedTile pick = G_BIG;
  auto offer = [&](GroupedTile t, int bm, int bn, double cost) {
    // one block per possible tile, 256 threads each: a launch holds less than 2^32 threads (the persistent blocks do not grow)
    if (((rows + bm - 1) / bm + experts) * div_up(N, bn) >= (1 << 24)) return;
    if (cost < best) best = cost, pick = t;
  };
  offer(G_MID, 128, 128, std::max(1.0, t128 / 512) * (1.2 * slabs + 6));
  if (K % 128) return pick;  // (the others take whole 128-byte stages)
  offer(G_MIDK, 128, 128, std::ceil(t128 / 256) * ((t128 <= 512 ? 0.5 : 0.6) * slabs + 5));
  offer(G_64, 64, 64, std::max(1.0, tiles(64, 64) / 512) * (0.4 * slabs + 5));
  offer(G_32, 32, 128, std::max(1.0, tiles(32, 128) / 512) * (0.45 * slabs + 5));
  return pick;
}

bool big_is_persistent(int64_t K) { return K % 128 == 0 && use_register_staged(MMA_I8); }

template <bool REF>
int launch_grouped(const GemmArgs& g0, const float* a_scale, const float* w_scale, const void* bias, int bias_dtype,
                   int muladd, void* y, int y_dtype, int64_t ldy, hipStream_t st) {
  if (!bias) bias_dtype = FMSMO_F32;
  GemmArgs g = g0;
  const GroupedTile t = pick_grouped_tile(g.num_experts, g.M, g.N, g.K);
  auto rows_of = [&](int bm) { return div_up(g.M, bm) + g.num_experts; };  // upper bound on the row tiles
  auto run = [&](const auto& epi) {
    switch (t) {
      case G_MIDK: g.grid_m = rows_of(TileMidK::BM); launch_tile<TileMidK, MMA_I8, true>(g, epi, st); break;
      case G_MID: g.grid_m = rows_of(TileMid::BM); launch_tile<TileMid, MMA_I8, true>(g, epi, st); break;
      case G_64: g.grid_m = rows_of(Tile64::BM); launch_tile<Tile64, MMA_I8, true>(g, epi, st); break;
      case G_32: g.grid_m = rows_of(Tile32::BM); launch_tile<Tile32, MMA_I8, true>(g, epi, st); break;
      default:
        g.grid_m = rows_of(256);
        if (big_is_persistent(g.K)) launch_rs<MMA_I8, true>(g, epi, st);
        else launch_tile<TileBig, MMA_I8, true>(g, epi, st);
    }
  };
#define GO(OUT, BIAS) run(EpiDequant<OUT, BIAS, REF, int, true>{y, ldy, a_scale, w_scale, bias, 1, 1, muladd})
#define GO_BIAS(OUT)                            \
  switch (bias_dtype) {                         \
    case FMSMO_F16: GO(OUT, FMSMO_F16); break;   \
    case FMSMO_BF16: GO(OUT, FMSMO_BF16); break; \
    default: GO(OUT, FMSMO_F32); break;          \
  }
  switch (y_dtype) {
    case FMSMO_F16: GO_BIAS(FMSMO_F16) break;
    case FMSMO_BF16: GO_BIAS(FMSMO_BF16) break;
    default: GO_BIAS(FMSMO_F32) break;
  }
#undef GO
#undef GO_BIAS
  return fmsmo_check_launch();
}

}  // namespace

extern "C" int fmsmo_grouped_gemm_i8_dq(const int8_t* a, int64_t lda, const int8_t* b,
                                        int64_t ldb, int64_t ldb_e, const int32_t* offsets,
                                        int num_experts, int64_t total_rows, const float* a_scale,
                                        const float* w_scale, const void* bias, int bias_dtype,
                                        int epilogue, void* y, int y_dtype, int64_t ldy, int64_t N,
                                        int64_t K, fmsmo_stream_t stream) {
  int rc = check_gemm(a, lda, b, ldb, y, ldy, total_rows, N, K);
  if (rc) return rc;
  if (!offsets || !a_scale || !w_scale) return FMSMO_ERR_NULL;
  if (num_experts <= 0 || ldb_e < N * ldb) return FMSMO_ERR_SHAPE;
  if ((int64_t)num_experts * ldb_e >= (1ll << 40)) return FMSMO_ERR_UNSUPPORTED;
  if (K % 64 || ldb_e % 16) return FMSMO_ERR_ALIGN;
  if (y_dtype < 0 || y_dtype > 2 || (bias && (bias_dtype < 0 || bias_dtype > 2))) return FMSMO_ERR_UNSUPPORTED;
  if (epilogue < FMSMO_EPI_REF_F16 || epilogue > FMSMO_EPI_F32_MULADD) return FMSMO_ERR_UNSUPPORTED;
  if (total_rows == 0) return FMSMO_OK;
  GemmArgs g{};
  g.a = (const uint8_t*)a; g.b = (const uint8_t*)b; g.lda = lda; g.ldb = ldb;
  g.M = (int)total_rows; g.N = (int)N; g.K = (int)K;
  g.offsets = offsets; g.num_experts = num_experts; g.ldb_e = ldb_e;
  if (epilogue == FMSMO_EPI_REF_F16)
    return launch_grouped<true>(g, a_scale, w_scale, bias, bias_dtype, 0, y, y_dtype, ldy, (hipStream_t)stream);
  return launch_grouped<false>(g, a_scale, w_scale, bias, bias_dtype, epilogue == FMSMO_EPI_F32_MULADD, y, y_dtype, ldy,
                               (hipStream_t)stream);
}

extern "C" int fmsmo_grouped_gemm_plan(int num_experts, int64_t total_rows, int64_t N, int64_t K, int* kernel, int* tile_m,
                                       int* tile_n, int* stage) {
  if (!kernel || !tile_m || !tile_n || !stage) return FMSMO_ERR_NULL;
  if (num_experts <= 0 || total_rows <= 0 || N <= 0 || K <= 0 || total_rows >= (1 << 30) || N >= (1 << 30) || K >= (1ll << 31))
    return FMSMO_ERR_SHAPE;
  if (K % 64) return FMSMO_ERR_ALIGN;
  const GroupedTile t = pick_grouped_tile(num_experts, total_rows, N, K);
  *kernel = t == G_BIG && big_is_persistent(K) ? FMSMO_PLAN_TILE_REGISTER_STAGED : FMSMO_PLAN_TILE_LDS_DMA;
  *tile_m = t == G_BIG ? 256 : t == G_64 ? Tile64::BM : t == G_32 ? Tile32::BM : TileMid::BM;
  *tile_n = t == G_BIG ? 256 : t == G_64 ? Tile64::BN : t == G_32 ? Tile32::BN : TileMid::BN;
  *stage = t == G_MID || (t == G_BIG && *kernel == FMSMO_PLAN_TILE_LDS_DMA) ? 64 : 128;
  return FMSMO_OK;
}
