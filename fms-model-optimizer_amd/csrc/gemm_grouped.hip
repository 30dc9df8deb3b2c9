// Grouped (mixture-of-experts) int8 GEMM: one launch over experts of uneven row counts, which only the device
// knows (offsets).
#include "gemm_launch.hpp"

namespace {

// A hundred rows per expert: the columns of a 128 x 128 tile, half its rows
struct TileHalfK { static constexpr int BM = 64, BN = 128, BK = 128, NST = 3, WGM = 2, WGN = 4; };

// The tile: rounds of tiles times what a tile takes as measured, 256 x 256 (persistent blocks) where the others are not clearly ahead (below 1024
// and K % 128 != 0 no more than that).  The host knows rows and experts, not their split, and takes every expert's last tile to be half full.
// A launch takes a round at least, however few its tiles (taken as half a one, up to a dozen tiles went to 256 x 256; us,
// -> as now: 4, 9, 130, 256 8.8 -> 3.9; 7, 949, 59, 448 24.7 -> 9.0; of 60 such launches all faster, 13.8 -> 6.2 in the mean).
// From K = 1024 on a finer estimate, for rows that fall on the experts alike, may choose another tile where 13 % are to be gained (with an eighth less
// asked for, 4, 3055, 3584, 1664 unevenly split ran 9 % longer).  With n the tiles per compute unit and s the stages of 128 bytes: one block to a unit,
// max(1, w ceil(n) + (1 - w) n) rounds of a + b s, of which a chip filled to n < 1 saves c (1 - n); two to a unit, the second one slows the first's
// stages by 1 + q; the mean over n 4 % and 1 % less and 6 % more, for the step at whole rounds.
// Parameters fitted to two thirds of 960 launches with every tile timed (4, 8, 16 experts, 128 .. 8192 rows, K and N of hidden sizes 1024 .. 4096 and
// intermediate ones to 14336), weights mostly in the last-level cache.  With weights from memory, over 1500 launches of those ranges: 0.917 of the time of the
// rounds alone in the mean, 11 of them longer by 8 % or more, 6 of those on the same tile (two runs of one differ by up to that).  us, rounds alone -> now (experts, rows,
// N, K): 8, 1643, 1152, 1792 18.4 -> 13.6; 16, 5405, 2048, 1280 34.1 -> 35.7; the longest 4, 552, 5120, 9984 64.3 -> 85.3 (128 x 128 -> 128 x 256).
enum GroupedTile { G_BIG, G_MID, G_WIDEK, G_MIDK, G_HALF, G_64, G_32, G_TILES };
struct GroupedCost { int bm, bn, units, threads; double a, b, c, w, q; };
constexpr GroupedCost GROUPED_COSTS[G_TILES] = {
    {256, 256, 1, 256, 15.66, 1.154, 0, .941, 0},    {128, 128, 2, 256, 2.315, .840, 0, .721, .409}, {128, 256, 1, 512, 5.578, .775, .254, .871, 0},
    {128, 128, 1, 512, 4.728, .460, .407, .982, 0}, {64, 128, 2, 512, 3.774, .422, 0, .554, .440},  {64, 64, 2, 256, .501, .243, 0, .610, 1.831},
    {32, 128, 2, 256, 1.680, .291, 0, .996, 1.344}};
GroupedTile pick_grouped_tile(int64_t experts, int64_t rows, int64_t N, int64_t K) {
  const double slabs = (double)K / 128;
  auto tiles = [&](int bm, int bn) {
    const double per = std::max(1.0, (double)rows / ((double)experts * bm) + 0.5);
    return (rows < experts ? (double)rows : experts * per) * div_up(N, bn);
  };
  // one block per possible tile: a launch holds less than 2^32 threads (the persistent blocks do not grow)
  auto fits = [&](GroupedTile t) {
    const GroupedCost& p = GROUPED_COSTS[t];
    return t == G_BIG || ((rows + p.bm - 1) / p.bm + experts) * div_up(N, p.bn) < (1ll << 32) / p.threads;
  };
  const double t256 = tiles(256, 256) / 256, t128 = tiles(128, 128);
  GroupedTile pick = G_BIG;
  double best = 0.95 * 0.5 * (std::max(1.0, std::ceil(t256 - 0.05)) + std::ceil(t256 + 0.05)) * (1.6 * slabs + 9);
  auto offer = [&](GroupedTile t, double cost) {
    if (cost < best && fits(t)) best = cost, pick = t;
  };
  offer(G_MID, std::max(1.0, t128 / 512) * (1.2 * slabs + 6));
  if (K % 128) return pick;  // (the others take whole 128-byte stages)
  offer(G_MIDK, std::ceil(t128 / 256) * ((t128 <= 512 ? 0.5 : 0.6) * slabs + 5));
  offer(G_64, std::max(1.0, tiles(64, 64) / 512) * (0.4 * slabs + 5));
  offer(G_32, std::max(1.0, tiles(32, 128) / 512) * (0.45 * slabs + 5));
  if (K < 1024) return pick;
  const double mean = (double)rows / experts;  // rows of an expert, of a standard deviation of sqrt(mean)
  auto below = [](double x) { return 0.5 * std::erfc(-x * M_SQRT1_2); };
  auto per_unit = [&](GroupedTile t) {  // tiles per compute unit
    const GroupedCost& p = GROUPED_COSTS[t];
    const double m = mean / p.bm, dev = std::sqrt(mean) / p.bm;
    double per = mean > 8 ? 1 : 1 - std::exp(-mean);  // row tiles of an expert: of the k-th there is one where its rows pass k bm
    if (dev > 0.5) {
      per = m + 0.5;
    } else {
      const int sure = (int)std::max(0.0, m - 6 * dev);
      per += sure;
      for (int k = sure + 1; k < m + 4 * dev; ++k) per += below((m - k) / dev);
    }
    return experts * per * div_up(N, p.bn) / 256;
  };
  auto estimate = [&](GroupedTile t) {
    const GroupedCost& p = GROUPED_COSTS[t];
    const double n0 = per_unit(t), a = p.a, b = p.b * slabs;
    double sum = 0;
    for (const double u : {0.96, 0.99, 1.06}) {
      const double n = u * n0, y = p.w * std::ceil(n) + (1 - p.w) * n;
      if (p.units == 1) sum += std::max(1.0, y) * (1 - p.c * (1 - std::min(1.0, n))) * (a + b);
      else if (n <= 1) sum += a + b;
      else if (n <= 2) sum += a * (1 + .4 * (y - 1)) + b * (1 + p.q * (y - 1));
      else sum += (1.4 * a + b * (1 + p.q)) * y / 2;
    }
    return sum / 3 + 2;
  };
  // With the weights from memory a chip half of whose units have no tile streams them slower than the estimate has it: 64 x 64 tiles, which fill it, are
  // left for 128 x 128 ones only beyond half a tile per unit, or under 16 MB of weights (3 launches, 0.92 .. 1.10), for 64 x 128 ones only beyond one per unit.
  // us, 64 x 64 | 128 x 128: 4, 239, 3712, 10240 37.7 | 53.7, 4, 229, 3968, 7936 29.6 | 39.1, 4, 558, 1792, 9344 44.5 | 51.2; of 40 launches of 72 .. 128 tiles 29
  // ran longer, by up to 42 %, and 11 shorter, by up to 14 %; of 28 of 144 and more all but two ran shorter.  Two 64 x 128 tiles of a unit stream long rows
  // against each other: 128 x 128 | 64 x 128, 16, 932, 4096, 7168 98.5 | 130.1, 8, 1073, 2432, 9472 61.0 | 76.3, 8, 1182, 2176, 3712 31.1 | 33.0, 4, 541, 4864, 2688 38.4 | 26.5.
  // For 32 x 128 tiles they come with a third tile on a part of the units, the more so where an expert's rows fit one tile of either: 32 x 128 | 64 x 128, 16, 406, 5760,
  // 4864 85.3 | 101.5, 16, 386, 4352, 6656 101 | 115, 16, 798, 4224, 6528 1.06 of the time; two to a unit, or more columns, the other way (8, 398, 7424, 5376 0.79, 16, 622, 5632, 5120 0.86).
  const bool streams = experts * N * K >= (16ll << 20);
  auto starved = [&](GroupedTile t) {
    if (pick == G_MIDK) return t == G_HALF && K > 3584;
    if (pick == G_32) return t == G_HALF && streams && per_unit(t) > 2 && (per_unit(t) <= 2.25 || (mean <= 32 && per_unit(t) < 3));
    return pick == G_64 && ((t == G_MIDK && streams && per_unit(t) <= 0.5) || (t == G_HALF && per_unit(t) <= 1));
  };
  GroupedTile other = pick;
  const double present = estimate(pick);
  double least = present;
  for (int i = G_BIG; i < G_TILES; ++i) {
    const GroupedTile t = (GroupedTile)i;
    if (t == G_MID || starved(t)) continue;  // (G_MID: offered above; as `other` it lost 7 % over five launches)
    const double cost = estimate(t);
    if (cost < least && fits(t)) least = cost, other = t;
  }
  return 1.15 * least < present ? other : pick;
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
      case G_WIDEK: g.grid_m = rows_of(TileWideK::BM); launch_tile<TileWideK, MMA_I8, true>(g, epi, st); break;
      case G_MIDK: g.grid_m = rows_of(TileMidK8::BM); launch_tile<TileMidK8, MMA_I8, true>(g, epi, st); break;
      case G_HALF: g.grid_m = rows_of(TileHalfK::BM); launch_tile<TileHalfK, MMA_I8, true>(g, epi, st); break;
      case G_MID: g.grid_m = rows_of(TileMid::BM); launch_tile<TileMid, MMA_I8, true>(g, epi, st); break;
      case G_64: g.grid_m = rows_of(TileSmallK::BM); launch_tile<TileSmallK, MMA_I8, true>(g, epi, st); break;
      case G_32: g.grid_m = rows_of(TileLowK::BM); launch_tile<TileLowK, MMA_I8, true>(g, epi, st); break;
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
  *tile_m = GROUPED_COSTS[t].bm;
  *tile_n = GROUPED_COSTS[t].bn;
  *stage = t == G_MID || (t == G_BIG && *kernel == FMSMO_PLAN_TILE_LDS_DMA) ? 64 : 128;
  return FMSMO_OK;
}
