// Host-side launch helpers shared by the GEMM translation units (int8 and e4m3 entry points are
// compiled separately to keep the build parallel): argument checks, tile choice, launchers.
#pragma once
#include "gemm_rs.hpp"
#include "gemm_k128.hpp"
#include <algorithm>
#include <cmath>
#include <cstdlib>

using namespace fmsmo;

int fmsmo_check_launch();
// Device buffer of 6 x 64 bit that later register-staged GEMM launches of this thread fill with
// block 0's clock readings (null = off); defined in gemm.hip.
unsigned long long*& fmsmo_clock_probe();
bool fmsmo_gemv_batch_ok(int64_t M, int64_t K);
bool fmsmo_gemv_any_ok(int64_t M, int64_t N, int64_t K, bool fp8);
int fmsmo_gemv_dispatch(int op, const void* a, int64_t lda, const void* b, int64_t ldb,
                        const float* a_scale, int64_t a_scale_n, const float* w_scale,
                        int64_t w_scale_n, const void* bias, int bias_dtype, int epilogue,
                        void* y, int y_dtype, int64_t ldy, int64_t M, int64_t N, int64_t K,
                        hipStream_t st);

namespace {

bool aligned16(const void* p) { return (((uintptr_t)p) & 15) == 0; }

int check_gemm(const void* a, int64_t lda, const void* b, int64_t ldb, const void* c,
               int64_t ldc, int64_t M, int64_t N, int64_t K) {
  if (!a || !b || !c) return FMSMO_ERR_NULL;
  if (M < 0 || N <= 0 || K <= 0 || lda < K || ldb < K || ldc < N) return FMSMO_ERR_SHAPE;
  // 32-bit byte offsets inside the kernels
  if ((M > 0 && (M * lda) >= (1ll << 31)) || N * ldb >= (1ll << 31) || M >= (1 << 30) ||
      N >= (1 << 30))
    return FMSMO_ERR_UNSUPPORTED;
  if (K % 16 || lda % 16 || ldb % 16 || !aligned16(a) || !aligned16(b)) return FMSMO_ERR_ALIGN;
  return FMSMO_OK;
}

// Tile shapes.  K is consumed in stages of BK bytes; K that are no multiple of a stage run the KT
// instances of the LDS-DMA kernel (a last stage that is cut at K), see cut_k_tile.
struct TileBig { static constexpr int BM = 256, BN = 256, BK = 64, NST = 4, WGM = 2, WGN = 2; };
struct TileWide { static constexpr int BM = 128, BN = 256, BK = 64, NST = 4, WGM = 2, WGN = 2; };
struct TileMid { static constexpr int BM = 128, BN = 128, BK = 64, NST = 4, WGM = 2, WGN = 2; };
// The same tiles with stages of 128 bytes of K (whole 128-byte lines per row and request, half as
// many barriers): K % 128 == 0, one block per compute unit (128 / 120 KiB of LDS).  Pipelines of
// three stages lose a third against five; six (tall) and five (square) change nothing.
struct TileMidK { static constexpr int BM = 128, BN = 128, BK = 128, NST = 4, WGM = 2, WGN = 2; };
struct TileTallK { static constexpr int BM = 128, BN = 64, BK = 128, NST = 5, WGM = 2, WGN = 2; };
// The two with eight waves, two per SIMD, which fill each other's waits at barriers and for fragments: e4m3 and, below this K,
// int8, whose longer loops four waves run up to 3 % faster.  us, weights in the cache | from HBM, four waves -> eight:
//   128 x 128, e4m3: 777 x 4096 x 12800 47.9 -> 45.0 | 51.0 -> 49.2, 777 x 4096 x 4096 18.9 -> 17.0 | 20.5 -> 19.9, 1400 x 2560 x 1024 8.7 -> 7.0 |
//   9.7 -> 9.0; int8: 1400 x 2560 x 1024 8.2 -> 7.2 | 9.6 -> 8.7, 777 x 4096 x 4096 18.4 -> 18.2 | 20.7 -> 20.2, K = 7168 32.4 -> 32.7 | 34.2 -> 34.0,
//   12800 49.5 -> 50.0 | 51.9 -> 52.1 (2 x 4 waves instead of 4 x 2: up to 5 % behind four)
//   128 x 64, e4m3: 100 x 13824 x 5120 17.0 -> 16.4 | 27.0 -> 24.9, 1000 x 2048 x 2048 8.5 -> 7.5 | 10.4 -> 9.8; int8: 100 x 13824 x 5120 17.3 ->
//   16.9 | 25.1 -> 24.5, 2000 x 640 x 1024 6.6 -> 6.1 | 7.4 -> 7.0, 200 x 8192 x 6144 19.9 -> 20.1 | 22.6 -> 22.5, 1300 x 1280 x 8192 22.7 -> 23.3 |
//   24.5 -> 25.2
//   int8, eight waves' time over four's, in the mean of 150 launches of one round and at most, K below 1536 | 2304 | 4096 | 6144: 128 x 128
//   0.84 | 0.87 | 0.91 | 0.95, at most 1.001; 128 x 64 (from 1536 on) 0.96 | 0.98 | 1.00, at most 1.016
constexpr int I8_EIGHT_WAVES_BELOW = 6144;
struct TileMidK8 { static constexpr int BM = 128, BN = 128, BK = 128, NST = 4, WGM = 4, WGN = 2; };
struct TileTallK8 { static constexpr int BM = 128, BN = 64, BK = 128, NST = 5, WGM = 4, WGN = 2; };
// One round of 128 x 192 or 128 x 256 tiles: eight waves (two per SIMD hide each other's LDS reads and barriers), 128-byte
// stages, 160 / 144 KiB of LDS.  Three stages suffice the wider one; four waves take 1 ... 4 % longer.
struct Tile192K { static constexpr int BM = 128, BN = 192, BK = 128, NST = 4, WGM = 4, WGN = 2; };
struct TileWideK { static constexpr int BM = 128, BN = 256, BK = 128, NST = 3, WGM = 2, WGN = 4; };

// 64 x 64 tiles, two blocks per compute unit, for launches that would leave most compute units idle or take
// K slices and a second kernel.
struct TileSmallK { static constexpr int BM = 64, BN = 64, BK = 128, NST = 4, WGM = 2, WGN = 2; };
// Up to 32 rows, see use_low_tiles
struct TileLowK { static constexpr int BM = 32, BN = 128, BK = 128, NST = 4, WGM = 1, WGN = 4; };

// Which launches they take: up to one block per compute unit on reductions under 2048 (one pass takes 3.3 us + 1.6
// per 1024 of K, less than a pass of any other tile; from there on slices of two or four come close), up to 3072
// above 128 rows, under 8192 above 256 rows, whose partial sums cost more than they save, and any length above 1024
// rows, which take no slices; up to two per compute unit on short ones.  33 .. 64 tiles up to 1024 rows keep the plans they
// had, two of which the tests pin (200 x 1024 x 1536 in three slices, 300 x 520 x 1024 on 128 x 128 tiles), and not for their speed: with K < 2048
// these tiles take 0.50 ... 0.78 of the time (33 launches, int8 8.2 -> 5.4 and 9.2 -> 5.1 in those two), above 256 rows with K = 2048 .. 7680
// 1.04 (int8) and 0.87 (e4m3) in the mean of 38.  Up to 64 tokens the decode kernels re-read the activations for every 16 weight
// rows and win until there are many of those.  us from a HIP graph, int8 | e4m3, before -> these:
//   N = 6144, K = 1024: M = 100 10.4 -> 5.3; N = 2432, K = 2048: 200 10.4 -> 6.8, 400 9.0 -> 8.1; N = 4096, K = 3072:
//   200 11.6 -> 8.9 | 10.7 -> 7.5; N = 1024: K = 4096, M = 800 13.5 -> 10.6, 1000 13.6 -> 10.9; K = 5120 / 6144, M = 1000
//   16.8 / 17.9 -> 12.3 / 14.0 | 16.5 / 17.0 -> 11.0 / 13.8; N = 2048, M = 500 17.7 / 18.6 -> 12.4 / 14.5; N = 512, K = 1024:
//   800 8.9 -> 5.1, 1500 8.3 -> 5.4, 2500 8.8 -> 6.3, 4000 8.6 -> 6.8 (504 tiles).
//   N = 640, M = 1400: K = 8192 27.2 -> 18.4 | 28.8 -> 17.7, 14336 43.2 -> 28.5 | 46.3 -> 28.0.
//   Up to 64 tokens: N = 12288, K = 1024: M = 17 5.1 -> 4.9 | 5.8 -> 4.6, 40 7.4 -> 5.2, 64 8.7 -> 5.1; N = 28672: 17 9.8 ->
//   6.0, 64 15.8 -> 6.8; N = 14336, K = 4096: 17 13.4 -> 11.4, 40 18.0 -> 12.2 | 18.8 -> 11.8; N = 8192: 33 11.0 -> 10.5, 64 14.9 ->
//   10.5; kept: N = 4096, K = 4096, 33 8.9 against 9.7; N = 8192, 32 9.6 against 10.5
inline bool use_small_tiles(int64_t M, int64_t N, int64_t K) {
  if (M <= 16) return K % 128 == 0 && !fmsmo_gemv_batch_ok(M, K) && !fmsmo_gemv_any_ok(M, N, K, false);
  if (K % 128 || (K >= 8192 && M <= 1024)) return false;
  const int64_t tiles = (int64_t)div_up(M, TileSmallK::BM) * div_up(N, TileSmallK::BN);
  if (tiles > 512) return false;
  if (fmsmo_gemv_batch_ok(M, K)) return K <= (tiles > 256 ? 2048 : 4096) && tiles >= (M > 32 ? 128 : 192);
  if (tiles > 256) return K <= 1536;
  if (M <= 64 && tiles > 32 && tiles <= 64) return K <= 2304;  // (us, 128 x 64 -> these, e4m3: 48 x 2385 x 1792 8.3 -> 6.5, 64 x 3262 x 1152 7.8 -> 5.7)
  if (tiles > 64) return K < 2048 || (M > 128 && K <= 3072) || M > 256;
  return M > 1024 || (tiles <= 32 && K < 2048);
}
// The decode kernels take the launch.
inline bool use_decode(int64_t M, int64_t N, int64_t K, bool fp8) {
  return fmsmo_gemv_batch_ok(M, K) ? !use_small_tiles(M, N, K) : fmsmo_gemv_any_ok(M, N, K, fp8);
}
// Up to 32 rows and more than a round of 64 x 64 tiles, half or more of whose rows are padding: 32 x 128, half as many (us, 64 x 64 / 32 x 128, int8:
// 24 x 25197 x 1616 12.0 / 10.9, 32 x 24387 x 1216 10.1 / 8.9, 16 x 18652 x 1648 11.1 / 9.3, 32 x 19476 x 5088 37.4 / 32.0; e4m3 32 x 18142 x 2112
// 12.4 / 10.2; at 8192 .. 16384 columns the other way: 32 x 10054 x 3408 11.5 / 15.3, 8 x 14307 x 1984 8.2 / 8.5).
inline bool use_low_tiles(int64_t M, int64_t N, int64_t K) {
  return M <= 32 && N > 256 * TileSmallK::BN && (use_small_tiles(M, N, K) || !fmsmo_gemv_batch_ok(M, K));
}

// A few hundred rows through a projection whose 128 x 64 tiles fill half a round of the 256
// compute units or more run as ONE pass of those tiles rather than as K slices with a second
// kernel: no partial sums to write and read back.  A block walks K in ~0.41 us per 128-byte stage (one
// round: 4.4 us + 3.3 us per 1024 of K whatever the rows), so the slices win again on long
// reductions.  us from a HIP graph, int8, before -> after (e4m3 within 5 % of these):
//   N = 4096, K = 4096: M = 129 17.5 -> 14.7, 256 21.4 -> 17.0, 512 25.7 -> 18.3 (vendor GEMM, int32
//   out: 18.1); N = 6144: 129 20.9 -> 16.1, 256 22.1 -> 17.3; N = 2048: 512 22.6 -> 16.1, 1024 25.9 ->
//   17.5; N = 1024: 1024 21.9 -> 15.6; K = 2048, N = 4096: 129 / 256 / 512 14.4 / 18.2 / 22.9 -> 9.5 /
//   10.7 / 11.3; K = 8192: 512 36.4 -> 31.6; half a round at K = 5120 / 8192 loses (256 rows: 21.1 ->
//   22.8, 24.5 -> 29.1) and so does K = 14336 (512 rows 48.2 -> 51.3): those keep the slices.
// Above 1024 rows there are no slices and up to a round of these tiles beats what else would run (128 x 128 tiles on at
// most half the compute units) at every K: us, int8 | e4m3, N = 1280, M = 1400: K = 2048 11.6 -> 9.8 | 11.9 -> 9.5, 4096
//   17.5 -> 14.9 | 17.9 -> 14.4, 14336 46.0 -> 38.2 | 47.2 -> 35.0; N = 640, M = 2800: 11.4 -> 9.8, 17.4 -> 15.0, 45.6 -> 38.2.
inline bool use_tall_tiles(int64_t M, int64_t N, int64_t K) {
  static const char* off = getenv("FMSMO_TALL");  // FMSMO_TALL=0 disables (tuning aid)
  if (off && off[0] == '0') return false;
  if (M <= 16 || K % 128) return false;
  const int64_t tiles = (int64_t)div_up(M, TileTallK::BM) * div_up(N, TileTallK::BN);
  if (tiles > 256) return false;
  if (M > 1024) return true;
  // three quarters of a round or more: also for a single row of tiles (batches of 17 .. 128 tokens
  // that the decode kernels do not take, through a wide projection; us, M = 33 / 64 / 128: N = 14336,
  // K = 8192 39.4 / 39.6 / 42.5 -> 32.2 / 33.8 / 38.3; N = 13824, K = 5120 26.2 / 28.1 -> 20.7 / 23.2;
  // N = 14336, K = 4096, M = 65 / 128 23.7 / 25.1 -> 19.6 / 20.1)
  if (tiles >= 192) return K <= 8192;
  return M > 128 && tiles >= 96 && K <= 4096;
}

// Pick the tile shape by (relative kernel efficiency) x (fill of the last round of tiles over
// the 256 compute units).  The efficiencies are measured loop efficiencies of the shapes
// (bigger tiles move fewer bytes per MFMA); 128x128 tiles fit two blocks per CU.  Shape 3 is the
// register-staged kernel with 256x192 tiles (K % 128 == 0 only): 8 % slower per operation than
// 256x256, but e.g. N = 6144 at M = 4096 then makes 512 tiles, two full rounds, instead of 384.
// Shape 4 is the same kernel with 256x128 tiles (the tile of the probabilities x values batched
// matmul): 0.85 of the 256x256 rate where both fill their rounds (4096 x 4096 x 4096: 73 -> 85 us),
// but 2048 rows x 4096 columns make 256 tiles instead of 128 (us, int8 / e4m3: K = 4096 45.8 ->
// 43.4 / 42.2 -> 38.7, K = 12800 141 -> 123 / 130 -> 114).
// A round also costs what does not depend on K (launch, first loads, epilogue): about as much as 400 / 250 / 500 / 400 of K
// for the four other shapes over the 128 x 128 one, whose two blocks per compute unit cover it for each other.  Short
// reductions take that one where this puts it well ahead (12 %, e4m3 18 %: nearer than that the faster one is hard to
// tell), up to the K where it no longer pays (int8 1280, e4m3 640; not measured below 512).  Of 412 launches of 130 .. 4096 rows
// and 640 .. 28672 columns up to there 107 changed, by 4 % in the mean of all 412 and none more than 3.3 % slower, e4m3 61 of
// 125, 5 %, 1.7 %.  us, int8 | e4m3, K = 512: 2000 x 2560 13.7 -> 9.8 | 11.2 -> 10.1, 4000 x 2560 22.3 -> 15.4 | 19.8 -> 16.2, 1400 x
// 25600 51.1 -> 41.9 | 51.1 -> 40.6.
constexpr double EFF_RS128 = 0.85;
int pick_tile(int M, int N, int K, bool rs192_ok, bool fp8) {
  static const char* force = getenv("FMSMO_TILE");  // tuning aid: 0 = 256x256, 1 = 128x256, 2 = 128x128, 3 = 256x192, 4 = 256x128
  if (force && force[0] >= '0' && force[0] <= '4') return (force[0] == '4' && !rs192_ok) ? 2 : force[0] - '0';
  // Fitted to measurements on the Llama / Granite shapes: relative loop efficiency of the three
  // tile shapes, and a sub-linear penalty for a partially filled last round (idle CUs leave
  // power, hence clock, to the busy ones).
  const double eff[5] = {1.0, 0.76, 0.70, 0.92, EFF_RS128};
  const int bm[5] = {256, 128, 128, 256, 256}, bn[5] = {256, 256, 128, 192, 128};
  const double fixed[5] = {400, 250, 0, 500, 400};
  double scores[5];
  int best = 0;
  double best_score = -1;
  for (int t = 0; t < (rs192_ok ? 5 : 3); ++t) {
    const long tiles = (long)div_up(M, bm[t]) * div_up(N, bn[t]);
    const long slots = (t == 2 && tiles > 256) ? 512 : 256;  // two 128x128 blocks fit per CU
    const long rounds = (tiles + slots - 1) / slots;
    const double fill = (double)tiles / (double)(rounds * slots);
    const double pad = ((double)M * N) / ((double)div_up(M, bm[t]) * bm[t] * (double)div_up(N, bn[t]) * bn[t]);
    const double score = scores[t] = eff[t] * pow(fill, 0.6) * pad;
    if (score > best_score) { best_score = score; best = t; }
  }
  if (!rs192_ok) return best;
  // (Below 512 the other shapes keep the launches they had, whose edges a test counts on reaching, and not for their speed: us, int8 | e4m3, K = 256,
  // 256 x 256 -> 128 x 256: 4342 x 3185 28.1 -> 19.3 | 22.8 -> 17.8; 256 x 192 -> 128 x 256: 3627 x 5389 27.2 -> 25.4 | 25.3 -> 21.5.)
  if (K < 512) return best == 3 ? 6 : best;
  if (K <= (fp8 ? 640 : 1280)) {
    if (scores[2] > (fp8 ? 1.18 : 1.12) * best_score * (1 + fixed[best] / 4096) * K / (K + fixed[best])) best = 2;
    if (best == 2) return best;
  }
  // One round of the compute units instead of an emptier one of bigger tiles or two of smaller ones: 128 x 192 where 128 x 128
  // needs more than a round, then 128 x 256, up to (not including) the full round that 256 x 128 tiles then make too.  The
  // smaller the tile that still fits a round the shorter the round.  Of 1384 launches with more than a round of 128 x 64
  // tiles (130 .. 4096 rows, 512 .. 28672 columns, K = 512 .. 16384) 323 changed, by 20 % in the mean, one more than 2 % slower.
  // us, int8 | e4m3, 256 x 128 or two rounds of 128 x 128 -> these: K = 4096: 1000 x 6144 36.2 -> 29.6 | 33.8 -> 29.2, 500 x 12288
  // 36.4 -> 29.6 | 33.9 -> 29.2, 2000 x 3072 36.2 -> 29.3 | 33.4 -> 29.2, 700 x 8192 36.1 -> 30.6 | 31.7 -> 29.8, 1500 x 4096 36.3 -> 30.7
  // | 33.4 -> 29.5.
  if ((long)div_up(M, 128) * div_up(N, 128) > 256) {
    if ((long)div_up(M, Tile192K::BM) * div_up(N, Tile192K::BN) <= 256) return 5;
    if ((long)div_up(M, TileWideK::BM) * div_up(N, TileWideK::BN) < 256) return 6;
  }
  // What a tile of 256 rows spends ahead of its reduction and behind it, with one block on a compute unit, the two rounds or three of the
  // 128-row ones of eight waves take less than on short reductions: rounds of a + b per 128 of K, us, fitted to 347 launches each; taken
  // where a tenth is to be gained.  Up to a round of 256 x 256 tiles: with more of them their rounds overlap and the estimate
  // no longer holds.  int8 2733 x 3200 x 1024 29.3 -> 22, 3367 x 2944 x 768 28 -> 22, e4m3 2733 x 3200 x 1024 0.79 of the time; 24 launches of 694 changed, by 13 %.
  if ((best == 0 || best == 3 || best == 4) && (long)div_up(M, 256) * div_up(N, 256) <= 256) {
    static const double A[2][5] = {{17.4, 14.1, 8.9, 3.6, 4.6}, {20.3, 11.4, 7.0, 2.9, 3.7}}, B[2][5] = {{.973, .857, .834, .613, .714}, {.75, .706, .666, .601, .823}};
    auto cost = [&](int i, int rows, int cols) {
      return std::ceil((double)div_up(M, rows) * div_up(N, cols) / 256) * (A[fp8][i] + B[fp8][i] * (K / 128));
    };
    const double now = best == 0 ? cost(0, 256, 256) : best == 3 ? cost(1, 256, 192) : cost(2, 256, 128);
    const double c192 = cost(3, 128, 192), cwide = cost(4, 128, 256);
    const bool full = best == 4 && (long)div_up(M, 256) * div_up(N, 128) > 230;  // (a full round of 256 x 128, see above)
    if (!full && 1.1 * std::min(c192, cwide) < now) return c192 < cwide ? 5 : 6;
  }
  return best;
}

template <class Tile, int OP, bool GROUPED, bool KT = false, class Epi>
void launch_tile(const GemmArgs& g0, const Epi& epi, hipStream_t st) {
  GemmArgs g = g0;
  g.grid_n = div_up(g.N, Tile::BN);
  if (!GROUPED) g.grid_m = div_up(g.M, Tile::BM);
  g.group_m = 4;
  dim3 grid((unsigned)(g.grid_m * g.grid_n)), block(Tile::WGM * Tile::WGN * 64);
  hipLaunchKernelGGL(
      (gemm_tile_kernel<Tile::BM, Tile::BN, Tile::BK, Tile::NST, Tile::WGM, Tile::WGN, OP, 1,
                        GROUPED, Epi, KT>),
      grid, block, 0, st, g, epi);
}

// 256x256 tiles with K a multiple of 128 run the register-staged pipeline (gemm_rs.hpp: whole
// 128-byte lines, half the L2 -> L1 traffic).  FMSMO_RS=0 / 1 forces the choice for tuning.
static bool use_register_staged(int op) {
  static const char* force = getenv("FMSMO_RS");
  if (force && (force[0] == '0' || force[0] == '1')) return force[0] == '1';
  (void)op;
  return true;
}
// Compute units of the current device (the grid of the persistent blocks).
inline int compute_units() {
  static thread_local int cached_dev = -1, cached = 0;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = 0;
  if (dev != cached_dev) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 256;
    cached_dev = dev;
    cached = cus;
  }
  return cached;
}

template <int OP, bool GROUPED = false, int BN = 256, class Epi>
void launch_rs(const GemmArgs& g0, const Epi& epi, hipStream_t st) {
  GemmArgs g = g0;
  g.clk = fmsmo_clock_probe();
  g.grid_n = div_up(g.N, BN);
  if (!GROUPED) g.grid_m = div_up(g.M, 256);
  g.group_m = 4;
  dim3 grid((unsigned)(g.grid_m * g.grid_n)), block(256);
  // mixture-of-experts mode: grid_m is only an upper bound on the row tiles (the row counts live
  // on the device); the blocks are persistent, one per compute unit, and count the tiles themselves
  if (GROUPED && g.rows_per_group == 0) grid.x = (unsigned)std::min<long>((long)grid.x, compute_units());
  if constexpr (OP == MMA_FP8) {
    // e4m3: the 16 x 16 x 128 matrix instruction (more work per joule under the power limit: the
    // four Llama-3-8B shapes at 4096 rows +1 ... +4 %) unless FMSMO_MFMA16=0 asks for 32 x 32 x 64
    // (tuning aid).  int8 stays with 32 x 32 x 32: its 16 x 16 x 64 form issues four times as many
    // instructions per slab and lost 3 ... 25 % in this kernel.
    static const char* force16 = getenv("FMSMO_MFMA16");
    if (!(force16 && force16[0] == '0')) {
      hipLaunchKernelGGL((gemm_rs_kernel<OP, Epi, GROUPED, BN, true>), grid, block, 0, st, g, epi);
      return;
    }
  }
  hipLaunchKernelGGL((gemm_rs_kernel<OP, Epi, GROUPED, BN, false>), grid, block, 0, st, g, epi);
}

// Reduction of exactly 128 bytes (attention scores): persistent blocks over 128 x 256 tiles, two
// per compute unit (FMSMO_K128_BLOCKS sets the grid, for tuning).
template <int OP, class Epi>
void launch_k128(const GemmArgs& g0, int batch, int M, const Epi& epi, hipStream_t st) {
  GemmArgs g = g0;
  g.grid_n = div_up(g.N, 256);
  g.grid_m = batch * div_up(M, 128);
  g.group_m = 4;
  static const int env_blocks = getenv("FMSMO_K128_BLOCKS") ? atoi(getenv("FMSMO_K128_BLOCKS")) : 0;
  const long tiles = (long)g.grid_m * g.grid_n;
  long blocks = env_blocks > 0 ? env_blocks : 512;
  if (blocks > tiles) blocks = tiles;
  hipLaunchKernelGGL((gemm_k128_kernel<OP, Epi>), dim3((unsigned)blocks), dim3(256), 0, st, g, epi);
}

// Up to 256 rows in one pass beside use_small_tiles and use_tall_tiles: 64 x 64 tiles up to a round of them, 128 x 64 ones up to a round (us, slices or 128 x
// 128 tiles before -> these, 64 x 64: int8 64 x 8461 x 2816 15.2 -> 9.5, 100 x 5021 x 3200 14.1 -> 10.2, 128 x 1808 x 2176 10.5 -> 8.1, 24 x 8696 x 6016 24.4 ->
// 19.5, 24 x 10874 x 7936 30.9 -> 25.0, 64 x 6923 x 3200 13.3 -> 10.1; 128 x 64: e4m3 100 x 8924 x 2816 16.9 -> 10.3, 100 x 11835 x 3584 21.7 -> 15.5).
enum FewRows { FEW_NONE, FEW_SMALL, FEW_TALL };
inline FewRows a_few_rows(int64_t M, int64_t N, int64_t K) {
  if (M > 256 || K % 128) return FEW_NONE;
  if ((int64_t)div_up(M, TileSmallK::BM) * div_up(N, TileSmallK::BN) <= 256) return K < 8192 ? FEW_SMALL : FEW_NONE;
  return (int64_t)div_up(M, TileTallK::BM) * div_up(N, TileTallK::BN) <= 256 ? FEW_TALL : FEW_NONE;
}

// K % 128 != 0: the KT instances (a last stage that is cut at K).  The tile by an estimate of the time: rounds of tiles times
// what a tile takes, a + b per 128 bytes of K, fitted to 520 launches of 65 .. 4096 rows, 256 .. 28672 columns and K = 512 .. 16384 with every
// tile timed; a partly filled last round and a half empty chip count between their fraction and a whole one.  Over those launches the tiles chosen
// take 0.854 (int8), 0.833 (e4m3) and 0.877 (fp16 instruction) of the time of the three shapes that served all of them before (128 x 64, 128 x 128 of
// four waves, 256 x 256), the best tile of each launch 0.849 / 0.825 / 0.871; 256 x 256 by 114
// more launches of 4000 columns and up (e4m3 3623 x 23627 x 4544 398, 128 x 256 475).  us, int8, before -> now: 2006 x 10495 x 1328 69.1 -> 56.4, 712 x 22911 x
// 3024 113.7 -> 85.9, 2517 x 4095 x 1456 40.2 -> 31.5, 373 x 711 x 1904 10.9 -> 8.2, 1671 x 262 x 14112 48.4 -> 34.9, 91 x 6131 x 9456 48.2 -> 30.4.
enum CutTile { CUT_SMALL, CUT_TALL, CUT_MID, CUT_192, CUT_WIDE, CUT_BIG, CUT_LOW };
struct CutCost { double a, b; };
constexpr CutCost CUT_COSTS[3][6] = {
    {{2.3, .261}, {3.2, .430}, {3.8, .631}, {5.4, .807}, {7.0, .967}, {15.8, 1.6}},  // int8
    {{2.1, .225}, {2.7, .356}, {3.5, .516}, {4.7, .717}, {6.3, .966}, {15.8, 1.38}},  // e4m3
    {{2.5, .377}, {3.4, .551}, {4.6, .824}, {5.8, 1.16}, {7.1, 1.48}, {0, 0}}};       // e4m3, K % 64 != 0
inline CutTile cut_k_tile(int64_t M, int64_t N, int64_t K, int op) {
  const int kind = op == MMA_I8 ? 0 : op == MMA_FP8 ? 1 : 2;
  const int bm[6] = {64, 128, 128, 128, 128, 256}, bn[6] = {64, 64, 128, 192, 256, 256};
  if (use_low_tiles(M, N, K)) return CUT_LOW;
  const double stages = (double)((K + 127) / 128);
  CutTile best = CUT_BIG;
  double least = HUGE_VAL;
  for (int t = 0; t < (kind == 2 ? 5 : 6); ++t) {
    const double a = CUT_COSTS[kind][t].a, b = CUT_COSTS[kind][t].b * stages;
    const double n = (double)div_up(M, bm[t]) * div_up(N, bn[t]) / 256, whole = std::ceil(n);
    // (two 64 x 64 tiles to a unit on a long reduction: int8 314 x 5681 x 15312 103, 128 x 128 92)
    if (t == CUT_SMALL && n > 1 && K >= 8192) continue;
    double cost;
    if (t == CUT_SMALL) cost = n <= 1 ? a + b : (1.4 * a + 1.8 * b) * whole / 2;  // (two of these share a compute unit)
    else cost = std::max(1.0, 0.72 * whole + 0.28 * n) * (a + b) * (1 - 0.25 * (1 - std::min(1.0, n)));
    if (t == CUT_BIG && kind == 1) cost *= n > 2.25 ? 0.92 : n <= 1 ? 1.1 : 1;
    if (cost < least) least = cost, best = (CutTile)t;
  }
  return best;
}
template <int OP, class Epi>
void launch_cut_k(const GemmArgs& g, const Epi& epi, hipStream_t st) {
  const CutTile t = cut_k_tile(g.M, g.N, g.K, OP);
  if constexpr (OP == MMA_I8) {  // (long reductions on four waves, as with whole stages)
    if (t == CUT_TALL && g.K >= I8_EIGHT_WAVES_BELOW) return launch_tile<TileTallK, OP, false, true>(g, epi, st);
    if (t == CUT_MID && g.K >= I8_EIGHT_WAVES_BELOW) return launch_tile<TileMidK, OP, false, true>(g, epi, st);
  }
  switch (t) {
    case CUT_SMALL: launch_tile<TileSmallK, OP, false, true>(g, epi, st); break;
    case CUT_TALL: launch_tile<TileTallK8, OP, false, true>(g, epi, st); break;
    case CUT_MID: launch_tile<TileMidK8, OP, false, true>(g, epi, st); break;
    case CUT_192: launch_tile<Tile192K, OP, false, true>(g, epi, st); break;
    case CUT_WIDE: launch_tile<TileWideK, OP, false, true>(g, epi, st); break;
    case CUT_LOW: launch_tile<TileLowK, OP, false, true>(g, epi, st); break;
    default:
      if constexpr (OP != MMA_FP8_F16) {
        if (g.K % 64 == 0) launch_tile<TileBig, OP, false>(g, epi, st);  // (64-byte stages: whole)
        else if constexpr (OP == MMA_I8) launch_tile<TileBig, OP, false, true>(g, epi, st);
      }
  }
}

template <int OP, class Epi>
void launch_any(const GemmArgs& g, const Epi& epi, hipStream_t st) {
  if constexpr (OP == MMA_FP8_F16) {
    launch_cut_k<OP>(g, epi, st);
  } else if (g.K % 128) {
    launch_cut_k<OP>(g, epi, st);
  } else if (use_low_tiles(g.M, g.N, g.K)) {
    launch_tile<TileLowK, OP, false>(g, epi, st);
  } else if (use_small_tiles(g.M, g.N, g.K)) {
    launch_tile<TileSmallK, OP, false>(g, epi, st);
  } else if (use_tall_tiles(g.M, g.N, g.K)) {
    if (OP != MMA_I8 || g.K < I8_EIGHT_WAVES_BELOW) launch_tile<TileTallK8, OP, false>(g, epi, st);
    else if constexpr (OP == MMA_I8) launch_tile<TileTallK, OP, false>(g, epi, st);
  } else if (const FewRows few = a_few_rows(g.M, g.N, g.K)) {
    if (few == FEW_SMALL) launch_tile<TileSmallK, OP, false>(g, epi, st);
    else launch_tile<TileTallK8, OP, false>(g, epi, st);
  } else {
    switch (pick_tile(g.M, g.N, g.K, use_register_staged(OP), OP != MMA_I8)) {
      case 0:
        if (use_register_staged(OP)) launch_rs<OP>(g, epi, st);
        else launch_tile<TileBig, OP, false>(g, epi, st);
        break;
      case 1: launch_tile<TileWide, OP, false>(g, epi, st); break;
      case 3:
        if (use_register_staged(OP)) launch_rs<OP, false, 192>(g, epi, st);
        else launch_tile<TileBig, OP, false>(g, epi, st);
        break;
      case 4: launch_rs<OP, false, 128>(g, epi, st); break;  // 4 .. 6 only offered beside the register-staged kernel
      case 5: launch_tile<Tile192K, OP, false>(g, epi, st); break;
      case 6: launch_tile<TileWideK, OP, false>(g, epi, st); break;
      default:
        // one round of 128 x 128 tiles: stages of 128 bytes (us, 1024 rows, N = 4096: K = 4096 29.0 ->
        // 25.6, 5120 36.8 -> 31.2; 512 rows, N = 6144, K = 4096: 28.0 -> 23.5); more than a round keeps
        // the 64-byte stages, whose blocks fit two to a compute unit
        if ((long)div_up(g.M, TileMidK::BM) * div_up(g.N, TileMidK::BN) <= 256) {
          if (OP != MMA_I8 || g.K < I8_EIGHT_WAVES_BELOW) launch_tile<TileMidK8, OP, false>(g, epi, st);
          else if constexpr (OP == MMA_I8) launch_tile<TileMidK, OP, false>(g, epi, st);
        } else {
          launch_tile<TileMid, OP, false>(g, epi, st);
        }
        break;
    }
  }
}

// A last round of 256x256 tiles that fills at most a quarter of the compute units costs most of
// a round.  Columns to cut off so that the remaining tiles make full rounds (0 = leave the GEMM
// whole); the cut columns then run as a second, small GEMM with the tile shape that suits them.
// Taken only when at least 1024 columns are cut: a narrower second GEMM is a latency-bound launch
// that costs as much as the sparse round it replaces (us, whole -> cut: 2048 x 25600 x 4096, 32
// tiles over 3 rounds, int8 263 -> 248, e4m3 224 -> 204; 4096 x 8448 x 8192, 16 tiles over 2
// rounds, one column tile cut: 316 -> 321).  FMSMO_TAIL_SPLIT=0 switches this off (tuning aid).
inline int tail_split_columns(int M, int N, int K, bool fp8) {
  static const char* off = getenv("FMSMO_TAIL_SPLIT");
  if (off && off[0] == '0') return 0;
  if (K % 128 || !use_register_staged(0) || pick_tile(M, N, K, true, fp8) != 0) return 0;
  const long gm = div_up(M, 256), gn = div_up(N, 256), tiles = gm * gn;
  if (tiles <= 256) return 0;
  const long last = tiles % 256;
  if (last == 0 || last > 64) return 0;
  const long cut = (last + gm - 1) / gm;  // column tiles
  if (cut < 4 || cut >= gn) return 0;
  return (int)(N - (gn - cut) * 256);
}

template <int OP, bool REF, class AccT>
int launch_dq(const GemmArgs& g, const float* a_scale, int a_stride, const float* w_scale,
              int w_stride, const void* bias, int bias_dtype, void* y, int y_dtype, int64_t ldy,
              hipStream_t st, bool may_split = true, int muladd = 0) {
  if (!bias) bias_dtype = FMSMO_F32;
  const int tail = may_split ? tail_split_columns(g.M, g.N, g.K, OP != MMA_I8) : 0;
  if (tail > 0) {
    const int64_t n0 = g.N - tail;
    GemmArgs g1 = g, g2 = g;
    g1.N = (int)n0;
    g2.N = tail;
    g2.b = g.b + n0 * g.ldb;
    const int64_t ysz = y_dtype == FMSMO_F32 ? 4 : 2, bsz = bias_dtype == FMSMO_F32 ? 4 : 2;
    int rc = launch_dq<OP, REF, AccT>(g1, a_scale, a_stride, w_scale, w_stride, bias, bias_dtype,
                                             y, y_dtype, ldy, st, false, muladd);
    if (rc) return rc;
    return launch_dq<OP, REF, AccT>(
        g2, a_scale, a_stride, w_scale + (w_stride ? n0 : 0), w_stride,
        bias ? (const void*)((const char*)bias + n0 * bsz) : nullptr, bias_dtype,
        (void*)((char*)y + n0 * ysz), y_dtype, ldy, st, false, muladd);
  }
#define GO(OUT, BIAS)                                                                         \
  {                                                                                           \
    EpiDequant<OUT, BIAS, REF, AccT, OP == MMA_I8 || OUT == FMSMO_F32> epi{y, ldy, a_scale, w_scale, bias, a_stride, w_stride, muladd}; \
    launch_any<OP>(g, epi, st);                                                               \
  }
#define GO_BIAS(OUT)                            \
  switch (bias_dtype) {                         \
    case FMSMO_F16: GO(OUT, FMSMO_F16) break;   \
    case FMSMO_BF16: GO(OUT, FMSMO_BF16) break; \
    default: GO(OUT, FMSMO_F32) break;          \
  }
  switch (y_dtype) {
    case FMSMO_F16: GO_BIAS(FMSMO_F16) break;
    case FMSMO_BF16: GO_BIAS(FMSMO_BF16) break;
    case FMSMO_F32: GO_BIAS(FMSMO_F32) break;
    default: return FMSMO_ERR_UNSUPPORTED;
  }
#undef GO
#undef GO_BIAS
  return fmsmo_check_launch();
}

int check_dq(const float* a_scale, int64_t a_scale_n, const float* w_scale, int64_t w_scale_n,
             const void* bias, int bias_dtype, int y_dtype, int64_t M, int64_t N) {
  if (!a_scale || !w_scale) return FMSMO_ERR_NULL;
  if ((a_scale_n != 1 && a_scale_n != M) || (w_scale_n != 1 && w_scale_n != N)) return FMSMO_ERR_SHAPE;
  if (y_dtype < 0 || y_dtype > 2 || (bias && (bias_dtype < 0 || bias_dtype > 2))) return FMSMO_ERR_UNSUPPORTED;
  return FMSMO_OK;
}

}  // namespace

// ---------------------------------------------------------------------------------- split K
// Few output tiles and a long reduction (a batch of tens to hundreds of tokens through a
// projection with few output columns) leave most compute units idle: 17 x 4096 x 14336 is 32 tiles
// of 128 x 128.  With a caller-provided workspace the reduction is cut into slices that run as
// the uniform "groups" of the grouped kernels (A and B advance along K per group, the partial
// sums of group s land in rows [s M, (s + 1) M) of the workspace) and a second kernel adds the
// slices in a fixed order and applies the dequantizing epilogue.  int32 partial sums are exact, so
// the int8 result is bit-identical to the single-pass one.
namespace {

struct SplitPlan {
  int splits;
  int64_t k_len, ws_bytes;
  bool rs;  // 256 x 128 tiles of the register-staged kernel instead of 128 x 128 LDS-DMA tiles
  bool tall = false;  // 128 x 64 tiles with 128-byte stages
  bool cut = false;   // the last slice is shorter than k_len (KT instances of the tall and the small tiles)
  bool small = false; // 64 x 64 tiles with 128-byte stages
};

// K in `s` slices of whole 128-byte stages of at least 1024 bytes on 128 x 64 tiles, the last one shorter
inline bool cut_slices(SplitPlan& p, int64_t M, int64_t N, int64_t K, int s) {
  s = (int)std::min<int64_t>(s, K / 1024);
  if (s < 2) return false;
  p.k_len = ((K + s - 1) / s + 127) / 128 * 128;
  p.splits = (int)((K + p.k_len - 1) / p.k_len);
  p.ws_bytes = (int64_t)p.splits * M * N * 4;
  p.tall = p.cut = true;
  return true;
}

// `limit` > 0: the workspace at hand; a plan that needs more is passed over for the next one (the
// register-staged slices need more partial sums than the 128 x 128 ones: more, shorter slices) or
// takes as many slices as there is room for.
inline SplitPlan plan_split_k(int64_t M, int64_t N, int64_t K, int64_t limit = 0, bool fp8 = false) {
  SplitPlan p{1, K, 0, false};
  static const char* off = getenv("FMSMO_SPLIT_K");  // FMSMO_SPLIT_K=0 disables (tuning aid)
  if (off && off[0] == '0') return p;
  if (M <= 16 || M > 1024 || use_small_tiles(M, N, K) || use_tall_tiles(M, N, K) || use_low_tiles(M, N, K)) return p;
  const int64_t tiles_t = (int64_t)div_up(M, TileTallK::BM) * div_up(N, TileTallK::BN);
  const int64_t room = limit > 0 ? limit / (M * N * 4) : 256;
  const int64_t tiles_s = (int64_t)div_up(M, TileSmallK::BM) * div_up(N, TileSmallK::BN);
  // Up to 256 rows one pass of the tiles of a_few_rows takes less than slices and their sums do: of 33 64 x 64 tiles or more below K = 4096, of 129 or more
  // below 6144 (where slices of 128 x 64 tiles would be but two), of more than a round always.  (int8 at K = 2048, up to 128 tiles, and 4096, where tests
  // count on slices, keeps them, and not for their speed.)  With the weights from HBM a pass of few tiles has too few loads in flight: then below
  // K = 3072 up to 64 rows, or up to 72 tiles, and below 3584 up to 128 tiles (us, one pass | slices, e4m3: 40 x 2176 x 3968 17.4 | 13.7, 40 x 4096 x 3072 15.3 |
  // 13.8, 32 x 6784 x 3584 17.2 | 16.2, 64 x 2176 x 2560 14.2 | 13.8, 64 x 8192 x 2560 15.3 | 16.8, 80 x 2176 x 3328 15.5 | 14.3, 128 x 4096 x 3328 16.1 | 17.7, 80 x
  // 5504 x 6912 26.7 | 23.8, 80 x 5504 x 4608 20.0 | 19.8, 128 x 5504 x 4608 20.6 | 21.2; int8 40 x 2176 x 3968 16.5 | 13.5, 64 x 4096 x 3584 16.1 | 15.5).
  const int64_t one_pass_below = M > 128 || tiles_s > 128 ? 4096 : M <= 64 || tiles_s <= 72 ? 3072 : 3584;
  if (M <= 256 && K % 128 == 0 && (tiles_s > 256 || (tiles_s > (fp8 || K > 2048 ? 32 : 128) && K >= 2048 && K < one_pass_below) ||
                                   (M <= 128 && tiles_s > 128 && tiles_t > 64 && K < 6144 && K >= (fp8 ? 4096 : 4224))))
    return p;
  if (K % 128 == 0 && tiles_s <= 32 && K > 2048) {
    // Few tiles: slices on 64 x 64 ones, four (eight of a long reduction: from then on the partial sums cost more
    // than a shorter pass saves).  us, slices of 128 x 64 tiles -> these, M = 100, N = 1024: K = 3072 8.7 -> 6.9, 4096 9.2 ->
    // 7.2, 6144 9.9 -> 8.0, 8192 9.8 -> 8.8, 14336 13.7 -> 10.8 (four: 11.2); N = 256, K = 4096 8.2 -> 6.9; 40 x 512 x 9344
    // 10.3 -> 9.3; e4m3 within 3 % of these
    const int want = (int)std::min<int64_t>(K >= 12288 ? 8 : 4, room);
    if (want >= 2) {
      p.k_len = ((K + want - 1) / want + 127) / 128 * 128;
      p.splits = (int)((K + p.k_len - 1) / p.k_len);
      p.ws_bytes = (int64_t)p.splits * M * N * 4;
      p.small = true;
      p.cut = K % p.k_len != 0;
      return p;
    }
  }
  if (K % 128) {
    // (us, one pass -> slices, M = 40: N = 1024, K = 4016 13.1 -> 8.8; N = 3072 13.6 -> 10.3; M = 100,
    // N = 3072, K = 8208 26.3 -> 14.4; M = 200, N = 1500, K = 11216 36.7 -> 16.7.  From a quarter of a
    // round of tiles on these shapes ask for no workspace, nor up to where one pass of 64 x 64 tiles takes as long: int8 177 x 301 x 3936
    // 10.9 against 11.0, 169 x 768 x 2848 10.1 against 8.9; e4m3, K % 64 != 0, 68 x 474 x 3424 11.6 against 14.5.)
    // With the weights from HBM up to 128 rows over more than 24 such tiles begin earlier (int8, one pass | slices: 41 x 3467 x 3120 18.8 | 15.8, 44 x 1673 x 3424 17.2 | 13.9,
    // 123 x 2739 x 3504 21.0 | 19.0, up to 64 rows over more than 36 47 x 2369 x 2960 16.7 | 15.1, 56 x 3671 x 2544 17.8 | 16.7; 35 x 3278 x 2448 1.04; in one pass 47 x
    // 2090 x 2704 0.91 of the time, 109 x 866 x 3264 0.83).
    const int64_t above = fp8 ? (K % 64 ? 2816 : 3584) : M <= 64 && tiles_t > 36 ? 2496 : M <= 128 && tiles_t > 24 ? 3072 : 3584;
    if (tiles_t < 64 && K > above) cut_slices(p, M, N, K, (int)std::min<int64_t>(256 / tiles_t, room));
    return p;
  }
  // Long reductions under a few hundred rows: 256 x 128 tiles of the register-staged kernel carry
  // the slices (us, 128 x 128 LDS-DMA tiles -> these, N = 4096, K = 14336: M = 384 51.4 -> 49.0,
  // 512 54.6 -> 48.3, 768 84.7 -> 68.2, 1024 87.6 -> 77.8; at K = 4096 they lose, M = 512 25.5 ->
  // 27.7, and below 384 rows their 256-row tiles are half empty)
  if (K >= 8192 && M >= 384 && use_register_staged(0)) {
    const int64_t t = (int64_t)div_up(M, 256) * div_up(N, 128);
    // 129 .. 256 tiles of 128 x 128 fill most of a round of the compute units in one pass with 128-byte
    // stages, without partial sums.  e4m3 is faster so throughout; int8 where the round is nearly full
    // or K short, else only with the weights in the last-level cache (us with weights from HBM, slices ->
    // one pass, int8 | e4m3: 777 x 4096 x 12800, 224 tiles, 64.1 -> 52.5 | 74.3 -> 53.0; 896 x 4096 x 14336,
    // 224, 68.0 -> 65.0 | 81.2 -> 65.1; 700 x 4096 x 8192, 192, 40.5 -> 32.8 | 48.8 -> 33.0; 1000 x 2304 x
    // 9216, 144, 36.3 -> 30.2 | 42.1 -> 31.8; 640 x 4096 x 14336, 160, 60.1 -> 64.4 | 73.5 -> 67.5; 640 x 5120
    // x 13824, 200, 63.6 -> 68.2 | 76.1 -> 68.4; 600 x 4352 x 11008, 170, 48.5 -> 52.1 | 58.8 -> 51.3;
    // 1024 x 4096 x 14336, 256, 80.0 -> 72.5; 512 x 7168, 224: K = 10240 63.8 -> 57.5, 12288 66.5 -> 67.3,
    // 14336 78.7 -> 75.2, 16384 83.1 -> 80.2; of 58 shapes with 224 .. 256 tiles and K = 10240 .. 16384 56 gained
    // up to 17 %, two lost 1 %)
    const int64_t t128 = (int64_t)div_up(M, TileMidK::BM) * div_up(N, TileMidK::BN);
    if (t128 > 128 && t128 <= 256 && (fp8 || t128 >= 224 || K <= 9216)) return p;
    if (t <= 128) {
      int s = (int)(256 / t);
      while (s > 1 && (K % (s * 128) != 0 || K / s < 512)) --s;
      if (s >= 2 && (limit <= 0 || (int64_t)s * M * N * 4 <= limit)) {
        p.splits = s;
        p.k_len = K / s;
        p.ws_bytes = (int64_t)s * M * N * 4;
        p.rs = true;
        return p;
      }
    }
  }
  // Slices of at least 1024 on 128 x 64 tiles with 128-byte stages: twice the blocks of the
  // 128 x 128 tiles for the same partial sums, or the same blocks for half of them (us, 128 x 128
  // tiles with 64-byte stages -> these, M = 65 / 100 / 128: N = 4096, K = 4096 15.8 / 16.9 / 16.5 ->
  // 13.4 / 14.2 / 14.9; N = 2048 13.2 / 13.5 / 11.9 -> 9.4 / 9.9 / 9.7; N = 1000 12.6 / 13.0 / 12.7 ->
  // 10.3 / 10.8 / 10.7; N = 4096, K = 2048 12.8 / 14.4 / 13.6 -> 10.1 / 11.5 / 11.4; K = 5120 17.3 /
  // 19.4 / 17.9 -> 13.8 / 15.5 / 16.3; K = 8192 18.9 / 19.6 / 18.3 -> 17.4 / 18.5 / 17.2; N = 1024,
  // K = 8192 14.3 / 14.6 / 13.1 -> 10.6 / 11.2 / 11.2; K = 14336, N = 4096, M = 33 / 128 / 256 22.7 /
  // 25.1 / 34.1 -> 22.1 / 24.3 / 33.0).  At most 256 blocks of 128 x 64 partial sums: 8 MiB.
  if (tiles_t <= 128) {
    int s = (int)std::min<int64_t>(256 / tiles_t, room);
    const int most = (int)std::min<int64_t>(s, K / 1024);
    while (s > 1 && (K % (s * 128) != 0 || K / s < 1024)) --s;
    // no even split near the one wanted (K = 128 x a prime): slices of whole stages, the last shorter
    // (us, K = 9344 = 73 x 128: 33 x 250 28.3 -> 10.5, 80 x 768 28.5 -> 11.2)
    if (most >= 2 && s * 4 < most * 3 && cut_slices(p, M, N, K, most)) return p;
    if (s >= 2) {
      p.splits = s;
      p.k_len = K / s;
      p.ws_bytes = (int64_t)s * M * N * 4;
      p.tall = true;
      return p;
    }
  }
  // shorter reductions: 128 x 128 tiles, slices of at least 512
  const int64_t tiles = (int64_t)div_up(M, TileMid::BM) * div_up(N, TileMid::BN);
  if (tiles > 128) return p;
  // one block per compute unit; 512 and 1024 blocks measured slower
  int s = (int)std::min<int64_t>(256 / tiles, room);
  while (s > 1 && (K % (s * 128) != 0 || K / s < 512)) --s;
  // Slices of 512 are mostly prologue and partial-sum traffic (as many bytes as the weights at
  // 128 rows): from K = 4096 on, half as many slices of 1024 are faster while 64 blocks remain
  // (us, M = 65 / 100 / 128: N = 4096, K = 4096 16.4 / 18.8 / 18.1 -> 15.8 / 17.2 / 16.5; N = 2048
  // 13.8 / 15.1 / 14.1 -> 13.2 / 13.5 / 11.8; N = 1024, K = 8192 15.5 / 16.7 / 15.4 -> 14.2 / 14.6 /
  // 13.1; N = 1000, K = 4096, where 32 blocks would remain, 12.7 -> 14.1; K = 2048 no difference)
  if (K >= 4096 && K / s <= 512 && s >= 4 && s % 2 == 0 && tiles * (s / 2) >= 64) s /= 2;
  if (s < 2) return p;
  p.splits = s;
  p.k_len = K / s;
  p.ws_bytes = (int64_t)s * M * N * 4;
  return p;
}

template <class AccT, class Epi>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const AccT* __restrict__ ws, int S, int M,
                                                            int N, Epi epi) {
  const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
  if (n >= N) return;
  AccT sum = ws[(int64_t)m * N + n];
  for (int s = 1; s < S; ++s) sum += ws[((int64_t)s * M + m) * N + n];
  epi.store(m, n, sum, epi.row(m), epi.col(n, 0, N));
}

// c = sum over K slices (int32, exact), see above.  The caller has checked the operands.
inline int launch_split_k_i32(const SplitPlan& p, const GemmArgs& g0, void* workspace, int32_t* c, int64_t ldc,
                              hipStream_t st) {
  GemmArgs g = g0;
  g.K = (int)p.k_len;
  g.num_experts = p.splits;
  g.rows_per_group = g0.M;
  g.M = p.splits * g0.M;
  g.lda_e = p.k_len;
  g.ldb_e = p.k_len;
  g.k_total = g0.K;
  g.grid_m = p.splits * div_up(g0.M, p.rs ? 256 : p.small ? TileSmallK::BM : TileMid::BM);
  if (p.small && p.cut) launch_tile<TileSmallK, MMA_I8, true, true>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
  else if (p.small) launch_tile<TileSmallK, MMA_I8, true>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
  else if (p.rs) launch_rs<MMA_I8, true, 128>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
  else if (p.cut) launch_tile<TileTallK, MMA_I8, true, true>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
  else if (p.tall) launch_tile<TileTallK, MMA_I8, true>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
  else launch_tile<TileMid, MMA_I8, true>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
  dim3 grid(div_up(g0.N, 256), (unsigned)g0.M), block(256);
  EpiStoreI32 epi{c, ldc};
  hipLaunchKernelGGL((splitk_reduce_kernel<int, EpiStoreI32>), grid, block, 0, st, (const int*)workspace,
                     p.splits, g0.M, g0.N, epi);
  return fmsmo_check_launch();
}

// y = epilogue( sum over K slices ), see above.  The caller has checked the operands.
template <int OP, bool REF, class AccT>
int launch_split_k(const SplitPlan& p, const GemmArgs& g0, void* workspace, const float* a_scale,
                   int a_stride, const float* w_scale, int w_stride, const void* bias,
                   int bias_dtype, void* y, int y_dtype, int64_t ldy, hipStream_t st, int muladd = 0) {
  GemmArgs g = g0;
  g.K = (int)p.k_len;
  g.num_experts = p.splits;
  g.rows_per_group = g0.M;
  g.M = p.splits * g0.M;
  g.lda_e = p.k_len;
  g.ldb_e = p.k_len;
  g.k_total = g0.K;
  g.grid_m = p.splits * div_up(g0.M, p.rs ? 256 : p.small ? TileSmallK::BM : TileMid::BM);
  if constexpr (OP == MMA_FP8_F16) {  // K % 64 != 0: such plans are cut ones
    launch_tile<TileTallK, OP, true, true>(g, EpiStoreF32{(float*)workspace, g0.N}, st);
  } else if (p.small && p.cut) {
    if constexpr (OP == MMA_I8) launch_tile<TileSmallK, OP, true, true>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
    else launch_tile<TileSmallK, OP, true, true>(g, EpiStoreF32{(float*)workspace, g0.N}, st);
  } else if (p.small) {
    if constexpr (OP == MMA_I8) launch_tile<TileSmallK, OP, true>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
    else launch_tile<TileSmallK, OP, true>(g, EpiStoreF32{(float*)workspace, g0.N}, st);
  } else if (p.rs) {
    if constexpr (OP == MMA_I8) launch_rs<OP, true, 128>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
    else launch_rs<OP, true, 128>(g, EpiStoreF32{(float*)workspace, g0.N}, st);
  } else if (p.cut) {
    if constexpr (OP == MMA_I8) launch_tile<TileTallK, OP, true, true>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
    else launch_tile<TileTallK, OP, true, true>(g, EpiStoreF32{(float*)workspace, g0.N}, st);
  } else if (p.tall) {
    if constexpr (OP == MMA_I8) launch_tile<TileTallK, OP, true>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
    else launch_tile<TileTallK, OP, true>(g, EpiStoreF32{(float*)workspace, g0.N}, st);
  } else if constexpr (OP == MMA_I8) launch_tile<TileMid, OP, true>(g, EpiStoreI32{(int32_t*)workspace, g0.N}, st);
  else launch_tile<TileMid, OP, true>(g, EpiStoreF32{(float*)workspace, g0.N}, st);
  if (!bias) bias_dtype = FMSMO_F32;
  dim3 grid(div_up(g0.N, 256), (unsigned)g0.M), block(256);
#define GO(OUT, BIAS)                                                                         \
  {                                                                                           \
    EpiDequant<OUT, BIAS, REF, AccT, OP == MMA_I8 || OUT == FMSMO_F32> epi{y, ldy, a_scale, w_scale, bias, a_stride, w_stride, muladd}; \
    hipLaunchKernelGGL((splitk_reduce_kernel<AccT, decltype(epi)>), grid, block, 0, st,       \
                       (const AccT*)workspace, p.splits, g0.M, g0.N, epi);                    \
  }
#define GO_BIAS(OUT)                            \
  switch (bias_dtype) {                         \
    case FMSMO_F16: GO(OUT, FMSMO_F16) break;   \
    case FMSMO_BF16: GO(OUT, FMSMO_BF16) break; \
    default: GO(OUT, FMSMO_F32) break;          \
  }
  switch (y_dtype) {
    case FMSMO_F16: GO_BIAS(FMSMO_F16) break;
    case FMSMO_BF16: GO_BIAS(FMSMO_BF16) break;
    case FMSMO_F32: GO_BIAS(FMSMO_F32) break;
    default: return FMSMO_ERR_UNSUPPORTED;
  }
#undef GO
#undef GO_BIAS
  return fmsmo_check_launch();
}

}  // namespace

// ------------------------------------------------------------------------------ batched matmul
namespace {

// Batches are the "groups" of the grouped kernels with a uniform row count: the rows of A (and of
// y) of all batches are stacked, B advances by stride_b per batch, the bias by N.
template <int OP, class AccT>
int launch_bmm(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t stride_b,
               const float* a_scale, const float* b_scale, const float* bias, void* y, int y_dtype,
               int64_t ldy, int64_t batch, int64_t M, int64_t N, int64_t K, hipStream_t st, float sc = 1.0f,
               const int32_t* sums = nullptr, int parts = 0, int zero = 0) {
  int rc = check_gemm(a, lda, b, ldb, y, ldy, batch * M, N, K);
  if (rc) return rc;
  if (!sums && (!a_scale || !b_scale)) return FMSMO_ERR_NULL;
  if (batch <= 0 || M <= 0 || stride_b < N * ldb) return FMSMO_ERR_SHAPE;
  if (batch * stride_b >= (1ll << 40) || batch >= (1 << 20)) return FMSMO_ERR_UNSUPPORTED;
  if (K % 64 || stride_b % 16) return FMSMO_ERR_ALIGN;
  if (y_dtype < 0 || y_dtype > 2) return FMSMO_ERR_UNSUPPORTED;
  GemmArgs g{};
  g.a = (const uint8_t*)a; g.b = (const uint8_t*)b; g.lda = lda; g.ldb = ldb;
  g.M = (int)(batch * M); g.N = (int)N; g.K = (int)K;
  g.num_experts = (int)batch; g.ldb_e = stride_b; g.rows_per_group = (int)M;
  g.lda_e = M * lda;
  // small per-batch outputs (attention heads: N or M of 128) take the 128x128 tile
  const bool mid = N <= 128 || M <= 128;
  // probabilities x values: many rows, one head dimension of columns, a long reduction whose
  // A operand is read exactly once -- 256 x 128 tiles of the register-staged pipeline (whole
  // 128-byte lines of P), every block starting its reduction at a different slab: with all blocks
  // sweeping K in step, rows a power of two apart ask for the same memory channels at the same
  // time (4096 x 128 x 4096 per head, 32 heads: 0.144 ms in step, 0.118 ms staggered).  Operands
  // that several tiles share (the large GEMMs) want the opposite: their tiles meet in L2 because
  // they sweep K together (K = 14336: 205 -> 255 us when staggered).
  const bool tall = N > 64 && N <= 128 && M >= 256 && K % 128 == 0 && K >= 512 && use_register_staged(OP);
  g.k_rotate = tall ? 5 : 0;
  // (the kernel for a reduction of 128 has 32-bit output offsets per batch entry)
  const bool k128 = !tall && !mid && K == 128 && use_register_staged(OP) && M * ldy * 4 < (1ll << 31);
  auto run = [&](const auto& epi) {
    if (tall) {
      g.grid_m = (int)batch * div_up(M, 256);
      launch_rs<OP, true, 128>(g, epi, st);
    } else if (mid) {
      g.grid_m = (int)batch * div_up(M, TileMid::BM);
      launch_tile<TileMid, OP, true>(g, epi, st);
    } else {
      g.grid_m = (int)batch * div_up(M, 256);
      if (K % 128 == 0 && use_register_staged(OP)) launch_rs<OP, true>(g, epi, st);
      else launch_tile<TileBig, OP, true>(g, epi, st);
    }
  };
#define GO(OUT)                                                                                          \
  {                                                                                                      \
    const EpiScaleBias<OUT, AccT> sb{y, ldy, a_scale, b_scale, bias, sc, sums, parts, zero, batch * N};  \
    if (k128) {                                                                                          \
      g.grid_m = (int)batch * div_up(M, 256);                                                            \
      launch_k128<OP>(g, (int)batch, (int)M, sb, st);                                                    \
    } else if constexpr (OP == MMA_I8) {                                                                 \
      if (sums && parts > 1) run(sb);                                                                    \
      else if (sums) run(EpiZeroPoint<OUT>{y, ldy, sc, sums, zero});                                     \
      else run(EpiDequant<OUT, FMSMO_F32, false, AccT>{y, ldy, a_scale, b_scale, bias, 0, 0});           \
    } else {                                                                                             \
      run(EpiDequant<OUT, FMSMO_F32, false, AccT>{y, ldy, a_scale, b_scale, bias, 0, 0});                \
    }                                                                                                    \
  }
  switch (y_dtype) {
    case FMSMO_F16: GO(FMSMO_F16) break;
    case FMSMO_BF16: GO(FMSMO_BF16) break;
    default: GO(FMSMO_F32) break;
  }
#undef GO
  return fmsmo_check_launch();
}

}  // namespace
