// Chunked reduced-precision-accumulation matmuls (int8 -> int32 and e4m3/f16/bf16/f32 -> fp32).
//
// D[M,N] = sum over K-chunks of round_trunc( A_chunk . B_chunk^T ) (+ C).  Every chunk is
// multiplied into a FRESH MFMA accumulator (the C operand is the inline constant 0 for the
// first MFMA of the chunk), the chunk result is range-clamped / LSB-rounded on the vector ALU,
// and only then added to the running accumulator -- the same order of operations as the
// reference's Triton kernels, whose BLOCK_SIZE_K equals the chunk size.  A caller who passes a workspace lets
// reductions be cut into slices of whole chunks whose sums are added behind (plan_chunk): the same int32 sums, but
// another grouping of fp32 ones, whose last bits then depend on the tile a row falls into.
//
// Two kernels.  Operands within 2^31 bytes each: the pipelined tile kernel of chunk_tile.hpp.
// Larger ones: the simple kernel below, which addresses its rows with 64 bits.
//
// Simple kernel tiling: 128x128 block, 4 waves of 64x64 (2x2 MFMA 32x32 blocks each); K advances in 64-byte
// stages through two LDS buffers filled with bounds-checked 16-byte loads (zero fill past M, N
// and K, which is what "the K tail is masked to 0" means).  One MFMA k-step is 32 bytes of K
// for every operand type, so chunk boundaries (multiples of 32 bytes) always fall between
// k-steps.
#include "chunk_tile.hpp"
#include <algorithm>

namespace fmsmo {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

struct ChunkArgs {
  const uint8_t* a;
  const uint8_t* b;
  int64_t lda, ldb;  // bytes
  int M, N, Kb;      // Kb = K in bytes
  int chunk_bytes;
  int trun_bits, max_acc_bits, dl16, tta;
  const void* c_in;
  int64_t ldc;  // row stride of c_in (elements)
};

template <int OP>
struct ChunkMma;
template <>
struct ChunkMma<FMSMO_OP_I8> {
  typedef int Elem;
  typedef v16i Acc;
  __device__ static __forceinline__ Acc mma(const v4i& a, const v4i& b, const Acc& c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
  }
};
template <>
struct ChunkMma<FMSMO_OP_E4M3> {
  typedef float Elem;
  typedef v16f Acc;
  __device__ static __forceinline__ Acc mma(const v4i& a, const v4i& b, const Acc& c) {
    // two K=16 MFMAs on the low / high 8 bytes of the lane's 16-byte operand chunk
    const long a0 = ((long)(unsigned)a[1] << 32) | (unsigned)a[0];
    const long a1 = ((long)(unsigned)a[3] << 32) | (unsigned)a[2];
    const long b0 = ((long)(unsigned)b[1] << 32) | (unsigned)b[0];
    const long b1 = ((long)(unsigned)b[3] << 32) | (unsigned)b[2];
    Acc t = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(a0, b0, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(a1, b1, t, 0, 0, 0);
  }
};
template <>
struct ChunkMma<FMSMO_OP_F16> {
  typedef float Elem;
  typedef v16f Acc;
  __device__ static __forceinline__ Acc mma(const v4i& a, const v4i& b, const Acc& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a),
                                                  __builtin_bit_cast(v8h, b), c, 0, 0, 0);
  }
};
template <>
struct ChunkMma<FMSMO_OP_BF16> {
  typedef float Elem;
  typedef v16f Acc;
  __device__ static __forceinline__ Acc mma(const v4i& a, const v4i& b, const Acc& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a),
                                                   __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  }
};

template <>
struct ChunkMma<FMSMO_OP_F32> {
  typedef float Elem;
  typedef v16f Acc;
  __device__ static __forceinline__ Acc mma(const v4i& a, const v4i& b, const Acc& c) {
    // four K=2 fp32 MFMAs, one per float of the lane's 16-byte operand chunk
    Acc t = c;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      t = __builtin_amdgcn_mfma_f32_32x32x2f32(__int_as_float(a[e]), __int_as_float(b[e]), t, 0, 0, 0);
    return t;
  }
};

template <int OP>
__global__ __launch_bounds__(256) void chunk_matmul_kernel(ChunkArgs g, EpiChunk<typename ChunkMma<OP>::Elem> epi) {
  typedef ChunkMma<OP> MM;
  typedef typename MM::Acc Acc;
  typedef typename MM::Elem Elem;
  constexpr int BM = 128, BN = 128, BK = 64, CPR = 4;
  __shared__ __attribute__((aligned(16))) uint8_t lds[2][(BM + BN) * BK];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;

  // loader: thread -> (row = tid / 4 + 64 j, 16-byte chunk = tid % 4), swizzled position in LDS
  const int lr = tid >> 2, lc = tid & 3;
  auto sw = [](int r) { return ((r >> 1) & 3) ^ ((r >> 3) & 1); };
  v4i stage_reg[4];
  auto gload = [&](int k0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int ra = row0 + lr + 64 * j, rb = col0 + lr + 64 * j;
      const int kb = k0 + lc * 16;
      const bool kin = kb + 16 <= g.Kb;
      stage_reg[j] = (ra < g.M && kin) ? *(const v4i*)(g.a + (int64_t)ra * g.lda + kb) : v4i{0, 0, 0, 0};
      stage_reg[2 + j] = (rb < g.N && kin) ? *(const v4i*)(g.b + (int64_t)rb * g.ldb + kb) : v4i{0, 0, 0, 0};
    }
  };
  auto lstore = [&](int buf) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = lr + 64 * j;
      const int pos = lc ^ sw(r);
      *(v4i*)(&lds[buf][r * BK + pos * 16]) = stage_reg[j];
      *(v4i*)(&lds[buf][BM * BK + r * BK + pos * 16]) = stage_reg[2 + j];
    }
  };

  const int fr = lane & 31, fg = lane >> 5, fsw = sw(fr);

  Acc acc[2][2], tmp[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        tmp[i][j][v] = 0;
        Elem init = 0;
        if (g.c_in) {
          const int m = row0 + wm * 64 + i * 32 + (v >> 2) * 8 + fg * 4 + (v & 3);
          const int n = col0 + wn * 64 + j * 32 + fr;
          if (m < g.M && n < g.N) init = ((const Elem*)g.c_in)[(int64_t)m * g.ldc + n];
        }
        acc[i][j][v] = init;
      }

  const int t = g.dl16 ? 14 : g.trun_bits;
  const unsigned round_bit = t > 0 ? 1u << (t - 1) : 0u;
  const unsigned mask = ~((1u << t) - 1u);
  const int lo = g.max_acc_bits < 32 ? -(1 << (g.max_acc_bits - 1)) : (int)0x80000000;
  const int hi = g.max_acc_bits < 32 ? (1 << (g.max_acc_bits - 1)) - 1 : 0x7fffffff;
  const bool post = g.dl16 || t > 0 || g.max_acc_bits < 32;

  auto finish_chunk = [&]() {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          Elem p = tmp[i][j][v];
          if (post) {
            if constexpr (OP == FMSMO_OP_I8) p = trunc_i32(p, lo, hi, (int)round_bit, t);
            else p = trunc_f32(p, round_bit, mask, g.dl16);
          }
          if (g.tta) {
            if constexpr (OP == FMSMO_OP_I8) acc[i][j][v] = (int)((unsigned)acc[i][j][v] + (unsigned)p);
            else acc[i][j][v] += p;
            tmp[i][j][v] = 0;
          } else {
            acc[i][j][v] = p;   // the running accumulator itself was rounded
            tmp[i][j][v] = p;
          }
        }
  };
  if (!g.tta) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) tmp[i][j] = acc[i][j];
  }

  const int nstage = (g.Kb + BK - 1) / BK;
  gload(0);
  lstore(0);
  __syncthreads();
  int in_chunk = 0;  // bytes of the current chunk already multiplied
  for (int st = 0; st < nstage; ++st) {
    const int cur = st & 1;
    if (st + 1 < nstage) gload((st + 1) * BK);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int c = (2 * s + fg) ^ fsw;
      v4i af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) af[i] = *(const v4i*)(&lds[cur][(wm * 64 + i * 32 + fr) * BK + c * 16]);
#pragma unroll
      for (int j = 0; j < 2; ++j) bf[j] = *(const v4i*)(&lds[cur][BM * BK + (wn * 64 + j * 32 + fr) * BK + c * 16]);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) tmp[i][j] = MM::mma(af[i], bf[j], tmp[i][j]);
      in_chunk += 32;
      if (in_chunk == g.chunk_bytes) {
        finish_chunk();
        in_chunk = 0;
      }
    }
    if (st + 1 < nstage) {
      lstore(cur ^ 1);
      __syncthreads();
    }
  }
  if (in_chunk != 0) finish_chunk();  // zero-padded K tail

  // finished half a wave tile (32 rows) at a time in the wave's quarter of the stage buffers
  Elem* const mine = (Elem*)&lds[0][0] + wave * (32 * 64);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) mine[((v >> 2) * 8 + fg * 4 + (v & 3)) * 64 + j * 32 + fr] = acc[i][j][v];
    __syncthreads();
    chunk_finish<64>(epi, mine, 32, row0 + wm * 64 + i * 32, col0 + wn * 64, g.M, g.N, lane);
  }
}

}  // namespace fmsmo

using namespace fmsmo;
int fmsmo_check_launch();

// How the tiles of the pipelined kernel are laid over the 256 compute units: the tiles past the last whole
// round of 256 are cut along K into `slices` pieces of whole chunks, where that is estimated to be faster.
// (us, uncut -> cut as planned here, int8 chunk 64: 16 x 4096 x 14336 70.1 -> 17.2 in 8 slices, 512 rows 73.8 ->
// 49.8 in 2, 1069 rows 126.4 -> 95.1 (32 of 288 tiles in 8), 100 x 700 x 8192 44.2 -> 12.2 in 16, 100 x 1024 x 2048
// 16.5 -> 9.5 in 8; left whole: 300 x 4096 x 4096 26.7 with 96 tiles of 64 stages; fp16 chunk 32 100 x 4096 x 4096
// 75.6 -> 20.4 in 8, 600 rows 77.0 -> 52.3 in 3; e4m3 chunk 64 1024 x 700 x 8192 84.6 -> 28.0 in 5)
struct ChunkPlan {
  int full, slices, slice_len;
  int64_t ws_bytes;
};
static ChunkPlan plan_chunk(int mma, int64_t M, int64_t N, int64_t Kb, int64_t chunk_bytes, bool may_cut, int64_t limit) {
  const int64_t tiles = (int64_t)div_up(M, 128) * div_up(N, 128), rest = tiles % 256;
  ChunkPlan p{(int)tiles, 1, (int)Kb, 0};
  if (!may_cut || rest == 0) return p;
  const int64_t unit = std::max<int64_t>(64, chunk_bytes), units = (Kb + unit - 1) / unit;
  // us: a round of one tile per compute unit takes `stage` per 64 bytes of K; a slice costs its first loads and
  // its accumulators written and read again, the second launch 4
  const double stage = mma == MMA_I8 ? 0.34 : mma == MMA_F32 ? 1.2 : 0.6;
  const double rows = std::min<double>(1.0, (double)M / 128);
  double best = stage * (Kb / 64.0);
  for (int64_t s = 2; s <= std::min<int64_t>(units, 64); ++s) {
    const int64_t len = (units + s - 1) / s;  // in units; the slices that are left
    const int64_t n = (units + len - 1) / len, bytes = rest * n * 65536;
    if (n != s || len * unit < 256) continue;
    if (limit >= 0 && bytes > limit) break;
    const double t = (double)((rest * n + 255) / 256) * (stage * (len * unit / 64.0) + 2.0) + 4.0 + bytes * rows / 2.5e6;
    if (t < best) {
      best = t;
      p = ChunkPlan{(int)(tiles - rest), (int)n, (int)(len * unit), bytes};
    }
  }
  return p;
}

// fp32 accumulators add their chunks one after the other, so a reduction is not to be cut where the caller has not said
// that it may be.  Up to two 64 x 64 tiles per compute unit take those instead: a wave then rounds and adds a quarter
// as many elements per stage (us, 128 x 128 -> 64 x 64, the tiles of 64 in front, chunks one after the other, bits the
// same: fp16 4, 47 x 231 x 6992 94.8 -> 48.6; 94, 107 x 2992 x 3584 55.0 -> 28.1; bf16 333, 151 x 7093 x 5760 71.7 -> 44.8;
// e4m3 414, 1096 x 1439 x 4224 77.4 -> 35.5; fp32 152, 203 x 2372 x 3392 227 -> 74; with the DL16 clamp fp16 490, 632 x 3080
// x 4432 267 -> 104; beyond: fp16 680, 603 x 4326 x 6848 103 -> 107, 837, 561 x 5895 x 5888 82 -> 113; of 105 launches up to
// 490 tiles all faster, 0.43 in the mean).  int32 sums are cut (or take the interleaved schedules of the big tiles).
static bool small_chunk_tiles(int64_t M, int64_t N) {
  return (int64_t)div_up(M, 64) * div_up(N, 64) <= 512;
}

// Pipelined path.  Needs 32-bit row offsets (chunks are whole 32-byte k-steps: a power of two of at
// least 32 bytes).
static bool chunk_tile_ok(const ChunkArgs& c) {
  return c.chunk_bytes % 32 == 0 && (int64_t)c.M * c.lda < (1ll << 31) && (int64_t)c.N * c.ldb < (1ll << 31);
}
template <int MMA, class AccT>
static bool launch_chunk_tile(const ChunkArgs& c, const EpiChunk<AccT>& epi, void* ws, int64_t ws_bytes, hipStream_t st) {
  if (!chunk_tile_ok(c)) return false;
  ChunkTileArgs g{};
  g.a = c.a; g.b = c.b; g.lda = c.lda; g.ldb = c.ldb;
  g.M = c.M; g.N = c.N; g.K = c.Kb;
  const bool fast = c.tta && !c.dl16 && c.max_acc_bits >= 32;
  const ChunkPlan p =
      plan_chunk(MMA, c.M, c.N, c.Kb, c.chunk_bytes, c.tta && !c.c_in && ws, std::max<int64_t>(0, ws_bytes));
  // (a size below zero is no room, not the query's "as much as it takes")
  const int tile = MMA != MMA_I8 && c.tta && p.slices == 1 && small_chunk_tiles(c.M, c.N) ? 64 : 128;
  g.grid_m = div_up(c.M, tile); g.grid_n = div_up(c.N, tile);
  g.chunk_ks = c.chunk_bytes / 32;
  g.t = c.dl16 ? 14 : c.trun_bits;
  g.round_bit = g.t > 0 ? 1u << (g.t - 1) : 0u;
  g.mask = ~((1u << g.t) - 1u);
  g.lo = c.max_acc_bits < 32 ? -(1 << (c.max_acc_bits - 1)) : (int)0x80000000;
  g.hi = c.max_acc_bits < 32 ? (1 << (c.max_acc_bits - 1)) - 1 : 0x7fffffff;
  g.post = c.dl16 || g.t > 0 || c.max_acc_bits < 32;
  g.c_in = c.c_in; g.ldc = c.ldc;
  g.full = tile == 64 ? g.grid_m * g.grid_n : p.full; g.slices = p.slices; g.slice_len = p.slice_len; g.ws = ws;
  const int cut = g.grid_m * g.grid_n - g.full;
  const dim3 grid((unsigned)(g.full + cut * p.slices)), block(256);
  auto go = [&](auto kt_c) {
    constexpr bool KT = decltype(kt_c)::value;
    // the schedules that round one block while the matrix unit multiplies the others: a chunk of one
    // 64-byte stage (every operand type), of several stages or of one 32-byte k-step (int8)
    auto run = [&](auto hook_c, auto sched_c) {
      hipLaunchKernelGGL((chunk_tile_kernel<MMA, decltype(hook_c)::value, decltype(sched_c)::value, KT>), grid, block, 0, st, g, epi);
    };
    typedef std::integral_constant<int, CHUNK_FAST> Fast;
    typedef std::integral_constant<int, 0> S0;
    if constexpr (MMA != MMA_I8)
      if (tile == 64) {
        if (fast) hipLaunchKernelGGL((chunk_tile_kernel<MMA, CHUNK_FAST, 0, KT, 64>), grid, block, 0, st, g, epi);
        else hipLaunchKernelGGL((chunk_tile_kernel<MMA, CHUNK_CLAMP, 0, KT, 64>), grid, block, 0, st, g, epi);
        return;
      }
    if (!c.tta && c.dl16 && MMA != MMA_I8) {
      if constexpr (MMA != MMA_I8) run(std::integral_constant<int, CHUNK_RUNNING_DL16>{}, S0{});
    } else if (!c.tta) run(std::integral_constant<int, CHUNK_RUNNING>{}, S0{});
    else if (!fast) run(std::integral_constant<int, CHUNK_CLAMP>{}, S0{});
    else if (c.chunk_bytes == 64) run(Fast{}, std::integral_constant<int, 1>{});
    else if constexpr (MMA != MMA_I8) run(Fast{}, S0{});
    else if (c.chunk_bytes == 32) run(Fast{}, std::integral_constant<int, 3>{});
    else run(Fast{}, std::integral_constant<int, 2>{});
  };
  if (g.K % 64) go(std::true_type{});
  else go(std::false_type{});
  if (cut > 0)
    hipLaunchKernelGGL((chunk_reduce_kernel<AccT>), dim3((unsigned)cut, 16), block, 0, st, g, epi);
  return true;
}

static int check_chunk(const void* a, int64_t lda, const void* b, int64_t ldb, const void* d,
                       int64_t ldd, int64_t M, int64_t N, int64_t K, int64_t esz, int chunk_size,
                       int min_chunk) {
  if (!a || !b || !d) return FMSMO_ERR_NULL;
  if (M < 0 || N <= 0 || K <= 0 || lda < K || ldb < K || ldd < N) return FMSMO_ERR_SHAPE;
  if (M >= (1 << 30) || N >= (1 << 30) || K * esz >= (1ll << 31)) return FMSMO_ERR_UNSUPPORTED;
  if (chunk_size < min_chunk || (chunk_size & (chunk_size - 1))) return FMSMO_ERR_UNSUPPORTED;
  if ((K * esz) % 16 || (lda * esz) % 16 || (ldb * esz) % 16 || (((uintptr_t)a) & 15) ||
      (((uintptr_t)b) & 15))
    return FMSMO_ERR_ALIGN;
  return FMSMO_OK;
}

static int check_chunk_dq(const float* a_scale, int64_t a_scale_n, const float* w_scale,
                          int64_t w_scale_n, const void* bias, int bias_dtype, int epilogue,
                          int y_dtype, int64_t M, int64_t N) {
  if (!a_scale || !w_scale) return FMSMO_ERR_NULL;
  if ((a_scale_n != 1 && a_scale_n != M) || (w_scale_n != 1 && w_scale_n != N)) return FMSMO_ERR_SHAPE;
  if (y_dtype < 0 || y_dtype > 2 || (bias && (bias_dtype < 0 || bias_dtype > 2))) return FMSMO_ERR_UNSUPPORTED;
  if (epilogue < FMSMO_EPI_REF_F16 || epilogue > FMSMO_EPI_SEQ_OUT) return FMSMO_ERR_UNSUPPORTED;
  return FMSMO_OK;
}

template <class AccT>
static EpiChunk<AccT> epi_raw(void* d, int64_t ldd) {
  EpiChunk<AccT> e{};
  e.y = d; e.ldy = ldd; e.mode = CHUNK_EPI_RAW;
  e.vec4 = ldd % 4 == 0 && ((uintptr_t)d & 15) == 0;
  return e;
}
template <class AccT>
static EpiChunk<AccT> epi_dq(const float* a_scale, int64_t a_scale_n, const float* w_scale, int64_t w_scale_n,
                             const void* bias, int bias_dtype, int epilogue, void* y, int y_dtype, int64_t ldy) {
  return EpiChunk<AccT>{y, ldy, a_scale, w_scale, bias, a_scale_n == 1 ? 0 : 1, w_scale_n == 1 ? 0 : 1, epilogue,
                        y_dtype, bias ? bias_dtype : FMSMO_F32,
                        ldy % 4 == 0 && ((uintptr_t)y & (y_dtype == FMSMO_F32 ? 15 : 7)) == 0};
}

static int run_chunk_i8(const ChunkArgs& g, const EpiChunk<int>& epi, void* ws, int64_t ws_bytes, hipStream_t st) {
  if ((uintptr_t)ws & 15) return FMSMO_ERR_ALIGN;
  if (launch_chunk_tile<MMA_I8>(g, epi, ws, ws_bytes, st)) return fmsmo_check_launch();
  dim3 grid(div_up(g.N, 128), div_up(g.M, 128));
  hipLaunchKernelGGL((chunk_matmul_kernel<FMSMO_OP_I8>), grid, dim3(256), 0, st, g, epi);
  return fmsmo_check_launch();
}

static int run_chunk_fp(int op_dtype, const ChunkArgs& g, const EpiChunk<float>& epi, void* ws, int64_t ws_bytes,
                        hipStream_t st) {
  if ((uintptr_t)ws & 15) return FMSMO_ERR_ALIGN;
  const bool done = op_dtype == FMSMO_OP_E4M3 ? launch_chunk_tile<MMA_FP8_K32>(g, epi, ws, ws_bytes, st)
                    : op_dtype == FMSMO_OP_F16 ? launch_chunk_tile<MMA_F16>(g, epi, ws, ws_bytes, st)
                    : op_dtype == FMSMO_OP_BF16 ? launch_chunk_tile<MMA_BF16>(g, epi, ws, ws_bytes, st)
                                                : launch_chunk_tile<MMA_F32>(g, epi, ws, ws_bytes, st);
  if (done) return fmsmo_check_launch();
  dim3 grid(div_up(g.N, 128), div_up(g.M, 128));
  if (op_dtype == FMSMO_OP_E4M3)
    hipLaunchKernelGGL((chunk_matmul_kernel<FMSMO_OP_E4M3>), grid, dim3(256), 0, st, g, epi);
  else if (op_dtype == FMSMO_OP_F16)
    hipLaunchKernelGGL((chunk_matmul_kernel<FMSMO_OP_F16>), grid, dim3(256), 0, st, g, epi);
  else if (op_dtype == FMSMO_OP_F32)
    hipLaunchKernelGGL((chunk_matmul_kernel<FMSMO_OP_F32>), grid, dim3(256), 0, st, g, epi);
  else
    hipLaunchKernelGGL((chunk_matmul_kernel<FMSMO_OP_BF16>), grid, dim3(256), 0, st, g, epi);
  return fmsmo_check_launch();
}

static ChunkArgs chunk_args_i8(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb, int64_t M,
                               int64_t N, int64_t K, int chunk_size, int chunk_trun_bits,
                               int max_acc_bits, int tta, const void* c_in, int64_t ldc) {
  ChunkArgs g{};
  g.a = (const uint8_t*)a; g.b = (const uint8_t*)b; g.lda = lda; g.ldb = ldb;
  g.M = (int)M; g.N = (int)N; g.Kb = (int)K; g.chunk_bytes = chunk_size;
  g.trun_bits = chunk_trun_bits; g.max_acc_bits = max_acc_bits; g.dl16 = 0;
  g.tta = tta != 0; g.c_in = c_in; g.ldc = ldc;
  return g;
}

// (the mma code of an operand type and its element size, or -1)
static int chunk_mma(int op_dtype, int* esz) {
  *esz = op_dtype == FMSMO_OP_I8 || op_dtype == FMSMO_OP_E4M3 ? 1 : op_dtype == FMSMO_OP_F32 ? 4 : 2;
  switch (op_dtype) {
    case FMSMO_OP_I8: return MMA_I8;
    case FMSMO_OP_E4M3: return MMA_FP8_K32;
    case FMSMO_OP_F16: return MMA_F16;
    case FMSMO_OP_BF16: return MMA_BF16;
    case FMSMO_OP_F32: return MMA_F32;
    default: return -1;
  }
}
extern "C" int64_t fmsmo_matmul_chunk_workspace_bytes(int op_dtype, int64_t M, int64_t N, int64_t K, int chunk_size,
                                                      int truncate_then_accumulate) {
  int esz;
  const int mma = chunk_mma(op_dtype, &esz);
  if (mma < 0 || M <= 0 || N <= 0 || K <= 0 || M >= (1 << 30) || N >= (1 << 30) || K * esz >= (1ll << 31) ||
      chunk_size * esz < 32 || chunk_size > (1 << 28))
    return 0;
  return plan_chunk(mma, M, N, K * esz, (int64_t)chunk_size * esz, truncate_then_accumulate != 0, -1).ws_bytes;
}

extern "C" int fmsmo_matmul_chunk_i8_ws(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                                     const int32_t* c_in, int32_t* d, int64_t ldd, int64_t M,
                                     int64_t N, int64_t K, int chunk_size, int chunk_trun_bits,
                                     int max_acc_bits, int truncate_then_accumulate,
                                     void* workspace, int64_t workspace_bytes, fmsmo_stream_t stream) {
  int rc = check_chunk(a, lda, b, ldb, d, ldd, M, N, K, 1, chunk_size, 32);
  if (rc) return rc;
  if (chunk_trun_bits < 0 || chunk_trun_bits > 31 || max_acc_bits < 2 || max_acc_bits > 32)
    return FMSMO_ERR_UNSUPPORTED;
  if (M == 0) return FMSMO_OK;
  // Nothing to round or clamp: int32 addition wraps and is associative, so the chunked sum is
  // the plain int32 GEMM.
  if (chunk_trun_bits == 0 && max_acc_bits == 32 && !c_in)
    return fmsmo_gemm_i8_i32(a, lda, b, ldb, d, ldd, M, N, K, stream);
  const ChunkArgs g = chunk_args_i8(a, lda, b, ldb, M, N, K, chunk_size, chunk_trun_bits, max_acc_bits,
                                    truncate_then_accumulate, c_in, ldd);
  return run_chunk_i8(g, epi_raw<int>(d, ldd), workspace, workspace_bytes, (hipStream_t)stream);
}
extern "C" int fmsmo_matmul_chunk_i8(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                                     const int32_t* c_in, int32_t* d, int64_t ldd, int64_t M,
                                     int64_t N, int64_t K, int chunk_size, int chunk_trun_bits,
                                     int max_acc_bits, int truncate_then_accumulate, fmsmo_stream_t stream) {
  return fmsmo_matmul_chunk_i8_ws(a, lda, b, ldb, c_in, d, ldd, M, N, K, chunk_size, chunk_trun_bits, max_acc_bits,
                                  truncate_then_accumulate, nullptr, 0, stream);
}

extern "C" int fmsmo_matmul_chunk_i8_dq_ws(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                                        const float* a_scale, int64_t a_scale_n,
                                        const float* w_scale, int64_t w_scale_n, const void* bias,
                                        int bias_dtype, int epilogue, void* y, int y_dtype,
                                        int64_t ldy, int64_t M, int64_t N, int64_t K,
                                        int chunk_size, int chunk_trun_bits, int max_acc_bits,
                                        int truncate_then_accumulate,
                                     void* workspace, int64_t workspace_bytes, fmsmo_stream_t stream) {
  int rc = check_chunk(a, lda, b, ldb, y, ldy, M, N, K, 1, chunk_size, 32);
  if (rc) return rc;
  rc = check_chunk_dq(a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype, epilogue, y_dtype, M, N);
  if (rc) return rc;
  if (chunk_trun_bits < 0 || chunk_trun_bits > 31 || max_acc_bits < 2 || max_acc_bits > 32)
    return FMSMO_ERR_UNSUPPORTED;
  if (M == 0) return FMSMO_OK;
  // nothing to round or clamp: the plain int8 GEMM with the same epilogue, where it has it
  if (chunk_trun_bits == 0 && max_acc_bits == 32 && epilogue != FMSMO_EPI_SEQ_OUT && K % 16 == 0)
    return fmsmo_gemm_i8_dq(a, lda, b, ldb, a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype,
                            epilogue, y, y_dtype, ldy, M, N, K, stream);
  const ChunkArgs g = chunk_args_i8(a, lda, b, ldb, M, N, K, chunk_size, chunk_trun_bits, max_acc_bits,
                                    truncate_then_accumulate, nullptr, 0);
  const EpiChunk<int> epi = epi_dq<int>(a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype, epilogue, y, y_dtype, ldy);
  return run_chunk_i8(g, epi, workspace, workspace_bytes, (hipStream_t)stream);
}
extern "C" int fmsmo_matmul_chunk_i8_dq(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                                        const float* a_scale, int64_t a_scale_n,
                                        const float* w_scale, int64_t w_scale_n, const void* bias,
                                        int bias_dtype, int epilogue, void* y, int y_dtype,
                                        int64_t ldy, int64_t M, int64_t N, int64_t K,
                                        int chunk_size, int chunk_trun_bits, int max_acc_bits,
                                        int truncate_then_accumulate, fmsmo_stream_t stream) {
  return fmsmo_matmul_chunk_i8_dq_ws(a, lda, b, ldb, a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype,
                                     epilogue, y, y_dtype, ldy, M, N, K, chunk_size, chunk_trun_bits, max_acc_bits,
                                     truncate_then_accumulate, nullptr, 0, stream);
}

static int chunk_args_fp(const void* a, int64_t lda, const void* b, int64_t ldb, int op_dtype,
                         const void* d, int64_t ldd, int64_t M, int64_t N, int64_t K, int chunk_size,
                         int chunk_trun_bits, int clamp_dl16, int tta, const void* c_in, int64_t ldc,
                         ChunkArgs* out) {
  if (op_dtype != FMSMO_OP_E4M3 && op_dtype != FMSMO_OP_F16 && op_dtype != FMSMO_OP_BF16 &&
      op_dtype != FMSMO_OP_F32)
    return FMSMO_ERR_UNSUPPORTED;
  const int esz = op_dtype == FMSMO_OP_E4M3 ? 1 : op_dtype == FMSMO_OP_F32 ? 4 : 2;
  int rc = check_chunk(a, lda, b, ldb, d, ldd, M, N, K, esz, chunk_size, esz == 1 ? 32 : 16);
  if (rc) return rc;
  if (chunk_trun_bits < 0 || chunk_trun_bits > 22) return FMSMO_ERR_UNSUPPORTED;
  ChunkArgs g{};
  g.a = (const uint8_t*)a; g.b = (const uint8_t*)b; g.lda = lda * esz; g.ldb = ldb * esz;
  g.M = (int)M; g.N = (int)N; g.Kb = (int)(K * esz); g.chunk_bytes = chunk_size * esz;
  g.trun_bits = chunk_trun_bits; g.max_acc_bits = 32; g.dl16 = clamp_dl16 != 0;
  g.tta = tta != 0; g.c_in = c_in; g.ldc = ldc;
  *out = g;
  return FMSMO_OK;
}

extern "C" int fmsmo_matmul_chunk_fp_ws(const void* a, int64_t lda, const void* b, int64_t ldb,
                                     int op_dtype, const float* c_in, float* d, int64_t ldd,
                                     int64_t M, int64_t N, int64_t K, int chunk_size,
                                     int chunk_trun_bits, int clamp_dl16,
                                     int truncate_then_accumulate,
                                     void* workspace, int64_t workspace_bytes, fmsmo_stream_t stream) {
  ChunkArgs g{};
  int rc = chunk_args_fp(a, lda, b, ldb, op_dtype, d, ldd, M, N, K, chunk_size, chunk_trun_bits,
                         clamp_dl16, truncate_then_accumulate, c_in, ldd, &g);
  if (rc) return rc;
  if (M == 0) return FMSMO_OK;
  return run_chunk_fp(op_dtype, g, epi_raw<float>(d, ldd), workspace, workspace_bytes, (hipStream_t)stream);
}
extern "C" int fmsmo_matmul_chunk_fp(const void* a, int64_t lda, const void* b, int64_t ldb,
                                     int op_dtype, const float* c_in, float* d, int64_t ldd,
                                     int64_t M, int64_t N, int64_t K, int chunk_size,
                                     int chunk_trun_bits, int clamp_dl16,
                                     int truncate_then_accumulate, fmsmo_stream_t stream) {
  return fmsmo_matmul_chunk_fp_ws(a, lda, b, ldb, op_dtype, c_in, d, ldd, M, N, K, chunk_size, chunk_trun_bits,
                                  clamp_dl16, truncate_then_accumulate, nullptr, 0, stream);
}

extern "C" int fmsmo_matmul_chunk_fp_dq_ws(const void* a, int64_t lda, const void* b, int64_t ldb,
                                        int op_dtype, const float* a_scale, int64_t a_scale_n,
                                        const float* w_scale, int64_t w_scale_n, const void* bias,
                                        int bias_dtype, int epilogue, void* y, int y_dtype,
                                        int64_t ldy, int64_t M, int64_t N, int64_t K,
                                        int chunk_size, int chunk_trun_bits, int clamp_dl16,
                                        int truncate_then_accumulate,
                                     void* workspace, int64_t workspace_bytes, fmsmo_stream_t stream) {
  ChunkArgs g{};
  int rc = chunk_args_fp(a, lda, b, ldb, op_dtype, y, ldy, M, N, K, chunk_size, chunk_trun_bits,
                         clamp_dl16, truncate_then_accumulate, nullptr, 0, &g);
  if (rc) return rc;
  rc = check_chunk_dq(a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype, epilogue, y_dtype, M, N);
  if (rc) return rc;
  if (M == 0) return FMSMO_OK;
  const EpiChunk<float> epi = epi_dq<float>(a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype, epilogue, y, y_dtype, ldy);
  return run_chunk_fp(op_dtype, g, epi, workspace, workspace_bytes, (hipStream_t)stream);
}
extern "C" int fmsmo_matmul_chunk_fp_dq(const void* a, int64_t lda, const void* b, int64_t ldb,
                                        int op_dtype, const float* a_scale, int64_t a_scale_n,
                                        const float* w_scale, int64_t w_scale_n, const void* bias,
                                        int bias_dtype, int epilogue, void* y, int y_dtype,
                                        int64_t ldy, int64_t M, int64_t N, int64_t K,
                                        int chunk_size, int chunk_trun_bits, int clamp_dl16,
                                        int truncate_then_accumulate, fmsmo_stream_t stream) {
  return fmsmo_matmul_chunk_fp_dq_ws(a, lda, b, ldb, op_dtype, a_scale, a_scale_n, w_scale, w_scale_n, bias,
                                     bias_dtype, epilogue, y, y_dtype, ldy, M, N, K, chunk_size, chunk_trun_bits,
                                     clamp_dl16, truncate_then_accumulate, nullptr, 0, stream);
}
