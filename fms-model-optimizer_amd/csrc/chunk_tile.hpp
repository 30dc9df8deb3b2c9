// Pipelined kernel of the chunked reduced-precision-accumulation matmuls (see chunk.hip): tiles of 128 x 128 or
// 64 x 64, four waves (of 2 x 2 MFMA blocks of 32 x 32, or of one), K in stages of 64 bytes through a ring
// of four LDS buffers that DMA loads fill three stages ahead, two blocks per compute unit.
//
// Every `chunk_ks` MFMA k-steps (32 bytes of K) the partial product is range-clamped / LSB-rounded on
// the vector ALU and folded into the running accumulator (or the running accumulator itself is rounded
// when tta == 0).  HOOK says how: CHUNK_FAST = the common configuration (truncate-then-accumulate, no integer
// clamp, no DL16 clamp), the others are below.  SCHED (with CHUNK_FAST): the schedules that round one block while the matrix unit multiplies the
// others inside one wave; 1 = a chunk is one stage, 2 = several whole stages (integers), 3 = one k-step
// (integers), 0 = the generic hook.  Each is a kernel of its own (one kernel with all three loops spills).
//
// K only has to be a multiple of 16 bytes: in the last stage lanes whose 16 bytes lie past K fetch the
// row's first bytes of that stage instead and zeros are written over what they brought, which is what
// "the K tail is masked to 0" means (a chunk of zeros rounds to zero).
#pragma once
#include "gemm_tile.hpp"

namespace fmsmo {

// 32-byte k-steps for the chunked-accumulation kernels (chunk boundaries are multiples of 32
// bytes of K for every operand type): two legacy K=16 e4m3 MFMAs, one K=16 f16 / bf16 MFMA, four
// K=2 fp32 MFMAs per 16-byte lane operand.
template <>
struct Mma<MMA_FP8_K32> {
  typedef v4i Frag;
  typedef v16f Acc;
  typedef float Elem;
  static constexpr int KSTEP = 32;
  __device__ static __forceinline__ Acc mma(const Frag& a, const Frag& b, const Acc& c) {
    const long a0 = ((long)(unsigned)a[1] << 32) | (unsigned)a[0];
    const long a1 = ((long)(unsigned)a[3] << 32) | (unsigned)a[2];
    const long b0 = ((long)(unsigned)b[1] << 32) | (unsigned)b[0];
    const long b1 = ((long)(unsigned)b[3] << 32) | (unsigned)b[2];
    Acc t = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(a0, b0, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(a1, b1, t, 0, 0, 0);
  }
};
template <>
struct Mma<MMA_F16> {
  typedef v4i Frag;
  typedef v16f Acc;
  typedef float Elem;
  static constexpr int KSTEP = 32;
  typedef _Float16 v8h __attribute__((ext_vector_type(8)));
  __device__ static __forceinline__ Acc mma(const Frag& a, const Frag& b, const Acc& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a),
                                                  __builtin_bit_cast(v8h, b), c, 0, 0, 0);
  }
};
template <>
struct Mma<MMA_BF16> {
  typedef v4i Frag;
  typedef v16f Acc;
  typedef float Elem;
  static constexpr int KSTEP = 32;
  typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
  __device__ static __forceinline__ Acc mma(const Frag& a, const Frag& b, const Acc& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a),
                                                   __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  }
};
template <>
struct Mma<MMA_F32> {
  typedef v4i Frag;
  typedef v16f Acc;
  typedef float Elem;
  static constexpr int KSTEP = 32;
  __device__ static __forceinline__ Acc mma(const Frag& a, const Frag& b, const Acc& c) {
    Acc t = c;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      t = __builtin_amdgcn_mfma_f32_32x32x2f32(__int_as_float(a[e]), __int_as_float(b[e]), t, 0, 0, 0);
    return t;
  }
};

__device__ __forceinline__ int trunc_i32(int p, int lo, int hi, int round_bit, int t) {
  p = max(min(p, hi), lo);
  // (p + 2^(t-1)) >> t << t with two's-complement wrap on the add, arithmetic right shift
  p = (int)((unsigned)p + (unsigned)round_bit);
  return (int)((unsigned)(p >> t) << t);
}
__device__ __forceinline__ float trunc_f32(float p, unsigned round_bit, unsigned mask, int dl16) {
  float x = __uint_as_float((__float_as_uint(p) + round_bit) & mask);
  if (dl16) {
    x = x >= 8581545984.0f ? __builtin_inff() : x;
    x = x <= -8581545984.0f ? -__builtin_inff() : x;
    x = fabsf(x) < 4.665707820095122e-10f ? 0.0f : x;
  }
  return x;
}

// What happens to a finished accumulator element.  One functor type per accumulator type with the
// mode, the output dtype and the bias dtype as run-time fields (wave-uniform), which keeps the number of
// instantiations of the kernel (operand types x schedules) unchanged.
//   CHUNK_EPI_RAW        d[m,n] = acc                                  (int32 / fp32 out)
//   FMSMO_EPI_REF_F16    f16( f32(acc) * f16(as ws) + b )              (iaddmm_int's plain branch)
//   FMSMO_EPI_F32        fma( f32(acc), as ws, b )
//   FMSMO_EPI_F32_MULADD ( f32(acc) * (as ws) ) + b, every step rounded (iaddmm_int's chunk loop)
//   FMSMO_EPI_SEQ_OUT    T( T( (f32(acc) * as) * ws ) + T(b) ), T = output dtype
//                        (LinearFuncFPxFwdBwd / LinearFuncINT8FwdFP32Bwd: descale, cast, add bias)
enum { CHUNK_EPI_RAW = -1 };
template <class AccT>
struct EpiChunk {
  void* y;
  int64_t ldy;
  const float* a_scale;
  const float* w_scale;
  const void* bias;
  int a_stride, w_stride;
  int mode, out_dt, bias_dt;
  int vec4;  // rows of y start on a multiple of four elements: four neighbours may be stored at once
  struct Col {
    float ws, b;
  };
  __device__ __forceinline__ Col col(int n) const {
    Col c{1.0f, -0.0f};
    if (mode == CHUNK_EPI_RAW) return c;
    c.ws = w_scale[w_stride ? n : 0];
    if (bias) {
      c.b = bias_dt == FMSMO_F16 ? load_as_f32<FMSMO_F16>(bias, n)
            : bias_dt == FMSMO_BF16 ? load_as_f32<FMSMO_BF16>(bias, n) : load_as_f32<FMSMO_F32>(bias, n);
      if (mode == FMSMO_EPI_SEQ_OUT)
        c.b = out_dt == FMSMO_F16 ? round_to<FMSMO_F16>(c.b) : out_dt == FMSMO_BF16 ? round_to<FMSMO_BF16>(c.b) : c.b;
    }
    return c;
  }
  __device__ __forceinline__ float row(int m) const {
    return mode == CHUNK_EPI_RAW ? 1.0f : a_scale[a_stride ? m : 0];
  }
  // the 32 bits of the result (16-bit outputs: in the low half)
  template <int MODE, int OUT>
  __device__ __forceinline__ uint32_t bits(AccT v, float as, Col c) const {
    if constexpr (MODE == CHUNK_EPI_RAW) {
      return __builtin_bit_cast(uint32_t, v);
    } else {
      float t;
      if constexpr (MODE == FMSMO_EPI_REF_F16) {
        const float sc = round_to<FMSMO_F16>(__fmul_rn(as, c.ws));
        t = __fadd_rn(__fmul_rn((float)v, sc), c.b);
        if constexpr (OUT != FMSMO_F32) t = round_to<FMSMO_F16>(t);  // the fp16 accumulator dtype, then the output dtype
      } else if constexpr (MODE == FMSMO_EPI_F32) {
        t = __fmaf_rn((float)v, __fmul_rn(as, c.ws), c.b);
      } else if constexpr (MODE == FMSMO_EPI_F32_MULADD) {
        t = __fadd_rn(__fmul_rn((float)v, __fmul_rn(as, c.ws)), c.b);
      } else {  // (no bias: -0 is added, which changes nothing)
        t = __fadd_rn(round_to<OUT>(__fmul_rn(__fmul_rn((float)v, as), c.ws)), c.b);
      }
      if constexpr (OUT == FMSMO_F16) return f32_to_f16(t);
      else if constexpr (OUT == FMSMO_BF16) return f32_to_bf16(t);
      else return __float_as_uint(t);
    }
  }
  template <int MODE, int OUT>
  __device__ __forceinline__ void put(int64_t idx, uint32_t u) const {
    if constexpr (MODE == CHUNK_EPI_RAW || OUT == FMSMO_F32) ((uint32_t*)y)[idx] = u;
    else ((u16*)y)[idx] = (u16)u;
  }
  // f(mode, output dtype) as constants: one rolled loop per pair, decided once per block (decided per
  // element, 150 branches per four elements, a 128 x 128 tile took 10 us to finish)
  template <class F>
  __device__ __forceinline__ void dispatch(F&& f) const {
    auto with_out = [&](auto mode_c) __attribute__((always_inline)) {
      if (out_dt == FMSMO_F16) f(mode_c, std::integral_constant<int, FMSMO_F16>{});
      else if (out_dt == FMSMO_BF16) f(mode_c, std::integral_constant<int, FMSMO_BF16>{});
      else f(mode_c, std::integral_constant<int, FMSMO_F32>{});
    };
    if (mode == CHUNK_EPI_RAW) f(std::integral_constant<int, CHUNK_EPI_RAW>{}, std::integral_constant<int, FMSMO_F32>{});
    else if (mode == FMSMO_EPI_REF_F16) with_out(std::integral_constant<int, FMSMO_EPI_REF_F16>{});
    else if (mode == FMSMO_EPI_F32) with_out(std::integral_constant<int, FMSMO_EPI_F32>{});
    else if (mode == FMSMO_EPI_F32_MULADD) with_out(std::integral_constant<int, FMSMO_EPI_F32_MULADD>{});
    else with_out(std::integral_constant<int, FMSMO_EPI_SEQ_OUT>{});
  }
};

// What bounds the kernel: MFMAs and roundings of one wave per SIMD while the tiles fill the compute units once
// (0.33 us per 64-byte stage), around them 4 us of first loads and finish.  The finish was 10 us while mode and
// dtypes were tested per element in a fully unrolled epilogue (us, before -> after, chunk 64: 1069 x 4096 x
// 14336 139.6 -> 128.2, 300 x 4096 x 4096 39.3 -> 27.7, 1024 x 12000 x 2048 69.5 -> 46.0).
//
// A wave finishes `height` rows of W accumulators that lie in LDS row by row (rows m0 .., columns n0 ..
// of the result): a rolled loop, four neighbours of a row per lane, whole 128-byte lines of 16-bit results.
template <int W, class AccT>
__device__ __forceinline__ void chunk_finish(const EpiChunk<AccT>& epi, const AccT* acc, int height, int m0, int n0,
                                             int M, int N, int lane) {
  constexpr int LPR = W / 4;  // lanes per row
  const int n = n0 + lane % LPR * 4;
  const int rows = min(height, M - m0);
  if (rows <= 0) return;
  const float as_all = epi.row(min(m0 + lane, M - 1));  // lane r holds the scale of row r
  typename EpiChunk<AccT>::Col cc[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) cc[e] = epi.col(min(n + e, N - 1));
  const bool vec = epi.vec4 && n + 4 <= N;
  epi.dispatch([&](auto mode_c, auto out_c) __attribute__((always_inline)) {
    constexpr int MODE = decltype(mode_c)::value, OUT = decltype(out_c)::value;
#pragma unroll 1
    for (int r0 = 0; r0 < rows; r0 += 64 / LPR) {
      const int r = r0 + lane / LPR;
      const float as = __shfl(as_all, r);
      AccT val[4];
      *(v4i*)val = *(const v4i*)(acc + r * W + lane % LPR * 4);
      uint32_t u[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) u[e] = epi.template bits<MODE, OUT>(val[e], as, cc[e]);
      const int64_t idx = (int64_t)(m0 + r) * epi.ldy + n;
      if (r < rows && vec) {
        if constexpr (MODE == CHUNK_EPI_RAW || OUT == FMSMO_F32)
          *(uint4*)((uint32_t*)epi.y + idx) = uint4{u[0], u[1], u[2], u[3]};
        else
          *(uint2*)((u16*)epi.y + idx) = uint2{u[0] | (u[1] << 16), u[2] | (u[3] << 16)};
      } else if (r < rows) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) epi.template put<MODE, OUT>(idx + e, u[e]);
      }
    }
  });
}

struct ChunkTileArgs {
  const uint8_t* a;
  const uint8_t* b;
  int64_t lda, ldb;    // bytes
  int M, N, K;         // K in bytes, a multiple of 16
  int grid_m, grid_n;  // tiles
  int chunk_ks;        // MFMA k-steps (32 bytes of K) per chunk
  int t, lo, hi;       // LSBs to round away; integer clamp range
  unsigned round_bit, mask;
  int post;            // something to round or clamp
  const void* c_in;    // optional initial accumulator [M, N], same element type as the accumulator
  int64_t ldc;
  // Tiles [0, full) of the tile sequence are whole; of the others every block takes one of `slices` pieces of
  // the reduction of slice_len bytes (whole chunks; the last one shorter) and leaves its accumulators in `ws`
  // for chunk_reduce_kernel.  Rounded chunks are added, so slices of whole chunks give the same int32 sums and fp32
  // ones in another grouping, which is the caller's choice (a workspace or none).  Not with a running accumulator
  // that is itself rounded, nor with c_in.
  int full, slices, slice_len;
  void* ws;
};
constexpr int CHUNK_GROUP_M = 8;  // tile order: column-major in groups of as many tile rows

// What happens at the end of a chunk, beside the common configuration: a clamped chunk is folded (integers: to
// fewer bits, floating point: to DL16), or the running accumulator itself is rounded, in floating point without or
// with the DL16 clamp.  As constants: tested per element, and with the other form's accumulators in registers, these
// kernels needed more than 256 registers, ran one block per compute unit and copied their accumulators between the two
// halves of the register file at every stage (us, before -> after, chunk 64: fp16 running sum 435 x 857 x 1472 51.8 ->
// 16.9, e4m3 333 x 56 x 7296 349 -> 65; chunk 32: int8 clamped to 20 bits 5 x 25 x 6720 277 -> 164, fp16 running sum
// with DL16 33 x 315 x 1568 149 -> 78).  Now 106 ... 178 registers.
enum { CHUNK_FAST, CHUNK_CLAMP, CHUNK_RUNNING, CHUNK_RUNNING_DL16 };
// KT: K is no multiple of a stage.  TILE: rows and columns of a block's tile.
template <int OP, int HOOK, int SCHED, bool KT, int TILE = 128>
__global__ __launch_bounds__(256, 2) void chunk_tile_kernel(ChunkTileArgs g, EpiChunk<typename Mma<OP>::Elem> epi) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stub
  constexpr bool FAST = HOOK == CHUNK_FAST;
  constexpr bool TTA = HOOK <= CHUNK_CLAMP;  // the rounded chunk is added; else the running accumulator is rounded
  static_assert(FAST || SCHED == 0, "the interleaved schedules exist for the fast configuration only");
  typedef Mma<OP> MM;
  typedef typename MM::Frag Frag;
  typedef typename MM::Acc Acc;
  typedef typename MM::Elem Elem;
  static_assert(MM::KSTEP == 32, "a lane's operand of a k-step is one 16-byte chunk");
  static_assert(TILE == 128 || SCHED == 0, "the interleaved schedules take four blocks per wave");
  constexpr int BM = TILE, BN = TILE, BK = 64, NSTAGE = 4;
  constexpr int CPR = BK / 16, RPI = 256 / CPR;  // chunks per tile row, rows per block-wide load
  constexpr int NIA = BM / RPI, NIB = BN / RPI;
  constexpr int TM = BM / 2, TN = BN / 2, FM = TM / 32, FN = TN / 32, NKS = 2;
  constexpr int NMMA = FM * FN, NLD = NIA + NIB;
  constexpr int STAGE_BYTES = (BM + BN) * BK;
  __shared__ __attribute__((aligned(16))) uint8_t lds[NSTAGE * STAGE_BYTES];
  static_assert(NSTAGE * STAGE_BYTES >= BM * BN * 4, "the finished tile passes through the ring's buffers");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  int tile_m, tile_n;
  int k_len = g.K, unit = -1;
  int64_t k_lo = 0;
  if ((int)blockIdx.x < g.full) {
    tile_of_block(blockIdx.x, g.full, g.grid_m, g.grid_n, CHUNK_GROUP_M, tile_m, tile_n);
  } else {
    // slice by slice, and an XCD's blocks are neighbours in that order: they share rows of A and B
    const int cut = g.grid_m * g.grid_n - g.full;
    const int idx = blockIdx.x - g.full, nblk = cut * g.slices, per = nblk >> 3, rem = nblk & 7;
    const int xcd = idx & 7;
    unit = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + (idx >> 3);
    const int slice = unit / cut;
    tile_of_pid(g.full + unit - slice * cut, g.grid_m, g.grid_n, CHUNK_GROUP_M, tile_m, tile_n);
    k_lo = (int64_t)slice * g.slice_len;
    k_len = min(g.slice_len, g.K - (int)k_lo);
  }
  const int row_lo = tile_m * BM, col_lo = tile_n * BN;

  // ---- global -> LDS loader addressing (per thread, constant over the K loop)
  const int ld_row = tid / CPR;
  const int ld_chunk = (tid % CPR) ^ swz<CPR, 1>(ld_row);
  uint32_t a_off[NIA], b_off[NIB];
#pragma unroll
  for (int j = 0; j < NIA; ++j) {
    const int r = min(row_lo + ld_row + j * RPI, g.M - 1);    // clamp: rows past the end re-read
    a_off[j] = (uint32_t)r * (uint32_t)g.lda + ld_chunk * 16;  // the last valid row, never stored
  }
#pragma unroll
  for (int j = 0; j < NIB; ++j) {
    const int r = min(col_lo + ld_row + j * RPI, g.N - 1);
    b_off[j] = (uint32_t)r * (uint32_t)g.ldb + ld_chunk * 16;
  }
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void*)(g.a + k_lo), 0, -1, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)(g.b + k_lo), 0, -1, 0x00020000);
  auto issue_part = [&](int stage, int k0, auto j0_c, auto j1_c) {
    constexpr int J0 = decltype(j0_c)::value, J1 = decltype(j1_c)::value;
    uint8_t* la = lds + stage * STAGE_BYTES + wave * 1024;
#pragma unroll
    for (int j = J0; j < J1; ++j) {
      if (j < NIA)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, FMSMO_LPTR(la + j * 4096), 16, a_off[j], k0, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, FMSMO_LPTR(la + j * 4096), 16, b_off[j - NIA], k0, 0, 0);
    }
  };
  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  typedef std::integral_constant<int, 2> I2;
  typedef std::integral_constant<int, 3> I3;
  typedef std::integral_constant<int, NLD> INLD;

  // ---- LDS -> MFMA operand addressing
  const int fr = lane & 31, fg = lane >> 5;
  const int fsw = swz<CPR, 1>(fr);
  int a_rd[NKS], b_rd[NKS];
#pragma unroll
  for (int s = 0; s < NKS; ++s) {
    const int c = s * 2 + fg;
    a_rd[s] = (wm * TM + fr) * BK + ((c ^ fsw) * 16);
    b_rd[s] = BM * BK + (wn * TN + fr) * BK + ((c ^ fsw) * 16);
  }
  auto read_frags = [&](const uint8_t* ls, int s, Frag* af, Frag* bf) {
#pragma unroll
    for (int i = 0; i < FM; ++i) af[i] = *(const v4i*)(ls + a_rd[s] + i * 32 * BK);
#pragma unroll
    for (int j = 0; j < FN; ++j) bf[j] = *(const v4i*)(ls + b_rd[s] + j * 32 * BK);
  };

  // MFMAs run into `work`, finished chunks are folded into `acc`
  Acc acc[FM][FN], work[FM][FN];
  int ks_cnt = 0;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = work[i][j][v] = 0;
  // element (i, j, v) of the initial accumulator
  auto initial = [&](int i, int j, int v) __attribute__((always_inline)) -> Elem {
    const int m = row_lo + wm * TM + i * 32 + (v >> 2) * 8 + fg * 4 + (v & 3);
    const int n = col_lo + wn * TN + j * 32 + fr;
    return m < g.M && n < g.N ? ((const Elem*)g.c_in)[(int64_t)m * g.ldc + n] : (Elem)0;
  };
  if (g.c_in) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const Elem init = initial(i, j, v);
            (TTA ? acc : work)[i][j][v] = init;
          }
  }

  const int nk = (k_len + BK - 1) / BK;
  // lanes whose chunk of the last stage lies past the end of the reduction
  [[maybe_unused]] const bool past_end = KT && (nk - 1) * BK + ld_chunk * 16 >= k_len;
  // before the DMA of stage st: from the last stage on those lanes fetch chunk 0 (in bounds)
  auto before_issue = [&](int st) __attribute__((always_inline)) {
    if constexpr (KT) {
      if (st == nk - 1 && past_end) {
#pragma unroll
        for (int j = 0; j < NIA; ++j) a_off[j] -= ld_chunk * 16;
#pragma unroll
        for (int j = 0; j < NIB; ++j) b_off[j] -= ld_chunk * 16;
      }
    }
  };
  // until stage st has landed for every wave (at most YOUNGER of this wave's DMA still in flight) and this
  // wave's LDS reads have returned
  auto wait_stage = [&](int st, auto younger_c) __attribute__((always_inline)) {
    constexpr int YOUNGER = decltype(younger_c)::value;
    if constexpr (KT) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");
      if (st == nk - 1 && past_end) {  // zeros over what those lanes fetched
        uint8_t* dst = lds + (st % NSTAGE) * STAGE_BYTES + tid * 16;
#pragma unroll
        for (int j = 0; j < NLD; ++j) *(v4i*)(dst + j * 4096) = v4i{0, 0, 0, 0};
      }
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(YOUNGER) : "memory");
    }
  };

#pragma unroll
  for (int st = 0; st < NSTAGE - 1; ++st) {
    before_issue(st);
    issue_part(st, min(st, nk - 1) * BK, I0{}, INLD{});
  }
  wait_stage(0, std::integral_constant<int, (NSTAGE - 2) * NLD>{});

  if constexpr (SCHED != 0) {
    // The fragments of all k-steps of a stage are register resident (two sets: the stage being
    // multiplied and the one being read), and the rounding of one 32x32 block is issued between the
    // MFMAs of the others, so that one wave keeps both units busy.  With all MFMAs of a chunk issued
    // before any rounding (the generic schedule) the units take turns, and only a second resident wave
    // overlaps them -- which a problem with about one tile per compute unit does not have.
    Frag ca[2][NKS][FM], cb[2][NKS][FN];
    constexpr bool INT = std::is_same<Elem, int>::value;
    static_assert(INT || SCHED == 1, "floating point: a chunk of exactly one stage");
    auto stage_top = [&](int kt, auto par_c) {
      constexpr int PAR = decltype(par_c)::value;
      // stage kt + 1 has landed for every wave; its fragments go to the other register set, and
      // the buffer of stage kt - 1 (last read a stage ago) is refilled with stage kt + 3
      wait_stage(kt + 1, std::integral_constant<int, (NSTAGE - 3) * NLD>{});
      const uint8_t* ls = lds + ((kt + 1) % NSTAGE) * STAGE_BYTES;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) read_frags(ls, ks, ca[PAR ^ 1][ks], cb[PAR ^ 1][ks]);
      before_issue(kt + NSTAGE - 1);
      issue_part((kt + NSTAGE - 1) % NSTAGE, min(kt + NSTAGE - 1, nk - 1) * BK, I0{}, INLD{});
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) read_frags(lds, ks, ca[0][ks], cb[0][ks]);
    if constexpr (INT) {
      // Integers: with R the running sum (a multiple of 2^t) and r the rounding bit, a chunk's
      // MFMAs started from C = R + r leave W = R + p + r, and (W & mask) = R + ((p + r) & mask) is
      // the new running sum: ONE operation per element and chunk, W <- (W & mask) | r, turns the
      // accumulator into the next chunk's C operand (low bits are zero, so OR adds r), and the
      // matrix unit does the accumulation.  8 such operations take as long as one MFMA, and a
      // chunk has 8 MFMAs and 64 elements per lane: the steady state below issues 8 operations in
      // front of every MFMA.  Block b's k-steps are two MFMA slots apart, its 16 operations follow
      // its second MFMA by a slot or more and are complete before its next first MFMA:
      //   slot       0       1       2       3       4       5       6       7
      //   rounding   b1 hi'  b2 lo'  b2 hi'  b3 lo'  b3 hi'  b0 lo   b0 hi   b1 lo    (' = previous chunk)
      //   MFMA       b0 k0   b1 k0   b0 k1   b1 k1   b2 k0   b3 k0   b2 k1   b3 k1
      // (a chunk of several stages rounds behind its last stage only; a chunk of one k-step has a
      // table of its own below)
      // Rounding an accumulator that holds C = R + r changes nothing, so the first chunk runs the
      // same code.  An initial accumulator enters as its multiple of 2^t; its low bits are added
      // at the end (adding a multiple of 2^t commutes with clearing the low bits).
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int jj = 0; jj < FN; ++jj)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            work[i][jj][v] = (int)(((unsigned)acc[i][jj][v] & g.mask) | g.round_bit);
      // (one v_and_or_b32: the instruction takes a single scalar operand, so the rounding bit
      // lives in a vector register)
      unsigned rbv = g.round_bit;
      asm volatile("" : "+v"(rbv));
      auto rnd = [&](auto b_c, auto h_c) {
        constexpr int I = decltype(b_c)::value / FN, J = decltype(b_c)::value % FN, H = decltype(h_c)::value;
#pragma unroll
        for (int v = H * 8; v < H * 8 + 8; ++v)
          work[I][J][v] = (int)(((unsigned)work[I][J][v] & g.mask) | rbv);
        __builtin_amdgcn_sched_barrier(0);
      };
      auto mm = [&](auto par_c, auto b_c, auto ks_c) {
        constexpr int PAR = decltype(par_c)::value, KS = decltype(ks_c)::value;
        constexpr int I = decltype(b_c)::value / FN, J = decltype(b_c)::value % FN;
        work[I][J] = MM::mma(ca[PAR][KS][I], cb[PAR][KS][J], work[I][J]);
        __builtin_amdgcn_sched_barrier(0);
      };
      auto run_stages = [&](auto&& chunk_stage) __attribute__((always_inline)) {
        int kt = 0;
        for (; kt + 1 < nk; kt += 2) {
          chunk_stage(kt, I0{});
          chunk_stage(kt + 1, I1{});
        }
        if (kt < nk) chunk_stage(kt, I0{});
      };
      if constexpr (SCHED == 1) {
        // a chunk is one stage: the table as it stands
        run_stages([&](int kt, auto par_c) {
          stage_top(kt, par_c);
          rnd(I1{}, I1{}); mm(par_c, I0{}, I0{});
          rnd(I2{}, I0{}); mm(par_c, I1{}, I0{});
          rnd(I2{}, I1{}); mm(par_c, I0{}, I1{});
          rnd(I3{}, I0{}); mm(par_c, I1{}, I1{});
          rnd(I3{}, I1{}); mm(par_c, I2{}, I0{});
          rnd(I0{}, I0{}); mm(par_c, I3{}, I0{});
          rnd(I0{}, I1{}); mm(par_c, I2{}, I1{});
          rnd(I1{}, I0{}); mm(par_c, I3{}, I1{});
        });
      } else if constexpr (SCHED == 2) {
        // a chunk is several whole stages: the roundings run only behind a chunk's last stage
        // (slots 5 - 7 of that stage, slots 0 - 4 of the following one)
        const int spc = g.chunk_ks / NKS;
        int phase = 0;  // stage index inside the chunk
        run_stages([&](int kt, auto par_c) {
          stage_top(kt, par_c);
          const bool prev_end = phase == 0, this_end = phase + 1 == spc;
          phase = this_end ? 0 : phase + 1;
          if (prev_end) rnd(I1{}, I1{});
          mm(par_c, I0{}, I0{});
          if (prev_end) rnd(I2{}, I0{});
          mm(par_c, I1{}, I0{});
          if (prev_end) rnd(I2{}, I1{});
          mm(par_c, I0{}, I1{});
          if (prev_end) rnd(I3{}, I0{});
          mm(par_c, I1{}, I1{});
          if (prev_end) rnd(I3{}, I1{});
          mm(par_c, I2{}, I0{});
          if (this_end) rnd(I0{}, I0{});
          mm(par_c, I3{}, I0{});
          if (this_end) rnd(I0{}, I1{});
          mm(par_c, I2{}, I1{});
          if (this_end) rnd(I1{}, I0{});
          mm(par_c, I3{}, I1{});
        });
      } else {
        // a chunk is one k-step (32 bytes of K): 16 roundings per MFMA, the vector ALU is the
        // bound (half the MFMA rate at best).  Per k-step: MFMA b0, round b2', MFMA b1, round b3',
        // MFMA b2, round b0, MFMA b3, round b1 (' = of the previous k-step).
        run_stages([&](int kt, auto par_c) {
          stage_top(kt, par_c);
          [&]<int... KS>(std::integer_sequence<int, KS...>) {
            (
                [&] {
                  typedef std::integral_constant<int, KS> CK;
                  mm(par_c, I0{}, CK{}); rnd(I2{}, I0{}); rnd(I2{}, I1{});
                  mm(par_c, I1{}, CK{}); rnd(I3{}, I0{}); rnd(I3{}, I1{});
                  mm(par_c, I2{}, CK{}); rnd(I0{}, I0{}); rnd(I0{}, I1{});
                  mm(par_c, I3{}, CK{}); rnd(I1{}, I0{}); rnd(I1{}, I1{});
                }(),
                ...);
          }(std::make_integer_sequence<int, NKS>{});
        });
      }
      // the sum of the rounded chunks, plus the low bits of the initial accumulator (read again
      // here: holding it in registers through the loop would cost 64 of them)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] = (int)((unsigned)work[i][j][v] & g.mask);
      if (g.c_in) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v)
              acc[i][j][v] = (int)((unsigned)acc[i][j][v] + ((unsigned)initial(i, j, v) & ~g.mask));
      }
    } else {
      // Floating point: the rounding works on the bits of the chunk's own sum, which is then added
      // in fp32 -- three operations per element (integer add, and, float add).  Block b's MFMAs
      // start from C = 0; block b - 1 is folded into `acc` while they run.
      Acc zero;
#pragma unroll
      for (int v = 0; v < 16; ++v) zero[v] = 0;
      auto fold = [&](auto b_c) {
        constexpr int I = decltype(b_c)::value / FN, J = decltype(b_c)::value % FN;
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[I][J][v] += __uint_as_float((__float_as_uint(work[I][J][v]) + g.round_bit) & g.mask);
      };
      auto chunk_stage = [&](int kt, auto par_c) {
        constexpr int PAR = decltype(par_c)::value;
        stage_top(kt, par_c);
        [&]<int... B>(std::integer_sequence<int, B...>) {
          (
              [&] {
                constexpr int I = B / FN, J = B % FN;
                work[I][J] = MM::mma(ca[PAR][0][I], cb[PAR][0][J], zero);
#pragma unroll
                for (int ks = 1; ks < NKS; ++ks)
                  work[I][J] = MM::mma(ca[PAR][ks][I], cb[PAR][ks][J], work[I][J]);
                __builtin_amdgcn_sched_barrier(0);
                // block B - 1 of this chunk, or the last block of the previous one (zeros before
                // the first chunk: a zero block folds to zero)
                fold(std::integral_constant<int, (B + NMMA - 1) % NMMA>{});
                __builtin_amdgcn_sched_barrier(0);
              }(),
              ...);
        }(std::make_integer_sequence<int, NMMA>{});
      };
      int kt = 0;
      for (; kt + 1 < nk; kt += 2) {
        chunk_stage(kt, I0{});
        chunk_stage(kt + 1, I1{});
      }
      if (kt < nk) chunk_stage(kt, I0{});
      fold(std::integral_constant<int, NMMA - 1>{});
    }
  } else {
    auto finish_chunk = [&]() __attribute__((always_inline)) {
      if (!TTA && !g.post) return;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            if constexpr (FAST) {
              // (p + 2^(t-1)) with the low t bits cleared: same bits for two's-complement integers
              // ((p + r) >> t << t) and for fp32 patterns; work is overwritten by the next chunk
              if constexpr (std::is_same<Elem, int>::value)
                acc[i][j][v] = (int)((unsigned)acc[i][j][v] + (((unsigned)work[i][j][v] + g.round_bit) & g.mask));
              else
                acc[i][j][v] += __uint_as_float((__float_as_uint(work[i][j][v]) + g.round_bit) & g.mask);
            } else {
              Elem p = work[i][j][v];
              if constexpr (std::is_same<Elem, int>::value) p = trunc_i32(p, g.lo, g.hi, (int)g.round_bit, g.t);
              else p = trunc_f32(p, g.round_bit, g.mask, HOOK != CHUNK_RUNNING);
              if constexpr (!TTA) work[i][j][v] = p;
              else if constexpr (std::is_same<Elem, int>::value) acc[i][j][v] = (int)((unsigned)acc[i][j][v] + (unsigned)p);
              else acc[i][j][v] += p;
              if constexpr (TTA) work[i][j][v] = 0;
            }
          }
    };
    auto chunk_tick = [&]() __attribute__((always_inline)) {
      if (++ks_cnt == g.chunk_ks) {
        finish_chunk();
        ks_cnt = 0;
      }
    };
    auto mma_any = [&](const Frag* af, const Frag* bf) __attribute__((always_inline)) {
      // first k-step of a chunk in FAST mode: the MFMA's C operand is the constant 0, so `work` needs
      // no clearing between chunks
      if (FAST && ks_cnt == 0) {
        Acc zero;
#pragma unroll
        for (int v = 0; v < 16; ++v) zero[v] = 0;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) work[i][j] = MM::mma(af[i], bf[j], zero);
      } else {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) work[i][j] = MM::mma(af[i], bf[j], work[i][j]);
      }
    };
    // One K-stage: while stage kt is multiplied, the DMA of stage kt + 3 refills the buffer that
    // stage kt - 1 occupied (free since the barrier at the end of stage kt - 1).  Stages past the end
    // of K re-read the last one into a buffer nobody consumes, which keeps the vmcnt bookkeeping uniform.
    Frag fa[2][FM], fb[2][FN];
    read_frags(lds, 0, fa[0], fb[0]);
    for (int kt = 0; kt < nk; ++kt) {
      const int fill = (kt + NSTAGE - 1) % NSTAGE;
      const int fill_k0 = min(kt + NSTAGE - 1, nk - 1) * BK;
      before_issue(kt + NSTAGE - 1);
      read_frags(lds + (kt % NSTAGE) * STAGE_BYTES, 1, fa[1], fb[1]);
      issue_part(fill, fill_k0, I0{}, std::integral_constant<int, NLD / 2>{});
      mma_any(fa[0], fb[0]);
      chunk_tick();
      // Last k-step: its operands are already in registers.  Wait until this wave's share of stage
      // kt + 1 has landed (younger DMA may stay in flight) and until its own LDS reads of stage kt
      // have returned, then barrier.
      wait_stage(kt + 1, std::integral_constant<int, (NSTAGE - 3) * NLD + NLD / 2>{});
      read_frags(lds + ((kt + 1) % NSTAGE) * STAGE_BYTES, 0, fa[0], fb[0]);
      issue_part(fill, fill_k0, std::integral_constant<int, NLD / 2>{}, INLD{});
      mma_any(fa[1], fb[1]);
      chunk_tick();
    }
    if (ks_cnt != 0) finish_chunk();  // K ended inside a chunk
    if constexpr (!TTA) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = work[i][j];
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no DMA may land in LDS any more

  // ---- epilogue: acc[i][j][v] is C(row, col) with
  //      row = 32 i + 8 (v / 4) + 4 (lane / 32) + v % 4,   col = 32 j + lane % 32
  if (unit >= 0) {
    // a slice: the accumulators as the lanes hold them, 16 bytes each, rows past the end left out
    int* dst = (int*)g.ws + (int64_t)unit * (BM * BN) + tid * 4;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (row_lo + wm * TM + i * 32 + q * 8 < g.M) {
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            Elem e[4] = {acc[i][j][q * 4], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3]};
            *(v4i*)(dst + ((i * FN + j) * 4 + q) * 1024) = *(const v4i*)e;
          }
        }
    return;
  }
  // The wave's 64 x 64 results pass through its quarter of the LDS ring and are finished in a rolled
  // loop, four neighbours of a row per lane.
  __syncthreads();
  Elem* const mine = (Elem*)lds + wave * (TM * TN);
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) mine[(i * 32 + (v >> 2) * 8 + fg * 4 + (v & 3)) * TN + j * 32 + fr] = acc[i][j][v];
  __syncthreads();
  chunk_finish<TN>(epi, mine, TM, row_lo + wm * TM, col_lo + wn * TN, g.M, g.N, lane);
#endif  // __HIP_DEVICE_COMPILE__
}

// Adds the slices' accumulators up, slice by slice, and finishes them: block (tile, piece) takes four rows per
// half wave of one 32-column block (the layout of the accumulators).
template <class AccT>
__global__ __launch_bounds__(256) void chunk_reduce_kernel(ChunkTileArgs g, EpiChunk<AccT> epi) {
  const int cut = gridDim.x, piece = blockIdx.y;
  const int i = piece >> 3, j = (piece >> 2) & 1, q = piece & 3;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int tile_m, tile_n;
  tile_of_pid(g.full + blockIdx.x, g.grid_m, g.grid_n, CHUNK_GROUP_M, tile_m, tile_n);
  const int m = tile_m * 128 + (wave >> 1) * 64 + i * 32 + q * 8 + (lane >> 5) * 4;
  const int n = tile_n * 128 + (wave & 1) * 64 + j * 32 + (lane & 31);
  if (m >= g.M || n >= g.N) return;
  const AccT* p = (const AccT*)g.ws + ((int64_t)blockIdx.x * 16 + piece) * 1024 + threadIdx.x * 4;
  const int64_t step = (int64_t)cut * 16384;
  AccT sum[4];
  *(v4i*)sum = *(const v4i*)p;
  for (int s = 1; s < g.slices; s += 4) {
    AccT v[4][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) *(v4i*)v[u] = *(const v4i*)(p + min(s + u, g.slices - 1) * step);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (s + u < g.slices) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (std::is_same<AccT, int>::value) sum[e] = (int)((unsigned)sum[e] + (unsigned)v[u][e]);
          else sum[e] += v[u][e];
        }
      }
  }
  const typename EpiChunk<AccT>::Col c = epi.col(n);
  epi.dispatch([&](auto mode_c, auto out_c) __attribute__((always_inline)) {
    constexpr int MODE = decltype(mode_c)::value, OUT = decltype(out_c)::value;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (m + e < g.M)
        epi.template put<MODE, OUT>((int64_t)(m + e) * epi.ldy + n, epi.template bits<MODE, OUT>(sum[e], epi.row(m + e), c));
  });
}

}  // namespace fmsmo
