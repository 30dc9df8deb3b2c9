// LDS-tiled MFMA GEMM core for gfx950:  C[M,N] = A[M,K] . B[N,K]^T with 1-byte operands.
//
// Data movement: both operands are K-contiguous, so a tile is a set of rows of BK bytes.  Tiles
// go HBM/L2 -> LDS with global_load_lds_dwordx4 (no VGPR staging); each wave instruction moves
// 64 x 16 B = 1 KiB that lands contiguously in LDS, i.e. 1024/BK whole rows, so every row is
// fetched as one BK-byte run (full 128-byte lines for BK = 128).  The 16-byte chunks of a row
// are XOR-permuted on the way in (the lane picks which global chunk it fetches) so that the
// ds_read_b128 operand fetches of the MFMA phase are bank-conflict free.
//
// Math: each wave owns a (BM/WGM) x (BN/WGN) sub-tile built from 32x32 MFMA blocks
// (v_mfma_i32_32x32x32_i8, or v_mfma_f32_32x32x64_f8f6f4 with both operands e4m3).  The MFMA
// sums over k, so any assignment of k-bytes to (lane group, register byte) is valid as long as
// A and B use the same one; the loaders exploit that and never transpose anything.
//
// Pipeline: NSTAGE LDS buffers.  The DMA of stage kt+NSTAGE is issued during the last MFMA k-step
// of stage kt, so every stage has NSTAGE-1 full iterations (> 1 us) to arrive from L2/HBM.
// One barrier per stage; the barrier, the DMA issue and the first operand reads of the next
// stage are hidden under MFMAs whose operands were read earlier (register double buffering).
//
// Reductions that are no multiple of a stage (KT instances; K is a multiple of 16 bytes, i.e. of the
// 16-byte chunks a lane moves): in the last stage the lanes whose chunk lies past K fetch the row's
// first chunk of that stage instead, and every wave overwrites what those lanes brought with zeros in
// LDS before the barrier that publishes the stage.  The rest of the pipeline does not know about it.
// (One thread per output with 4-byte dot products, which served those K before: 3868 x 542 x 688 int8
// 1195 us, now 14; e4m3, see MMA_FP8_F16, 386 x 531 x 11472 2110 -> 19, 57 x 17694 x 1136 1382 -> 13.)
#pragma once
#include "common.hpp"
#include <type_traits>
#include <utility>

namespace fmsmo {

enum { MMA_I8 = 0, MMA_FP8 = 1, MMA_FP8_K32 = 2, MMA_F16 = 3, MMA_BF16 = 4, MMA_F32 = 5, MMA_FP8_F16 = 6 };

struct GemmArgs {
  const uint8_t* a;
  const uint8_t* b;
  int64_t lda, ldb;  // bytes
  int M, N, K;
  int grid_m, grid_n;  // tiles along M and N (grid_m is an upper bound in grouped mode)
  int group_m;         // tile-order grouping along M
  // grouped (mixture-of-experts) mode
  const int32_t* offsets;
  int num_experts;
  int64_t ldb_e;  // bytes between experts in B
  int rows_per_group;  // > 0: every group owns this many rows (batched matmul, split K), offsets unused
  int64_t lda_e;       // uniform groups: bytes between groups in A (rows * lda for stacked batches,
                       // the K slice length when the groups are slices of one reduction)
  int k_total;         // KT instances, > 0: the groups are K slices of a reduction of this many bytes,
                       // the last one may be shorter than K
  int k_rotate;  // register-staged kernel: block b starts its reduction at slab (b * k_rotate) % slabs
  // optional clock probe (register-staged kernel): block 0 stores {core clock counter, 100 MHz
  // wall clock} at its start, after its K loop and after its epilogue; null = off
  unsigned long long* clk;
};

// 16-byte chunk c of row r is stored at chunk position c ^ swz(r).  Depends on r & 15 only.
template <int CPR, int SWZ>
__device__ __forceinline__ int swz(int r) {
  if constexpr (SWZ == 0) return 0;
  if constexpr (CPR == 8) {
    if constexpr (SWZ == 1) return (r & 7) ^ ((r >> 3) & 1);
    if constexpr (SWZ == 2) return (r & 7);
    return (r >> 1) & 7;
  } else {  // CPR == 4
    if constexpr (SWZ == 1) return ((r >> 1) & 3) ^ ((r >> 3) & 1);
    if constexpr (SWZ == 2) return (r >> 1) & 3;
    return (r >> 2) & 3;
  }
}

template <int OP>
struct Mma;
template <>
struct Mma<MMA_I8> {
  typedef v4i Frag;
  typedef v16i Acc;
  typedef int Elem;
  static constexpr int KSTEP = 32;  // bytes of K per MFMA
  __device__ static __forceinline__ Acc mma(const Frag& a, const Frag& b, const Acc& c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mma<MMA_FP8> {
  typedef v8i Frag;
  typedef v16f Acc;
  typedef float Elem;
  static constexpr int KSTEP = 64;
  __device__ static __forceinline__ Acc mma(const Frag& a, const Frag& b, const Acc& c) {
    // cbsz = blgp = 0: both operands OCP e4m3; zero scale operands select the unscaled form.
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
  }
};

// e4m3 operands widened to fp16 (exact) on their way from LDS into the fp16 matrix instruction, which adds
// their products as accurately as fp32 additions one after the other do (2-norm error of the sum against
// 64 bits at K = 544 / 1136 / 11472: 4.5e-9 / 1.4e-8 / 5.7e-8, the additions 4.7e-9 / 1.4e-8 / 8.6e-8; the
// e4m3 instruction, which keeps fewer bits while it adds, 1.3e-5).  Half the matrix rate and four
// conversions per instruction; us from a HIP graph, e4m3 instruction / this: 386 x 531 x 11472 15.7 / 18.8,
// 1000 x 4096 x 4016 27.8 / 36.0, 4096 x 4096 x 4016 73.9 / 146.
template <>
struct Mma<MMA_FP8_F16> {
  typedef v4i Frag;
  typedef v16f Acc;
  typedef float Elem;
  static constexpr int KSTEP = 32;
  typedef _Float16 v8h __attribute__((ext_vector_type(8)));
  __device__ static __forceinline__ v8h widen(int lo, int hi) {
    const uint32_t w[4] = {__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, false)),
                           __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, true)),
                           __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, false)),
                           __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, true))};
    return __builtin_bit_cast(v8h, v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]});
  }
  __device__ static __forceinline__ Acc mma(const Frag& a, const Frag& b, const Acc& c) {
    const Acc t = __builtin_amdgcn_mfma_f32_32x32x16_f16(widen(a[0], a[1]), widen(b[0], b[1]), c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(widen(a[2], a[3]), widen(b[2], b[3]), t, 0, 0, 0);
  }
};
// Position `pid` of the tile sequence: column-major inside groups of `group_m` tile rows (the
// second half of tile_of_block below, for blocks that walk the sequence themselves).
__device__ __forceinline__ void tile_of_pid(int pid, int grid_m, int grid_n, int group_m, int& tm, int& tn) {
  const int in_group = group_m * grid_n;
  const int gid = pid / in_group;
  const int first_m = gid * group_m;
  const int gsz = min(grid_m - first_m, group_m);
  const int r = pid - gid * in_group;
  tm = first_m + r % gsz;
  tn = r / gsz;
}

// Map the hardware block id to a tile.  Work-groups are dealt round-robin to the 8 XCDs (each
// with a private L2), so block b runs on XCD b % 8; give every XCD one contiguous span of the
// tile sequence, and order that sequence in column-major groups of `group_m` tile rows so the
// tiles resident on an XCD at the same time share A rows and B rows.
__device__ __forceinline__ void tile_of_block(int bid, int nblk, int grid_m, int grid_n,
                                              int group_m, int& tm, int& tn) {
  const int per = nblk >> 3, rem = nblk & 7;
  const int xcd = bid & 7, idx = bid >> 3;
  const int pid = (xcd < rem ? xcd * (per + 1) : rem * (per + 1) + (xcd - rem) * per) + idx;
  const int in_group = group_m * grid_n;
  const int gid = pid / in_group;
  const int first_m = gid * group_m;
  const int gsz = min(grid_m - first_m, group_m);
  const int r = pid - gid * in_group;
  tm = first_m + r % gsz;
  tn = r / gsz;
}

// Row tiles of `bm` rows over all groups (rows offsets[e] .. offsets[e + 1]), and the group that owns row tile
// `tile`: 64 groups at a time, one per lane (one after the other, each waiting for its offsets, 16 groups took
// 2 us of every block).
__device__ __forceinline__ int wave_scan_add(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(v, o, 64);
    v += lane >= o ? u : 0;
  }
  return v;
}
__device__ __forceinline__ int group_tiles(const int32_t* offsets, int groups, int bm, int lane) {
  int sum = 0;
  for (int e0 = 0; e0 < groups; e0 += 64) {
    const int e = e0 + lane;
    sum += e < groups ? (offsets[e + 1] - offsets[e] + bm - 1) / bm : 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
  return __builtin_amdgcn_readfirstlane(sum);
}
__device__ __forceinline__ void group_of_tile(const int32_t* offsets, int groups, int bm, int lane, int tile,
                                              int& group, int& row_lo, int& row_hi) {
  for (int e0 = 0, before = 0; e0 < groups; e0 += 64) {
    const int e = min(e0 + lane, groups - 1);
    const int lo = offsets[e], hi = offsets[e + 1];
    const int n = e0 + lane < groups ? (hi - lo + bm - 1) / bm : 0;
    const int incl = before + wave_scan_add(n, lane);
    const unsigned long long after = __ballot(incl > tile);  // the first such lane owns it
    if (after) {
      const int l = __builtin_ctzll(after);
      group = e0 + l;
      row_lo = __builtin_amdgcn_readlane(lo, l) + (tile - __builtin_amdgcn_readlane(incl - n, l)) * bm;
      row_hi = __builtin_amdgcn_readlane(hi, l);
      return;
    }
    before = __builtin_amdgcn_readlane(incl, 63);
  }
}

template <int BM, int BN, int BK, int NSTAGE, int WGM, int WGN, int OP, int SWZ, bool GROUPED,
          class Epi, bool KT = false>
__global__ __launch_bounds__(WGM* WGN * 64, 1) void gemm_tile_kernel(GemmArgs g, Epi epi) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stub
  typedef Mma<OP> MM;
  typedef typename MM::Frag Frag;
  typedef typename MM::Acc Acc;
  constexpr int THREADS = WGM * WGN * 64;
  constexpr int CPR = BK / 16;              // 16-byte chunks per tile row
  constexpr int RPI = THREADS / CPR;        // tile rows moved by one block-wide load instruction
  constexpr int NIA = BM / RPI, NIB = BN / RPI;
  constexpr int TM = BM / WGM, TN = BN / WGN;  // wave sub-tile
  constexpr int FM = TM / 32, FN = TN / 32;    // 32x32 MFMA blocks per wave
  constexpr int NKS = BK / MM::KSTEP;          // MFMA k-steps per stage
  constexpr int CL = MM::KSTEP / 32;           // 16-byte chunks per lane per k-step
  static_assert(RPI % 16 == 0 && BM % RPI == 0 && BN % RPI == 0, "loader shape");
  static_assert(TM % 32 == 0 && TN % 32 == 0, "wave tile");

  constexpr int STAGE_BYTES = (BM + BN) * BK;
  __shared__ __attribute__((aligned(16))) uint8_t lds[NSTAGE][STAGE_BYTES];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  int tile_m, tile_n;
  int row_lo = 0, row_hi = g.M, expert = 0;
  int64_t a_adj = 0;
  if constexpr (GROUPED) {
    if (g.rows_per_group > 0) {
      // batched matmul: every group has the same number of rows, the grid is exact
      const int nt = (g.rows_per_group + BM - 1) / BM;
      tile_of_block(blockIdx.x, gridDim.x, g.num_experts * nt, g.grid_n, g.group_m, tile_m, tile_n);
      expert = tile_m / nt;
      row_lo = expert * g.rows_per_group + (tile_m - expert * nt) * BM;
      row_hi = (expert + 1) * g.rows_per_group;
      // rows are numbered as stacked groups (that is how the output is laid out); A may be laid
      // out differently
      a_adj = (int64_t)expert * (g.lda_e - (int64_t)g.rows_per_group * g.lda);
    } else {
      // The launch grid is an upper bound (the host cannot see the expert sizes).  Count the
      // real row tiles and map only the first real_tiles block ids, so that every XCD gets an
      // equal share of real work; the surplus blocks are the last to be dispatched and exit at
      // once.
      const int real_tiles = group_tiles(g.offsets, g.num_experts, BM, lane) * g.grid_n;
      if ((int)blockIdx.x >= real_tiles) return;  // uniform for the whole block
      tile_of_block(blockIdx.x, real_tiles, real_tiles / g.grid_n, g.grid_n, g.group_m, tile_m, tile_n);
      group_of_tile(g.offsets, g.num_experts, BM, lane, tile_m, expert, row_lo, row_hi);
    }
  } else {
    tile_of_block(blockIdx.x, gridDim.x, g.grid_m, g.grid_n, g.group_m, tile_m, tile_n);
    row_lo = tile_m * BM;
  }
  const int col_lo = tile_n * BN;

  const uint8_t* __restrict__ A = g.a + a_adj;
  const uint8_t* __restrict__ B = g.b + (GROUPED ? (int64_t)expert * g.ldb_e : 0);

  // ---- global -> LDS loader addressing (per thread, constant over the K loop)
  const int ld_row = tid / CPR;
  const int ld_pos = tid % CPR;
  const int ld_chunk = ld_pos ^ swz<CPR, SWZ>(ld_row);
  uint32_t a_off[NIA], b_off[NIB];
#pragma unroll
  for (int j = 0; j < NIA; ++j) {
    const int r = min(row_lo + ld_row + j * RPI, row_hi - 1);  // clamp: rows past the end re-read
    a_off[j] = (uint32_t)r * (uint32_t)g.lda + ld_chunk * 16;  // the last valid row, never stored
  }
#pragma unroll
  for (int j = 0; j < NIB; ++j) {
    const int r = min(col_lo + ld_row + j * RPI, g.N - 1);
    b_off[j] = (uint32_t)r * (uint32_t)g.ldb + ld_chunk * 16;
  }

  // DMA instructions j in [j0, j1) of a stage (A rows first, then B rows).  Buffer addressing:
  // per-lane 32-bit row/chunk offset (constant over K) + scalar K offset, so the loop needs no
  // vector address arithmetic.
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc((void*)A, 0, -1, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc((void*)B, 0, -1, 0x00020000);
  auto issue_part = [&](int stage, int k0, auto j0_c, auto j1_c) {
    constexpr int J0 = decltype(j0_c)::value, J1 = decltype(j1_c)::value;
    uint8_t* la = &lds[0][0] + stage * STAGE_BYTES + wave * 1024;
#pragma unroll
    for (int j = J0; j < J1; ++j) {
      if (j < NIA)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, FMSMO_LPTR(la + j * THREADS * 16), 16,
                                                 a_off[j], k0, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_b, FMSMO_LPTR(la + j * THREADS * 16), 16,
                                                 b_off[j - NIA], k0, 0, 0);
    }
  };

  // ---- LDS -> MFMA operand addressing
  const int fr = lane & 31, fg = lane >> 5;
  const int fsw = swz<CPR, SWZ>(fr);
  int a_rd[NKS][CL], b_rd[NKS][CL];
#pragma unroll
  for (int s = 0; s < NKS; ++s)
#pragma unroll
    for (int e = 0; e < CL; ++e) {
      const int c = s * 2 * CL + fg * CL + e;
      a_rd[s][e] = (wm * TM + fr) * BK + ((c ^ fsw) * 16);
      b_rd[s][e] = BM * BK + (wn * TN + fr) * BK + ((c ^ fsw) * 16);
    }

  Acc acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;

  auto read_frags = [&](const uint8_t* ls, int s, Frag* af, Frag* bf) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      if constexpr (CL == 1) {
        af[i] = *(const v4i*)(ls + a_rd[s][0] + i * 32 * BK);
      } else {
        const v4i lo = *(const v4i*)(ls + a_rd[s][0] + i * 32 * BK);
        const v4i hi = *(const v4i*)(ls + a_rd[s][1] + i * 32 * BK);
        af[i] = Frag{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (CL == 1) {
        bf[j] = *(const v4i*)(ls + b_rd[s][0] + j * 32 * BK);
      } else {
        const v4i lo = *(const v4i*)(ls + b_rd[s][0] + j * 32 * BK);
        const v4i hi = *(const v4i*)(ls + b_rd[s][1] + j * 32 * BK);
        bf[j] = Frag{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
  };
  auto mma_step = [&](const Frag* af, const Frag* bf) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = MM::mma(af[i], bf[j], acc[i][j]);
  };
  // Instruction-order hints (DS read = 0x100, MFMA = 0x008, VMEM = 0x020): the operand reads of
  // the next k-step go between the first MFMAs of the current one, so their latency is covered
  // by the remaining MFMAs; the DMA instructions are spread evenly behind them (the texture
  // path takes ~16 cycles per 1 KiB wave instruction and is shared by the whole CU, so bursts
  // of DMA issue would stall the in-order wave and starve the MFMA pipe).
  constexpr int NRD = (FM + FN) * CL, NMMA = FM * FN, NLD = NIA + NIB;
  // DMA instructions [NLD * S / NKS, NLD * (S + 1) / NKS) are issued during k-step S
  static_assert(NSTAGE >= 3, "pipeline needs at least three LDS stages");
  auto interleave = [&](auto ldp_c) {
    constexpr int LDP = decltype(ldp_c)::value;  // DMA instructions issued in this k-step
    constexpr int PER = (NMMA / 2) / NRD > 0 ? (NMMA / 2) / NRD : 1;
#pragma unroll
    for (int r = 0; r < NRD; ++r) {
      __builtin_amdgcn_sched_group_barrier(0x008, PER, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    constexpr int REST = NMMA - PER * NRD > 0 ? NMMA - PER * NRD : 0;
    if constexpr (REST >= LDP && LDP > 0) {
      constexpr int MPL = REST / LDP;  // MFMAs per DMA instruction
#pragma unroll
      for (int r = 0; r < LDP; ++r) {
        __builtin_amdgcn_sched_group_barrier(0x008, MPL, 0);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
      if constexpr (REST - MPL * LDP > 0) __builtin_amdgcn_sched_group_barrier(0x008, REST - MPL * LDP, 0);
    } else if constexpr (REST > 0) {
      __builtin_amdgcn_sched_group_barrier(0x008, REST, 0);
    }
  };

  Frag fa[2][FM], fb[2][FN];
  int k_len = g.K;
  if constexpr (KT && GROUPED) {
    if (g.k_total > 0) k_len = min(k_len, g.k_total - expert * k_len);
  }
  const int nk = KT ? (k_len + BK - 1) / BK : k_len / BK;
  // KT: lanes whose chunk of the last stage lies past the end of the reduction
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
  // stage st has landed for this wave: replace what those lanes fetched by zeros
  auto zero_past_end = [&](int st) __attribute__((always_inline)) {
    if constexpr (KT) {
      if (st == nk - 1 && past_end) {
        uint8_t* dst = &lds[0][0] + (st % NSTAGE) * STAGE_BYTES + tid * 16;
#pragma unroll
        for (int j = 0; j < NIA + NIB; ++j) *(v4i*)(dst + j * THREADS * 16) = v4i{0, 0, 0, 0};
      }
    }
  };

  // One K-stage.  PAR = parity of kt * NKS, so that operand-register buffer indices are static.
  // While stage kt is multiplied, the DMA of stage kt+NSTAGE-1 refills the buffer that stage
  // kt-1 occupied (free since the barrier at the end of stage kt-1).  Stages past the end of K
  // are "phantom": their DMA re-reads the last real stage into a buffer nobody consumes, which
  // keeps the loop body and the vmcnt bookkeeping uniform.
  auto stage = [&](int kt, auto par_c) {
    constexpr int PAR = decltype(par_c)::value;
    const int cur = kt % NSTAGE;
    const int fill = (kt + NSTAGE - 1) % NSTAGE;
    const int fill_k0 = min(kt + NSTAGE - 1, nk - 1) * BK;
    const uint8_t* ls = &lds[0][0] + cur * STAGE_BYTES;
    before_issue(kt + NSTAGE - 1);
    auto dma = [&](auto s_c) {
      constexpr int S = decltype(s_c)::value;
      issue_part(fill, fill_k0, std::integral_constant<int, NLD * S / NKS>{},
                 std::integral_constant<int, NLD * (S + 1) / NKS>{});
    };
    [&]<int... S>(std::integer_sequence<int, S...>) {
      (
          [&] {
            read_frags(ls, S + 1, fa[(PAR + S + 1) & 1], fb[(PAR + S + 1) & 1]);
            dma(std::integral_constant<int, S>{});
            mma_step(fa[(PAR + S) & 1], fb[(PAR + S) & 1]);
            interleave(std::integral_constant<int, NLD * (S + 1) / NKS - NLD * S / NKS>{});
          }(),
          ...);
    }(std::make_integer_sequence<int, NKS - 1>{});
    // Last k-step: its operands are already in registers.  Wait until this wave's share of
    // stage kt+1 has landed (younger DMA may stay in flight) and until its own LDS reads of
    // stage kt have returned, then barrier: stage kt+1 is now complete for all waves and buffer
    // `cur` may be refilled during the next stage.
    if constexpr (KT) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NSTAGE - 3) * NLD + NLD * (NKS - 1) / NKS) : "memory");
      zero_past_end(kt + 1);
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NSTAGE - 3) * NLD + NLD * (NKS - 1) / NKS)
                 : "memory");
    const int nxt = (kt + 1) % NSTAGE;
    read_frags(&lds[0][0] + nxt * STAGE_BYTES, 0, fa[(PAR + NKS) & 1], fb[(PAR + NKS) & 1]);
    dma(std::integral_constant<int, NKS - 1>{});
    mma_step(fa[(PAR + NKS - 1) & 1], fb[(PAR + NKS - 1) & 1]);
    interleave(std::integral_constant<int, NLD - NLD * (NKS - 1) / NKS>{});
  };

#pragma unroll
  for (int st = 0; st < NSTAGE - 1; ++st) {
    before_issue(st);
    issue_part(st, min(st, nk - 1) * BK, std::integral_constant<int, 0>{},
               std::integral_constant<int, NLD>{});
  }
  if constexpr (KT) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NSTAGE - 2) * NLD) : "memory");
    zero_past_end(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NSTAGE - 2) * NLD) : "memory");
  }
  read_frags(&lds[0][0], 0, fa[0], fb[0]);
  {
    int kt = 0;
    if constexpr (NKS % 2 == 0) {
      for (; kt < nk; ++kt) stage(kt, std::integral_constant<int, 0>{});
    } else {
      for (; kt + 1 < nk; kt += 2) {
        stage(kt, std::integral_constant<int, 0>{});
        stage(kt + 1, std::integral_constant<int, 1>{});
      }
      if (kt < nk) stage(kt, std::integral_constant<int, 0>{});
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no DMA may be in flight when LDS is released
  // ---- epilogue: acc[i][j][v] is C(row, col) with
  //      row = 32 i + 8 (v / 4) + 4 (lane / 32) + v % 4,   col = 32 j + lane % 32
  const int m_base = row_lo + wm * TM + fg * 4;
  const int n_base = col_lo + wn * TN + fr;
  typename Epi::Col colctx[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) colctx[j] = epi.col(min(n_base + j * 32, g.N - 1), expert, g.N);
  // Whole tiles take a branch-free path.  The row operands (token scales) of up to two row blocks
  // are requested before the blocks' first store: a load may not be moved across a store through an
  // unrelated pointer, so requested block by block their latency is paid once per block.  Tiles cut
  // by the last row test rows in the groups of 8 that the accumulator layout makes wave-uniform
  // (whole groups store without per-lane tests, groups past the end are skipped by a scalar
  // branch); per-lane tests around every store would put each store into a basic block of its own.
  const bool cols_full = col_lo + BN <= g.N;
  const bool interior = (row_lo + BM <= row_hi) && cols_full;
  const int rows_left = row_hi - row_lo - wm * TM;  // valid rows from this wave's first row on; uniform
  constexpr int RBB = FM % 2 == 0 ? 2 : 1;
#pragma unroll
  for (int i0 = 0; i0 < FM; i0 += RBB) {
    if (rows_left - i0 * 32 <= 0) break;
    typename Epi::Row rowctx[RBB][16];
#pragma unroll
    for (int i = 0; i < RBB; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        rowctx[i][v] = epi.row(min(m_base + (i0 + i) * 32 + (v >> 2) * 8 + (v & 3), row_hi - 1));
    if (interior) {
#pragma unroll
      for (int i = 0; i < RBB; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int m = m_base + (i0 + i) * 32 + (v >> 2) * 8 + (v & 3);
#pragma unroll
          for (int j = 0; j < FN; ++j) epi.store(m, n_base + j * 32, acc[i0 + i][j][v], rowctx[i][v], colctx[j]);
        }
    } else {
#pragma unroll
      for (int i = 0; i < RBB; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int left = rows_left - (i0 + i) * 32 - q * 8;
          if (left >= 8 && cols_full) {
#pragma unroll
            for (int vv = 0; vv < 4; ++vv) {
              const int v = q * 4 + vv, m = m_base + (i0 + i) * 32 + q * 8 + vv;
#pragma unroll
              for (int j = 0; j < FN; ++j) epi.store(m, n_base + j * 32, acc[i0 + i][j][v], rowctx[i][v], colctx[j]);
            }
          } else if (left > 0) {
#pragma unroll
            for (int vv = 0; vv < 4; ++vv) {
              const int v = q * 4 + vv, m = m_base + (i0 + i) * 32 + q * 8 + vv;
              if (m < row_hi) {
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                  const int n = n_base + j * 32;
                  if (n < g.N) epi.store(m, n, acc[i0 + i][j][v], rowctx[i][v], colctx[j]);
                }
              }
            }
          }
        }
    }
  }
#endif  // __HIP_DEVICE_COMPILE__
}

// ------------------------------------------------------------------------------ epilogues
struct EpiStoreI32 {
  int32_t* c;
  int64_t ldc;
  struct Col {};
  struct Row {};
  __device__ __forceinline__ Col col(int, int, int) const { return Col{}; }
  __device__ __forceinline__ Row row(int) const { return Row{}; }
  __device__ __forceinline__ void store(int m, int n, int v, Row, Col) const {
    c[(int64_t)m * ldc + n] = v;
  }
};

struct EpiStoreF32 {
  float* c;
  int64_t ldc;
  struct Col {};
  struct Row {};
  __device__ __forceinline__ Col col(int, int, int) const { return Col{}; }
  __device__ __forceinline__ Row row(int) const { return Row{}; }
  __device__ __forceinline__ void store(int m, int n, float v, Row, Col) const {
    c[(int64_t)m * ldc + n] = v;
  }
};

// y = acc * (a_scale[m] x w_scale[n]) + bias[n], see FMSMO_EPI_* in fmsmo_hip.h.
// MULADD_SWITCH: whether the fp32-scale form looks at `muladd` at all.  The e4m3 GEMMs never ask
// for the separate multiply and add; without the test their 256 stores per lane are one straight
// run (the block-uniform test per element cost them 0.5 ... 1.5 % of the whole launch).  Their
// fp32-output instances keep the switch: without it the register allocation of the 256 x 256
// tile came out four registers short.
template <int OUT, int BIAS, bool REF_F16, class AccT, bool MULADD_SWITCH = true>
struct EpiDequant {
  void* y;
  int64_t ldy;
  const float* a_scale;
  const float* w_scale;
  const void* bias;
  int a_stride, w_stride;  // 0 = one value for all rows / columns, 1 = per row / column
  int muladd = 0;          // fp32-scale form only: separate multiply and add instead of one fma
  struct Col {
    float ws, b;
  };
  struct Row {
    float as;
  };
  __device__ __forceinline__ Col col(int n, int expert, int N) const {
    Col c;
    const int64_t o = (int64_t)expert * N + n;
    c.ws = w_scale[w_stride ? o : 0];
    c.b = bias ? load_as_f32<BIAS>(bias, o) : -0.0f;  // no bias: x + (-0) == x, the sign of a zero product included
    return c;
  }
  __device__ __forceinline__ Row row(int m) const { return Row{a_scale[a_stride ? m : 0]}; }
  __device__ __forceinline__ void store(int m, int n, AccT v, Row r, Col c) const {
    const int64_t idx = (int64_t)m * ldy + n;
    if constexpr (REF_F16) {
      // separate fp32 multiply and add (no fma), scale product rounded to fp16 first; a 16-bit
      // output is the fp16 accumulator dtype of from_fms_mo cast to the output dtype, an fp32
      // output is the fp32 accumulator dtype of from_torch_iW (no fp16 rounding of the result)
      const float sc = round_to<FMSMO_F16>(__fmul_rn(r.as, c.ws));
      const float t = __fadd_rn(__fmul_rn((float)v, sc), c.b);
      if constexpr (OUT == FMSMO_F32) ((float*)y)[idx] = t;
      else if constexpr (OUT == FMSMO_F16) __builtin_nontemporal_store(f32_to_f16(t), &((u16*)y)[idx]);
      else store_from_f32<OUT>(y, idx, f16_to_f32(f32_to_f16(t)));
    } else {
      const float sc = __fmul_rn(r.as, c.ws);
      const float t = (MULADD_SWITCH && muladd) ? __fadd_rn(__fmul_rn((float)v, sc), c.b) : __fmaf_rn((float)v, sc, c.b);
      store_from_f32<OUT>(y, idx, t);
    }
  }
};

// Sum of `parts` partial sums, `stride` apart: eight loads in flight (one after the other, 24 parts took
// 15 us of a product of one query row; so 9).
__device__ __forceinline__ int sum_parts(const int32_t* p, int64_t stride, int parts) {
  int sum = 0;
  for (int i = 0; i < parts; i += 8) {
    int v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[min(i + u, parts - 1) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) sum += i + u < parts ? v[u] : 0;
  }
  return sum;
}

// y = (acc - zero * sum[n]) * scale: the int8 batched matmul whose first operand has a zero point, in
// kernels that keep all their accumulators until the end.  sum: of the second operand's codes over the
// reduction, [batch * N].  One load per column, like EpiDequant: adding up partial sums here (EpiScaleBias
// below) cost the register-staged 256 x 256 tile 17 us of 44 (12 heads of 129 x 129 x 512: 27.5) and
// the 128 x 128 tile 14 of 47 (64 x 64 x 8192), more than the launch that adds them up first.
template <int OUT>
struct EpiZeroPoint {
  void* y;
  int64_t ldy;
  float sc;
  const int32_t* sums;
  int zero;
  struct Col {
    int z;
  };
  struct Row {};
  __device__ __forceinline__ Col col(int n, int expert, int N) const { return Col{zero * sums[(int64_t)expert * N + n]}; }
  __device__ __forceinline__ Row row(int) const { return Row{}; }
  __device__ __forceinline__ void store(int m, int n, int v, Row, Col c) const {
    store_from_f32<OUT>(y, (int64_t)m * ldy + n, __fmul_rn((float)(v - c.z), sc));
  }
};

// y = (acc - zero * sum[n]) * (a_scale * w_scale) + bias[n]: the epilogue of the batched matmul with a
// reduction of 128, one scale for the whole batch (EpiDequant's fp32-scale arithmetic with nothing to
// fetch per row).  sums: `parts` partial sums over the reduction of the second operand's codes,
// [parts][batch * N] (int32 operands only: the zero-point correction of the first one, exact in
// integers), or NULL.  The scale product is that of two device scalars, or `sc` itself where they are NULL.
template <int OUT, class AccT>
struct EpiScaleBias {
  static constexpr int OUT_DT = OUT;
  void* y;
  int64_t ldy;
  const float* a_scale;
  const float* w_scale;
  const float* bias;
  float sc = 1.0f;
  const int32_t* sums = nullptr;
  int parts = 0, zero = 0;
  int64_t part_stride = 0;
  struct Col {
    float b;
    AccT z;
  };
  struct Row {
    float sc;
  };
  __device__ __forceinline__ Col col(int n, int expert, int N) const {
    const int64_t o = (int64_t)expert * N + n;
    Col c{bias ? bias[o] : -0.0f, 0};
    if constexpr (std::is_same<AccT, int>::value) {
      if (sums) {
        c.z = zero * sum_parts(sums + o, part_stride, parts);
      }
    }
    return c;
  }
  __device__ __forceinline__ Row row(int) const { return Row{a_scale ? __fmul_rn(a_scale[0], w_scale[0]) : sc}; }
  __device__ __forceinline__ float value(AccT v, Row r, Col c) const {
    if constexpr (std::is_same<AccT, int>::value) v -= c.z;
    return __fmaf_rn((float)v, r.sc, c.b);
  }
  __device__ __forceinline__ void store(int m, int n, AccT v, Row r, Col c) const {
    store_from_f32<OUT>(y, (int64_t)m * ldy + n, value(v, r, c));
  }
};

}  // namespace fmsmo
