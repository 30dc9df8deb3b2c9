// Products of a few tokens (M <= 64) with weights of any K that is a multiple of 16: the weight-streaming decode
// kernel for the reductions that skinny.hip holds no instance of, with its quantizer inside for the smallest calls.
//
//   * a block owns groups of 16 weight rows (dealt out in units of 8, one block per compute unit); its NW waves take the
//     128-byte steps of K in turn, so that the block reads NW x 128 consecutive bytes of a row at a time;
//   * weights and activations come through buffer descriptors that end with the block's last row and with token row
//     M - 1: rows and 16-byte chunks past the end get an offset outside and read as zero, without a branch and without
//     traffic, and no K and no share of a block needs a form of its own;
//   * per step the 16 rows (two loads of 8 rows x 128 bytes) pass through a wave-private LDS buffer into the layout of
//     the 16 x 16 matrix instructions.  A wave has one step of loads in flight: with 8 or 16 waves two, three or four were
//     slower or the same at all but two of 18 shapes (3 x 2176 x 7808, 8 waves: 7.9 us with four steps, 9.8 with eight).
#include "gemv_args.hpp"
#include <algorithm>

namespace fmsmo {

// e4m3 on the fp16 instruction: codes widened to fp16 (exact), sums that keep what fp32 additions keep, which those of the
// e4m3 instruction, 64 elements and more at a time, do not
constexpr int GEMV_FP8_F16 = 6;
// It serves K % 64 != 0, as on the tiles, and one and two tokens of rows from 1024 on, whose other kernel adds in fp32: the weights'
// traffic bounds these (us, e4m3 instruction | this, one token, N = 3072 / 16384: K = 11008 10.7 / 36.7 | 10.9 / 37.1; two tokens,
// 1408 4.3 / 8.0 | 4.4 / 8.5, 4608 - / 16.2 | - / 17.4).
static bool e4m3_on_fp16(const GemvArgs& g) { return g.K % 64 || (g.M <= 2 && g.K >= 1024); }
// per token (int8: with divisors of the 16-bit dtype, or none), with fp32 divisors, static per tensor
enum { QUANT_TOKEN, QUANT_TOKEN_F32S, QUANT_STATIC };
constexpr unsigned GEMV_OUTSIDE = 0x80000000u;  // past the end of every descriptor made here
constexpr int UNIT = 512;                       // elements of a token row that a wave quantizes at a time

// ------------------------------------------------------------------ quantizers, in units of one wave
// Unit u holds the elements [seg UNIT, (seg + 1) UNIT) of token row m, u = m nseg + seg; wave w takes u = w, w + NW, ...
// Units never cross a row, so any number of rows of any length is dealt to the waves evenly.  The codes of a row lie
// xs bytes apart in LDS, those past K are zero.
template <int NW, int UPW>
struct Units {
  int M, nseg, count, nchunk;
  int wave, lane;
  __device__ __forceinline__ Units(const GemvArgs& g) {
    M = g.M;
    nseg = (g.K + UNIT - 1) / UNIT;
    count = M * nseg;
    nchunk = g.K / AQ_VEC;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = threadIdx.x & 63;
  }
  __device__ __forceinline__ int unit(int i) const { return wave + i * NW; }
  __device__ __forceinline__ int row(int i) const { return unit(i) / nseg; }
  __device__ __forceinline__ int chunk(int i) const { return (unit(i) - row(i) * nseg) * (UNIT / AQ_VEC) + lane; }
  __device__ __forceinline__ bool has(int i) const { return unit(i) < count; }
  // the largest of a row's entries in red (bit patterns of non-negative floats order like the floats, NaN above inf)
  __device__ __forceinline__ uint32_t row_max(const uint32_t* red, int m) const {
    return wave_max_u32(red[m * nseg + min(lane, nseg - 1)]);
  }
};

template <int NW, int UPW>
__device__ __forceinline__ void units_request(const GemvArgs& g, const Units<NW, UPW>& U, v4i (&cur)[UPW]) {
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    cur[i] = v4i{0, 0, 0, 0};
    if (U.has(i) && U.chunk(i) < U.nchunk)
      cur[i] = *(const v4i*)(g.x16 + (size_t)U.row(i) * g.ldx + (size_t)U.chunk(i) * AQ_VEC);
  }
}

// magnitudes of a packed pair, largest so far
__device__ __forceinline__ us2 pair_max(us2 a, int w) {
  const uint32_t mag = (uint32_t)w & 0x7fff7fffu;
  us2 m2;
  __builtin_memcpy(&m2, &mag, 4);
  return __builtin_elementwise_max(a, m2);
}

// Per-token int8 in a 16-bit compute dtype T: the arithmetic of the stand-alone quantizer (see rows_finish_i8).
// red: NW * UPW words, then NW floats for the IEEE routine; sc: the token scales
template <int T, int NW, int UPW>
__device__ __forceinline__ void units_i8(const GemvArgs& g, const Units<NW, UPW>& U, v4i (&cur)[UPW], const v4i (&sm)[UPW],
                                         uint8_t* xq, int xs, float* sc, uint32_t* red) {
  constexpr uint32_t INF_BITS = T == FMSMO_F16 ? 0x7c00u : 0x7f80u;
  const float floor_T = cvt16<T>(to16<T>(1e-5f));
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    if (!U.has(i)) continue;
    int bad = 0;
    us2 amax2 = {0, 0};
    if (U.chunk(i) < U.nchunk) {
      if (g.smooth) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t w = (uint32_t)cur[i][q], d = (uint32_t)sm[i][q];
          const float dl = cvt16<T>((u16)(d & 0xffff)), dh = cvt16<T>((u16)(d >> 16));
          if constexpr (T == FMSMO_BF16)
            bad |= !(fabsf(dl) >= 8.6736174e-19f && fabsf(dl) <= 1.1529215e18f) ||
                   !(fabsf(dh) >= 8.6736174e-19f && fabsf(dh) <= 1.1529215e18f);
          const u16 el = to16<T>(div16<T, false>(cvt16<T>((u16)(w & 0xffff)), dl, __builtin_amdgcn_rcpf(dl)));
          const u16 eh = to16<T>(div16<T, false>(cvt16<T>((u16)(w >> 16)), dh, __builtin_amdgcn_rcpf(dh)));
          cur[i][q] = (int)((uint32_t)el | ((uint32_t)eh << 16));
        }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) amax2 = pair_max(amax2, cur[i][q]);
    }
    // (a divisor outside the fast path's range marks the row for the IEEE routine)
    const uint32_t v = wave_max_u32(bad ? 0xffffu : (uint32_t)(amax2[0] > amax2[1] ? amax2[0] : amax2[1]));
    if (U.lane == 0) red[U.unit(i)] = v;
  }
  __syncthreads();
  static_assert(NW * UPW <= 64, "one lane per unit");
  // units of rows that the fast path does not cover (the same in every wave)
  const uint64_t off = __ballot(U.lane < U.count && red[min(U.lane, U.count - 1)] >= INF_BITS);
  auto row_off = [&](int m) { return (off >> (m * U.nseg) & (U.nseg >= 64 ? ~0ull : (1ull << U.nseg) - 1)) != 0; };
  if (off)
    for (int m = 0; m < U.M; ++m)  // by the whole block, with scratch of their own
      if (row_off(m))
        quant_i8_row_ieee16<T, NW * 64>(g.x16 + (size_t)m * g.ldx, g.smooth, g.saturate, (int8_t*)(xq + (size_t)m * xs),
                                        sc + m, g.K, (float*)(red + NW * UPW));
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    if (!U.has(i)) continue;
    const int m = U.row(i), c = U.chunk(i);
    const bool ieee = off && row_off(m);
    uint2 o = make_uint2(0, 0);
    if (!ieee) {
      const float s = cvt16<T>(to16<T>(fmaxf(cvt16<T>((u16)U.row_max(red, m)), floor_T) / 127.0f));
      const float rcp_s = __builtin_amdgcn_rcpf(s);
      if (c == 0) sc[m] = s;
      uint32_t code[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t w = (uint32_t)cur[i][q];
        float ql = div16<T, false>(cvt16<T>((u16)(w & 0xffff)), s, rcp_s);
        float qh = div16<T, false>(cvt16<T>((u16)(w >> 16)), s, rcp_s);
        if (g.saturate) {
          ql = fminf(fmaxf(ql, -127.0f), 127.0f);
          qh = fminf(fmaxf(qh, -127.0f), 127.0f);
        }
        code[q] = rint_codes<T>(to16<T>(ql), to16<T>(qh));
      }
      o = make_uint2(__builtin_amdgcn_perm(code[1], code[0], 0x06040200u),
                     __builtin_amdgcn_perm(code[3], code[2], 0x06040200u));
    }
    // (chunks past K hold zeros and get the code of zero; of an IEEE row only those are written here)
    if (!ieee || c >= U.nchunk) *(uint2*)(xq + (size_t)m * xs + (size_t)c * AQ_VEC) = o;
  }
}

// The same with fp32 SmoothQuant divisors: the whole quantizer in fp32 (see rows_finish_i8_f32s).
// red: 2 * NW * UPW words
template <int XT, int NW, int UPW>
__device__ __forceinline__ void units_i8_f32s(const GemvArgs& g, const Units<NW, UPW>& U, const v4i (&cur)[UPW],
                                              const float (&sd)[UPW][8], uint8_t* xq, int xs, float* sc, uint32_t* red) {
  const float nz = opaque_neg_zero();
  int bad = 0;
#pragma unroll
  for (int i = 0; i < UPW; ++i)
#pragma unroll
    for (int q = 0; q < 8; ++q) {  // (chunks past the row hold ones)
      const float a = fabsf(sd[i][q]);
      bad |= !(a >= 8.6736174e-19f && a <= 1.1529215e18f);  // outside 2^-60 .. 2^60, or NaN
    }
  const bool ieee_block = __syncthreads_or(bad) != 0;
  float e[UPW][8];
  // e <- x / smooth, the largest |e| of the unit into buf (a thread's maximum drops NaN)
  auto divide = [&](int i, bool ieee, uint32_t* buf) {
    float amax = 0.0f;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float xv = cvt16<XT>((u16)((uint32_t)cur[i][q >> 1] >> ((q & 1) * 16)));
      e[i][q] = ieee ? xv / sd[i][q] : div32_fast_mix(xv, sd[i][q], rcp_refined(sd[i][q]), nz);
      amax = fmaxf(amax, fabsf(e[i][q]));
    }
    const uint32_t b = wave_max_u32(__float_as_uint(amax) & 0x7fffffffu);
    if (U.lane == 0) buf[U.unit(i)] = b;
  };
  auto row_ieee = [&](uint32_t bits) {
    const float amax = __uint_as_float(bits);
    bool ieee = ieee_block || !(amax < __builtin_inff());
    if constexpr (XT == FMSMO_BF16) ieee = ieee || (amax != 0.0f && amax < 8.271806e-25f);
    return ieee;
  };
#pragma unroll
  for (int i = 0; i < UPW; ++i)
    if (U.has(i)) divide(i, ieee_block, red);
  __syncthreads();
  uint32_t bits[UPW];
  int again = 0;
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    bits[i] = 0;
    if (!U.has(i)) continue;
    bits[i] = U.row_max(red, U.row(i));
    again |= !ieee_block && row_ieee(bits[i]);
  }
  uint32_t* red2 = red + NW * UPW;
  if (__syncthreads_or(again)) {  // redo those rows with IEEE divisions
#pragma unroll
    for (int i = 0; i < UPW; ++i)
      if (U.has(i) && row_ieee(bits[i])) divide(i, true, red2);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    if (!U.has(i)) continue;
    const int m = U.row(i), c = U.chunk(i);
    const bool ieee = row_ieee(bits[i]);
    const uint32_t abits = ieee && !ieee_block ? U.row_max(red2, m) : bits[i];
    const float s = fmaxf(__uint_as_float(abits), 1e-5f) / 127.0f;
    const float rcp_s = rcp_refined(s);
    if (c == 0) sc[m] = s;
    uint32_t code[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      float r = ieee ? e[i][q] / s : div32_fast(e[i][q], s, rcp_s);
      if (g.saturate) r = fminf(fmaxf(r, -127.0f), 127.0f);
      code[q] = __float_as_uint(r + 12582912.0f);  // rounds to even, two's complement in the low mantissa bits
    }
    uint32_t o[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t lo = __builtin_amdgcn_perm(code[4 * h + 1], code[4 * h], 0x0c0c0400u);
      const uint32_t hi = __builtin_amdgcn_perm(code[4 * h + 3], code[4 * h + 2], 0x0c0c0400u);
      o[h] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
    }
    const uint2 v = c < U.nchunk ? make_uint2(o[0], o[1]) : make_uint2(0, 0);
    *(uint2*)(xq + (size_t)m * xs + (size_t)c * AQ_VEC) = v;
  }
}

// e4m3, the FP8Linear token recipe (see rows_finish_fp8).  red: NW * UPW words
template <int XT, int NW, int UPW>
__device__ __forceinline__ void units_fp8(const GemvArgs& g, const Units<NW, UPW>& U, const v4i (&cur)[UPW], uint8_t* xq,
                                          int xs, float* sc, uint32_t* red) {
  constexpr uint32_t INF_BITS = XT == FMSMO_F16 ? 0x7c00u : 0x7f80u;
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    if (!U.has(i)) continue;
    us2 amax2 = {0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) amax2 = pair_max(amax2, cur[i][q]);
    const uint32_t v = wave_max_u32((uint32_t)(amax2[0] > amax2[1] ? amax2[0] : amax2[1]));
    if (U.lane == 0) red[U.unit(i)] = v;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    if (!U.has(i)) continue;
    const int m = U.row(i), c = U.chunk(i);
    const uint32_t abits = U.row_max(red, m);
    const float s = fmaxf(cvt16<XT>((u16)abits) / 448.0f, 1e-12f);
    if (c == 0) sc[m] = s;
    float t[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float xv = cvt16<XT>((u16)((uint32_t)cur[i][q >> 1] >> ((q & 1) * 16)));
      t[q] = fminf(fmaxf(xv / s, -448.0f), 448.0f);
    }
    uint8_t* dst = xq + (size_t)m * xs;
    if (abits < INF_BITS) {
      int o0 = 0, o1 = 0;
      o0 = __builtin_amdgcn_cvt_pk_fp8_f32(t[0], t[1], o0, false);
      o0 = __builtin_amdgcn_cvt_pk_fp8_f32(t[2], t[3], o0, true);
      o1 = __builtin_amdgcn_cvt_pk_fp8_f32(t[4], t[5], o1, false);
      o1 = __builtin_amdgcn_cvt_pk_fp8_f32(t[6], t[7], o1, true);
      *(uint2*)(dst + (size_t)c * AQ_VEC) = make_uint2((uint32_t)o0, (uint32_t)o1);
    } else {
      uint8_t b[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) b[q] = c < U.nchunk ? f32_to_e4m3_sw(t[q]) : 0;
      store8(dst, (size_t)c * AQ_VEC, b);
    }
  }
}

// Static per-tensor int8 (FMSMO_SQ_FMO in fp32): no maxima, no scales to hand over.
template <int XT, int NW, int UPW>
__device__ __forceinline__ void units_static(const GemvArgs& g, const Units<NW, UPW>& U, const v4i (&cur)[UPW], uint8_t* xq,
                                             int xs) {
  const float nz = opaque_neg_zero();
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    if (!U.has(i)) continue;
    const int c = U.chunk(i);
    uint32_t code[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      code[q] = static_fmo32_codes<XT>((uint32_t)cur[i][q], g.q_lo, g.q_hi, g.q_step, g.q_rcp, g.q_zp, g.q_shift, nz);
    const uint2 o = make_uint2(__builtin_amdgcn_perm(code[1], code[0], 0x06040200u),
                               __builtin_amdgcn_perm(code[3], code[2], 0x06040200u));
    *(uint2*)(xq + (size_t)U.row(i) * xs + (size_t)c * AQ_VEC) = c < U.nchunk ? o : make_uint2(0, 0);
  }
}

// ------------------------------------------------------------------ the product
__device__ __forceinline__ h8 widen_fp8(int a, int b) {
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  const h2 p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(a, 1.0f, false), p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(a, 1.0f, true);
  const h2 p2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b, 1.0f, false), p3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(b, 1.0f, true);
  return h8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}
template <int OP, class Acc4>
__device__ __forceinline__ Acc4 gemv_mma(v4i w0, v4i w1, v4i x0, v4i x1, Acc4 acc) {
  if constexpr (OP == FMSMO_OP_I8) {
    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w0, x0, acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(w1, x1, acc, 0, 0, 0);
  } else if constexpr (OP == FMSMO_OP_E4M3) {
    const v8i w = {w0[0], w0[1], w0[2], w0[3], w1[0], w1[1], w1[2], w1[3]};
    const v8i x = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w, x, acc, 0, 0, 0, 0, 0, 0);
  } else {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(widen_fp8(w0[0], w0[1]), widen_fp8(x0[0], x0[1]), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(widen_fp8(w0[2], w0[3]), widen_fp8(x0[2], x0[3]), acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(widen_fp8(w1[0], w1[1]), widen_fp8(x1[0], x1[1]), acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(widen_fp8(w1[2], w1[3]), widen_fp8(x1[2], x1[3]), acc, 0, 0, 0);
  }
}
// The waves' parts of a sum in pairs, and pairs of pairs: a rounding per level, where one after the other takes one per wave
// (e4m3, one token, 4096 x 11008, error in the 2-norm 7.3e-8 -> 5.6e-8, the row kernel's 5.5e-8).
template <int NW, class F>
__device__ __forceinline__ auto sum_waves(const F& part) {
  decltype(part(0)) p[NW];
#pragma unroll
  for (int w = 0; w < NW; ++w) p[w] = part(w);
#pragma unroll
  for (int d = 1; d < NW; d *= 2)
#pragma unroll
    for (int w = 0; w + d < NW; w += 2 * d) p[w] += p[w + d];
  return p[0];
}

// XT >= 0: the activations are x16 (of that dtype), UPW units of them per wave quantized by every block for itself, in
// LDS, while the head of its weight stream is in flight, by the quantizer QUANT.
template <int OP, int NW, int MT = 1, int XT = -1, int UPW = 1, int QUANT = QUANT_TOKEN>
__global__ __launch_bounds__(NW * 64) void gemv_any_kernel(GemvArgs g, int halves) {
  constexpr bool FUSED = XT >= 0, SF32 = QUANT == QUANT_TOKEN_F32S, STATIC = QUANT == QUANT_STATIC;
  static_assert(!FUSED || MT == 1, "the fused form serves one tile of tokens");
  typedef typename std::conditional<OP == FMSMO_OP_I8, int, float>::type AccT;
  typedef AccT Acc4 __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(16))) uint8_t xq[FUSED ? NW * UPW * UNIT + 16 * 16 : 16];
  __shared__ float xsc[16];
  __shared__ uint32_t xred[FUSED ? 2 * NW * UPW + NW : 1];
  __shared__ __attribute__((aligned(16))) uint8_t stage[NW][2048];
  __shared__ AccT red[2][NW][256 * MT];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kg = lane >> 4;
  const int h_lo = (int)(((int64_t)blockIdx.x * halves) / gridDim.x);
  const int h_hi = (int)(((int64_t)(blockIdx.x + 1) * halves) / gridDim.x);
  const int row_lo = h_lo * 8, row_hi = min(h_hi * 8, g.N);  // this block's weight rows
  const int gcount = (h_hi - h_lo + 1) >> 1;                 // groups of 16 rows, the last maybe half
  const int kchunks = g.K >> 4;

  // weight loads: lane -> (row = lane / 8 [+ 8], 16-byte chunk = lane % 8).  Steps at `wlim` and beyond are past K for
  // this lane's chunk.
  const int drow = lane >> 3, dpos = lane & 7;
  const int wlim = (kchunks - dpos + 7) >> 3;
  const unsigned woff = (unsigned)drow * (unsigned)g.ldb + dpos * 16, woff8 = woff + 8u * (unsigned)g.ldb;
  auto weights = [&](int gi) {  // the rows of group gi (past the block's last group: nothing)
    const int row0 = row_lo + gi * 16, rows = min(16, row_hi - row0);
    return __builtin_amdgcn_make_buffer_rsrc((void*)(g.b + (int64_t)min(row0, g.N - 1) * g.ldb), 0,
                                             rows > 0 ? (rows - 1) * (int)g.ldb + g.K : 0, 0x00020000);
  };
  auto load_w = [&](__amdgpu_buffer_rsrc_t rs, int s, v4i (&w)[2]) {
    const unsigned k = (unsigned)s * 128u;
    const bool in = s < wlim;
    w[0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs, in ? woff + k : GEMV_OUTSIDE, 0, 2));
    w[1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rs, in ? woff8 + k : GEMV_OUTSIDE, 0, 2));
  };
  // activation fragments: lane (token r of the tile, kg) takes chunks kg and kg + 4 of a step
  const unsigned xrow = g.M > 1 ? (unsigned)g.lda : (unsigned)g.K;  // (of one token the stride means nothing)
  const __amdgpu_buffer_rsrc_t rsrc_x =
      __builtin_amdgcn_make_buffer_rsrc((void*)g.a, 0, FUSED ? 0 : (g.M - 1) * (int)xrow + g.K, 0x00020000);
  const int xlim0 = (kchunks - kg + 7) >> 3, xlim1 = (kchunks - kg + 3) >> 3;
  const unsigned xoff = (unsigned)r * xrow + kg * 16;
  auto load_x = [&](int s, v4i (&x)[MT][2]) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const unsigned v = xoff + t * 16 * xrow + (unsigned)s * 128u;
      x[t][0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, s < xlim0 ? v : GEMV_OUTSIDE, 0, 0));
      x[t][1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_x, s < xlim1 ? v + 64 : GEMV_OUTSIDE, 0, 0));
    }
  };
  // staging: row-major [16 rows][128 B], chunk c of row q stored at position c ^ (q % 8)
  const int wr0 = drow * 128 + ((dpos ^ drow) * 16), wr1 = wr0 + 8 * 128;
  const int rr = r & 7;
  const int rd0 = r * 128 + ((kg ^ rr) * 16), rd1 = r * 128 + (((4 + kg) ^ rr) * 16);

  // The static scale as it lies in memory, for the stores: requested ahead of the operands, by a vector load, which no
  // barrier waits for (us, bf16 scale, this | a number in the arguments: 2 x 640 x 1408 4.8 | 4.5, 2 x 4082 x 1152 5.3 | 5.0)
  uint32_t a_word = 0;
  if constexpr (STATIC)
    a_word = __builtin_amdgcn_raw_buffer_load_b32(
        __builtin_amdgcn_make_buffer_rsrc((void*)((uintptr_t)g.a_src & ~(uintptr_t)3), 0, g.a_src ? 4 : 0, 0x00020000), 0, 0, 0);
  v4i wb[2], xb[MT][2];
  const Units<NW, UPW> U(g);
  const int xs = U.nseg * UNIT + 16;
  v4i qcur[FUSED ? UPW : 1], qsm[FUSED && !SF32 && !STATIC ? UPW : 1];
  float qsd[SF32 ? UPW : 1][8];
  if constexpr (FUSED) {
#pragma unroll
    for (int i = 0; i < UPW; ++i) {
      const bool in = U.has(i) && U.chunk(i) < U.nchunk;
      if constexpr (SF32) {
#pragma unroll
        for (int q = 0; q < 8; ++q) qsd[i][q] = 1.0f;
        if (in) load8<FMSMO_F32>(g.smooth, (size_t)U.chunk(i) * AQ_VEC, qsd[i]);
      } else if constexpr (!STATIC) {
        qsm[i] = v4i{0, 0, 0, 0};
        if (in && g.smooth) qsm[i] = *(const v4i*)(g.smooth + (size_t)U.chunk(i) * AQ_VEC);
      }
    }
    units_request<NW, UPW>(g, U, qcur);
  } else {
    load_x(wave, xb);
  }
  __amdgpu_buffer_rsrc_t rc = weights(0), rn = weights(1);
  load_w(rc, wave, wb);

  const int em = min((int)(threadIdx.x & 15), g.M - 1);
  float as;
  if constexpr (FUSED) {
    if constexpr (STATIC) units_static<XT, NW, UPW>(g, U, qcur, xq, xs);
    else if constexpr (SF32) units_i8_f32s<XT, NW, UPW>(g, U, qcur, qsd, xq, xs, xsc, xred);
    else if constexpr (OP == FMSMO_OP_I8) units_i8<XT, NW, UPW>(g, U, qcur, qsm, xq, xs, xsc, xred);
    else units_fp8<XT, NW, UPW>(g, U, qcur, xq, xs, xsc, xred);
    __syncthreads();
    if constexpr (!STATIC) gemv_put_scales(g, xsc);
    as = STATIC ? g.a_value : xsc[em];
  } else {
    as = g.a_scale ? g.a_scale[g.a_stride ? em : 0] : 1.f;
  }
  // LDS: codes of this lane's token row (rows past M: any, they only reach output columns past M)
  const uint8_t* xl = xq + (FUSED ? min(r, g.M - 1) * xs + kg * 16 : 0);
  const int steps = (g.K + 127) / 128;
  uint8_t* st = &stage[wave][0];

  for (int gi = 0; gi < gcount; ++gi) {
    const int en = min(row_lo + gi * 16 + (int)((threadIdx.x >> 4) & 15), g.N - 1);
    const float ws = g.w_scale ? g.w_scale[g.w_stride ? en : 0] : 1.f;
    const float bv = gemv_bias(g, en);
    Acc4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = Acc4{0, 0, 0, 0};
    for (int s = wave; s < steps; s += NW) {
      // the step that takes this one's registers: the wave's next one, or its first of the next group (none after the
      // block's last group)
      const bool last = s + NW >= steps;
      const int sn = !last ? s + NW : gi + 1 < gcount ? wave : 1 << 24;
      *(v4i*)(st + wr0) = wb[0];
      *(v4i*)(st + wr1) = wb[1];
      __builtin_amdgcn_sched_barrier(0);  // keep the refill right behind the registers it frees
      load_w(last ? rn : rc, sn, wb);
      __builtin_amdgcn_sched_barrier(0);
      const v4i w0 = *(const v4i*)(st + rd0);
      const v4i w1 = *(const v4i*)(st + rd1);
      if constexpr (FUSED) {
        acc[0] = gemv_mma<OP>(w0, w1, *(const v4i*)(xl + s * 128), *(const v4i*)(xl + s * 128 + 64), acc[0]);
      } else {
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = gemv_mma<OP>(w0, w1, xb[t][0], xb[t][1], acc[t]);
        __builtin_amdgcn_sched_barrier(0);
        load_x(sn, xb);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    rc = rn;
    rn = weights(gi + 2);
    // acc[v] = partial C(n = 16 gi + 4 kg + v, m = r) of this wave's steps; two exchange buffers, one barrier per group
    AccT* mine = &red[gi & 1][wave][0];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) mine[t * 256 + (kg * 4 + v) * 16 + r] = acc[t][v];
    __syncthreads();
    static_assert(MT == 1 || (NW * 64) % 256 == 0, "outputs of a thread must share its column");
    for (int e = threadIdx.x; e < 256 * MT; e += NW * 64) {
      const int n = row_lo + gi * 16 + ((e >> 4) & 15), m = (e >> 8) * 16 + (e & 15);
      const AccT sum = sum_waves<NW>([&](int w) { return red[gi & 1][w][e]; });
      float am = as;
      if constexpr (STATIC) am = g.a_src ? scalar_of_word(a_word, (uintptr_t)g.a_src, g.a_src_dtype) : as;
      if (MT > 1) am = g.a_scale ? g.a_scale[g.a_stride ? min(m, g.M - 1) : 0] : 1.f;
      if (n < row_hi && m < g.M) gemv_store(g, m, n, sum, am, ws, bv);
    }
  }
}

// Up to 16 tokens of rows of at most 512: a wave takes one step of 128 and has all its loads out at once, straight into the operand registers; no
// staging, no loop.  A launch this short is bound by its latency (the chip reads 4 MB in 0.6 us): RG row groups of 16 to a block, so that
// there are up to 1024 blocks of them.  us, gemv_any_kernel -> this: int8 12 x 4230 x 256 5.1 -> 3.9, 1 x 3087 x 512 4.2 -> 3.6, 16 x 6655 x 512 6.1 -> 4.5.
template <int OP, int NW, int RG>
__global__ __launch_bounds__(NW * 64) void gemv_short_kernel(GemvArgs g) {
  typedef typename std::conditional<OP == FMSMO_OP_I8, int, float>::type AccT;
  typedef AccT Acc4 __attribute__((ext_vector_type(4)));
  __shared__ AccT red[NW][RG][16 * 17];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * (RG * 16), rows = min(RG * 16, g.N - n0);
  const int kchunks = g.K >> 4, c0 = wave * 8 + kg, c1 = c0 + 4;
  // (rows and chunks past the end read as zeros; rows of tokens past M only reach outputs that are not stored)
  const __amdgpu_buffer_rsrc_t rw =
      __builtin_amdgcn_make_buffer_rsrc((void*)(g.b + (int64_t)n0 * g.ldb), 0, (rows - 1) * (int)g.ldb + g.K, 0x00020000);
  const unsigned xrow = g.M > 1 ? (unsigned)g.lda : (unsigned)g.K;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)g.a, 0, (g.M - 1) * (int)xrow + g.K, 0x00020000);
  const unsigned wo = (unsigned)r * (unsigned)g.ldb, xo = (unsigned)min(r, g.M - 1) * xrow;
  v4i w[RG][2], x[2];
#pragma unroll
  for (int i = 0; i < RG; ++i) {
    const unsigned v = wo + (unsigned)(i * 16) * (unsigned)g.ldb;
    w[i][0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, c0 < kchunks ? v + c0 * 16 : GEMV_OUTSIDE, 0, 2));
    w[i][1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, c1 < kchunks ? v + c1 * 16 : GEMV_OUTSIDE, 0, 2));
  }
  x[0] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rx, c0 < kchunks ? xo + c0 * 16 : GEMV_OUTSIDE, 0, 0));
  x[1] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rx, c1 < kchunks ? xo + c1 * 16 : GEMV_OUTSIDE, 0, 0));
  // the scales and biases of this thread's outputs, with the operands
  constexpr int OUT = (RG * 256 + NW * 64 - 1) / (NW * 64);
  float as[OUT], ws[OUT], bv[OUT];
#pragma unroll
  for (int q = 0; q < OUT; ++q) {
    const int o = threadIdx.x + q * NW * 64, n = min(n0 + ((o >> 8) * 16) + (o & 15), g.N - 1), m = min((o >> 4) & 15, g.M - 1);
    as[q] = g.a_scale ? g.a_scale[g.a_stride ? m : 0] : 1.f;
    ws[q] = g.w_scale ? g.w_scale[g.w_stride ? n : 0] : 1.f;
    bv[q] = gemv_bias(g, n);
  }
#pragma unroll
  for (int i = 0; i < RG; ++i) {
    const Acc4 acc = gemv_mma<OP>(w[i][0], w[i][1], x[0], x[1], Acc4{0, 0, 0, 0});
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][i][(kg * 4 + v) * 17 + r] = acc[v];  // (n = 4 kg + v, m = r)
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < OUT; ++q) {
    const int o = threadIdx.x + q * NW * 64, i = o >> 8, n = n0 + i * 16 + (o & 15), m = (o >> 4) & 15;
    if (i >= RG || n >= g.N || m >= g.M) continue;
    const int e = (o & 15) * 17 + m;
    const AccT sum = sum_waves<NW>([&](int v) { return red[v][i][e]; });
    gemv_store(g, m, n, sum, as[q], ws[q], bv[q]);
  }
}

}  // namespace fmsmo

using namespace fmsmo;

int fmsmo_check_launch();
// skinny.hip: the fused forms of its kernels, or the one here
int fmsmo_decode_fused(int op, int x_dtype, const GemvArgs& g, hipStream_t st);
bool fmsmo_gemv_stream_k(int64_t K);

// Waves per block and blocks of a launch.  us, int8, waves x most blocks 16 x 256 | 8 x 256 | 8 x 512 | 4 x 1024:
//   up to 512 halves of row groups (N = 4096) a group per block, 16 waves, 8 where K has no more than that many steps:
//     1 x 3000: K = 1024 3.7 | 3.4, 2048 3.9 | 4.1, 7168 6.5 | 7.7; 16 x 3000: K = 2048 4.1 | 4.5, 8192 8.7 | 8.9
//   up to 1024 halves, several groups per block, whose ends two blocks per compute unit cover for each other:
//     4 x 6144: K = 2048 5.4 | - | 5.1, 8192 11.4 | - | 10.7
//   more of them a group per block again, whatever their number: a wave has one step of loads in flight, and up to four blocks of eight waves fit a unit.
//     Weights from HBM, at most 512 blocks (K = 768: 1024) | a group per block: 4 x 9216: K = 768 5.7 | 4.9, 1280 7.1 | 5.9, 2816 10.3 | 8.4; 10 x 11776: 1536 7.9 | 6.6,
//     2304 9.8 | 8.1; e4m3 2 x 9216 x 2304 9.7 | 7.7; 4 x 28672: K = 2560 0.93 of the time, 5376 0.90
//     With the quantizer inside, which every block repeats, as before (static 3 x 16384 x 864 7.1 | 8.7, e4m3 1 x 24576 x 896 8.3 | 10.0).
//   But on long rows, and from eleven tokens on beyond K = 2560, the activations that every block reads again weigh more: 4 x 9000 x 10880 1.08 of the
//   time, 16 x 13000 x 5376 1.04; long rows as up to 512 halves: 1 x 20000 x 7168 25.5 | - | 26.0, 8192 27.5 | - | 29.1
struct AnyPlan {
  int nw, blocks;
};
static AnyPlan any_plan(int64_t M, int64_t N, int64_t K, bool fused) {
  const int64_t steps = (K + 127) / 128, halves = (N + 7) / 8;
  const bool wide = steps > 8 && M <= 32;  // (four tiles of tokens have no LDS for 16 waves' sums)
  if (halves <= 512) return {wide ? 16 : 8, 256};
  // (65536 blocks: a launch holds less than 2^32 threads)
  if (!fused && halves > 1024 && K < 6144 && M <= (K <= 2560 ? 16 : 10)) return {steps <= 6 ? 4 : 8, (int)std::min<int64_t>((halves + 1) / 2, 65536)};
  if (fused && M <= 16 && steps <= 6 && halves > 1024) return {4, 1024};
  if (wide && M <= 16 && K >= 6144 && halves > 1024) return {16, 256};
  return {8, 512};
}

// Up to 16 tokens: every K that skinny.hip has no instance for, except short rows over more columns than one round of blocks takes, where tiles of
// 64 x 64 or 32 x 128 with their deeper loads win.  us with the tokens' quantizer, weights from HBM, tiles | this kernel:
//   up to 16384 columns: int8 2 x 9216 x 640 8.1 | 7.4, 5 x 9216 x 768 (e4m3) 8.8 | 8.1, 4 x 14336 x 1152 10.4 | 10.3, 5 x 14336 x 1536 11.9 | 10.9, 5 x 11008 x 2816 16.1 | 13.7 (e4m3 16.5 | 13.6),
//     16 x 9216 x 2816 14.9 | 14.7; K % 128 != 0 10 x 9216 x 3600 18.2 | 18.5, 16 x 9216 x 3600 18.3 | 20.2
//   more: 5 x 24576 x 1536 14.0 | 14.4, 10 x 24576 x 2176 16.9 | 18.6, 10 x 24576 x 2816 19.8 | 20.2, 10 x 18944 x 4480 (e4m3) 26.4 | 25.9, 16 x 24576 x 3584 23.8 | 26.6;
//     K % 128 != 0 5 x 18944 x 1616 16.4 | 14.9, 10 x 18944 x 3600 28.4 | 26.4, 16 x 18944 x 1616 16.8 | 16.8
//   rows of 512 at most, gemv_short_kernel (products alone, weights in cache): 4 x 17166 x 512 5.5 | 5.6, 8 x 10848 x 448 5.0 | 4.4, 16 x 26612 x 512 6.2 | 7.0, 4 x 53216 x 256 6.5 | 7.1
// More tokens: where the tiled kernels would take slices of K or launch too few tiles.  Products alone, weights in cache, tiles | this kernel, int8:
//   17 x 4096: K = 528 5.6 | 3.7, 1536 8.3 | 4.4, 4480 10.2 | 7.2, 9088 13.5 | 11.0; 32 x 1000: 896 5.1 | 3.9, 2304 7.4 | 5.8, 4480 8.2 | 8.4; 32 x 4096 x 4480 10.7 | 8.8;
//   40 x 2100: 896 7.1 | 4.8, 3328 9.3 | 8.4; from 48 tokens on, and e4m3 from 33 on, 64 x 64 tiles: 33 x 2081 x 1536 6.9 | 6.4, 48 x 3256 x 1280 6.7 | 6.7, 64 x 1857 x
//   1792 7.4 | 7.9, e4m3 33 x 2277 x 1152 5.6 | 6.1, 64 x 1776 x 1792 6.4 | 7.9
//   From 4096 columns on 64 x 64 tiles fill the chip in one pass (32 x 8192 x 1536 6.6 | 7.2).  Longer rows: the activations that every block reads
//   again cost more than the slices' sums (32 x 1000 x 6144 9.0 | 9.4).
bool fmsmo_gemv_any_ok(int64_t M, int64_t N, int64_t K, bool fp8) {
  if (M < 1 || M > 64 || K % 16) return false;
  if (fp8 && M == 2 && K >= 1024 && K % 128 == 0) return true;  // (the tiles' e4m3 instruction keeps fewer bits)
  if (M <= 16) {
    if (M == 1 || N <= (K <= 512 ? 24576 : 8192) || fmsmo_gemv_stream_k(K)) return true;
    if (M > 10 && (K % 128 || N > 16384)) return K > 4608;
    return K > (N <= 16384 ? (M <= 10 ? 512 : 1024) : K % 128 ? 1024 : 2304);
  }
  if (N > 4096) return false;
  if (M <= 32) return K <= (M > 24 ? 4096 : fp8 ? 6144 : 8192);
  return K % 128 ? K <= 1024 : !fp8 && M <= 48 && N > 1024 && K > 640 && K <= 2304;
}

// 32-bit offsets into the rows of a block (four groups at most) and into the activations
static bool any_offsets_ok(const GemvArgs& g) {
  return (std::min(g.N, 64) - 1) * g.ldb + g.K < (1ll << 31) && (g.M > 1 ? (g.M - 1) * g.lda : 0) + g.K < (1ll << 31);
}

template <int OP, int MT, int XT = -1, int QUANT = QUANT_TOKEN>
static int any_launch(const GemvArgs& g, hipStream_t st) {
  const AnyPlan p = any_plan(g.M, g.N, g.K, XT >= 0);
  const int halves = (g.N + 7) / 8;
  const dim3 grid((unsigned)std::min(halves, p.blocks));
  // (fused: 64 units of 512 elements with 16 waves, which the host's rule keeps to, 32 with 8, 16 with 4)
  constexpr int UPW = XT >= 0 ? 4 : 1;
  const int units = g.M * ((g.K + UNIT - 1) / UNIT);
  // Launches that no rule leads to have no instance: per-token int8 with its quantizer leaves N > 8192 to the row kernel, and with fp32
  // divisors stops at K = 1024
  constexpr bool TOKEN_I8 = XT >= 0 && OP == FMSMO_OP_I8 && QUANT != QUANT_STATIC;
  if constexpr (MT == 1 && !TOKEN_I8) {
    if (p.nw == 4 && units <= 4 * UPW) {
      hipLaunchKernelGGL((gemv_any_kernel<OP, 4, MT, XT, UPW, QUANT>), grid, dim3(256), 0, st, g, halves);
      return fmsmo_check_launch();
    }
  }
  if constexpr (MT <= 2 && QUANT != QUANT_TOKEN_F32S) {
    if (p.nw == 16 || (XT >= 0 && units > 8 * UPW)) {
      if (XT >= 0 && units > 16 * UPW) return FMSMO_ERR_UNSUPPORTED;
      hipLaunchKernelGGL((gemv_any_kernel<OP, 16, MT, XT, UPW, QUANT>), grid, dim3(1024), 0, st, g, halves);
      return fmsmo_check_launch();
    }
  }
  if (XT >= 0 && units > 8 * UPW) return FMSMO_ERR_UNSUPPORTED;
  hipLaunchKernelGGL((gemv_any_kernel<OP, 8, MT, XT, UPW, QUANT>), grid, dim3(512), 0, st, g, halves);
  return fmsmo_check_launch();
}

template <int OP, int NW>
static int short_launch(const GemvArgs& g, hipStream_t st) {
  const int groups = (g.N + 15) / 16;
  const dim3 block(NW * 64);
  if (groups > 2048) hipLaunchKernelGGL((gemv_short_kernel<OP, NW, 4>), dim3((unsigned)((groups + 3) / 4)), block, 0, st, g);
  else if (groups > 1024) hipLaunchKernelGGL((gemv_short_kernel<OP, NW, 2>), dim3((unsigned)((groups + 1) / 2)), block, 0, st, g);
  else hipLaunchKernelGGL((gemv_short_kernel<OP, NW, 1>), dim3((unsigned)groups), block, 0, st, g);
  return fmsmo_check_launch();
}
template <int OP>
static int short_waves(const GemvArgs& g, hipStream_t st) {
  return g.K <= 128 ? short_launch<OP, 1>(g, st) : g.K <= 256 ? short_launch<OP, 2>(g, st) : short_launch<OP, 4>(g, st);
}

// FMSMO_ERR_UNSUPPORTED: offsets past 32 bits (nothing was launched)
int fmsmo_gemv_any(int op, const GemvArgs& g, hipStream_t st) {
  if (!any_offsets_ok(g)) return FMSMO_ERR_UNSUPPORTED;
  if (g.M <= 16 && g.K <= 512)
    return op == FMSMO_OP_I8 ? short_waves<FMSMO_OP_I8>(g, st)
           : e4m3_on_fp16(g) ? short_waves<GEMV_FP8_F16>(g, st)
                             : short_waves<FMSMO_OP_E4M3>(g, st);
#define GO(OP)                                    \
  if (g.M <= 16) return any_launch<OP, 1>(g, st); \
  if (g.M <= 32) return any_launch<OP, 2>(g, st); \
  return any_launch<OP, 4>(g, st)
  if (op == FMSMO_OP_I8) { GO(FMSMO_OP_I8); }
  if (e4m3_on_fp16(g)) { GO(GEMV_FP8_F16); }
  GO(FMSMO_OP_E4M3);
#undef GO
}

template <int XT>
static int any_fused(int op, const GemvArgs& g, hipStream_t st) {
  if (op == FMSMO_OP_I8) {
    if (g.smooth && g.smooth_f32) return any_launch<FMSMO_OP_I8, 1, XT, QUANT_TOKEN_F32S>(g, st);
    return any_launch<FMSMO_OP_I8, 1, XT>(g, st);
  }
  if (e4m3_on_fp16(g)) return any_launch<GEMV_FP8_F16, 1, XT>(g, st);
  return any_launch<FMSMO_OP_E4M3, 1, XT>(g, st);
}
// the fused form; FMSMO_ERR_UNSUPPORTED: offsets past 32 bits, or more rows and elements than a block quantizes
int fmsmo_gemv_any_fused(int op, int x_dtype, const GemvArgs& g, hipStream_t st) {
  if (g.M > 16 || !any_offsets_ok(g)) return FMSMO_ERR_UNSUPPORTED;
  return x_dtype == FMSMO_F16 ? any_fused<FMSMO_F16>(op, g, st) : any_fused<FMSMO_BF16>(op, g, st);
}

// ------------------------------------------------------------------ quantizer and product in one launch, any K
// One token, and a few short ones.  Every block quantizes all of them, which more tokens or longer rows make longer than the
// launch it saves, and blocks with several row groups hide it worse.  us, quantizer + product -> one launch, int8 from
// fp16 with SmoothQuant, N = 4096: one token K = 10240 12.9 -> 11.6, 16384 17.6 -> 19.1; two tokens K = 1024 5.9 -> 4.9, 3072 7.7 -> 6.8, 5376 9.7 -> 9.3, 7168 11.2 -> 10.5 (N = 1024 8.5 -> 8.9); three 2048 6.6 -> 6.3,
// 5376 9.8 -> 10.7; four 1024 5.8 -> 4.9, 3072 7.7 -> 7.8; six 512 5.7 -> 4.8, 1024 5.9 -> 6.1; eight 512 5.7 -> 4.8, 1024 5.9 -> 6.3; N = 12000: three
// tokens 640 7.4 -> 8.8, 2048 9.5 -> 10.5.  e4m3 and int8 without SmoothQuant: the same or up to 25 % better.  fp32 divisors: 1 x 1024 5.8 -> 5.7,
// 4 x 512 5.7 -> 5.7, 1 x 2048 6.4 -> 7.4.
// (Those N = 4096 times had the product that streamed such K then; against the present ones and other N, see fmsmo_small_linear_better.)
extern "C" int fmsmo_small_linear_ok(int64_t M, int64_t N, int64_t K, int smooth_f32) {
  if (M < 1 || N < 1 || K < 16 || K % 16 || N >= (1 << 30)) return 0;
  if (smooth_f32 ? fmsmo_decode_linear_f32s_ok(M, K) : fmsmo_decode_linear_ok(M, K)) return 1;
  if (smooth_f32) return M <= 16 && K <= 1024 && M * K <= 2048 && N <= 8192;
  if (M == 1) return K <= 12288;
  return N <= 8192 && (M <= 4 ? M * K <= 12288 : M <= 8 && K <= 512);
}

// Where one launch is the better one of those it takes: 1.  2: where a second launch and its buffers cost the host 3 us, the calls that keep
// the GPU longer but still take less of its time than two calls take of the host's (int8, whose results are the same bits either way).  Weights from HBM,
// us on the GPU, one launch | two calls:
//   int8, one token: 640 x 8208 8.7 | 7.3, 640 x 12288 10.1 | 7.2, 5504 x 12288 22.6 | 17.9, 4096 x 10240 12.4 | 12.6; up to K = 8192 0.5 .. 1.9 less,
//     over 5504 columns and more down to the same
//   e4m3, one token: 640 x 12288 10.5 | 9.0, 1024 x 9216 9.1 | 8.6, 2048 x 9216 10.4 | 10.2, 3072 x 9216 10.6 | 12.2; 7168 x 4352 12.8 | 11.1, 8192 x 6144 16.2 |
//     14.0, 11008 x 7168 22.9 | 20.8, 11008 x 6144 17.3 | 17.6, 7168 x 3072 9.4 | 9.0
//   two tokens, int8: 1024 x 3072 6.3 | 6.1, 256 x 4224 7.3 | 6.9, 4096 x 4224 8.8 | 9.5, 6144 x 3072 9.4 | 8.7, 6144 x 4224 13.2 | 10.9, 1024 x 6144 8.5 | 7.5; e4m3: 6144 x
//     5376 15.1 | 13.8, 6144 x 4224 12.1 | 11.9, 1024 x 6144 8.7 | 7.8
//   three, int8: 6144 x 3072 11.5 | 10.4, 6144 x 2304 10.2 | 9.6, 6144 x 1152 8.1 | 7.5; four: 6144 x 3072 12.9 | 10.7, 6144 x 1152 8.2 | 7.4, 6144 x 1024 6.8 | 6.9, 2048 x
//     2048 6.6 | 5.9, 2048 x 2304 7.1 | 7.2; e4m3 6144 x 3072 11.5 | 9.7, 6144 x 2304 9.9 | 9.2; six, int8: 6144 x 256 6.2 | 5.0, 4096 x 256 4.7 | 4.8
//   fp32 divisors: 1 x 6793 x 512 7.0 | 5.5, 1 x 6144 x 640 7.1 | 6.7, 2 x 4096 x 512 5.4 | 4.9, 2 x 6144 x 512 7.1 | 5.6, 2 x 6144 x 1024 7.3 | 7.1, 6 x 2048 x 256 5.9 | 4.7
// (eager, weights in cache: int8 4 x 2048 x 1024 6.0 | 9.3, 6 x 256 x 6144 6.2 | 9.4 - 10.4, 1 x 11264 x 640 9.1 | 9.2 - 10.0; e4m3 1 x 4992 x 7168 10.9 | 9.6 - 10.0)
extern "C" int fmsmo_small_linear_better(int fp8, int64_t M, int64_t N, int64_t K, int smooth_f32) {
  if (!fmsmo_small_linear_ok(M, N, K, smooth_f32)) return 0;
  if (smooth_f32 ? fmsmo_decode_linear_f32s_ok(M, K) : fmsmo_decode_linear_ok(M, K)) return 1;
  if (smooth_f32) return K > 512 && (M <= 2 || N <= 4096) ? 1 : 2;
  if (fp8) {
    if (M == 1) return K > 8192 ? N > 2048 : N <= 4096 || K <= (N > 8192 ? 6144 : 4096);
    return N <= 4096 || K <= (M == 2 ? 4608 : M == 3 ? 4096 : 2304);
  }
  if (M == 1) return K <= 8192 ? 1 : N <= 2048 ? 2 : 0;
  if (N > 4096) {
    if (K > (M == 2 ? 3072 : 2304)) return 0;
    return K <= (M == 2 ? 2048 : M <= 4 ? 1024 : 0) ? 1 : 2;
  }
  if (M == 2) return K <= (N > 2048 ? 4608 : 3072) ? 1 : 2;
  return M == 4 && fmsmo_gemv_stream_k(K) && K > 1024 ? 2 : 1;
}

static int small_linear(int op, const void* x, int x_dtype, int64_t ldx, const void* smooth, int smooth_dtype, const void* w,
                        int64_t ldw, const float* w_scale, int64_t w_scale_n, const void* bias, int bias_dtype, int epilogue,
                        void* y, int y_dtype, int64_t ldy, float* a_scale_out, float* clips, int64_t M, int64_t N, int64_t K,
                        fmsmo_stream_t stream) {
  if (!x || !w || !w_scale || !y) return FMSMO_ERR_NULL;
  if (M <= 0 || N <= 0 || K <= 0 || (M > 1 && ldx < K) || ldw < K || ldy < N) return FMSMO_ERR_SHAPE;
  if (w_scale_n != 1 && w_scale_n != N) return FMSMO_ERR_SHAPE;
  if (x_dtype != FMSMO_F16 && x_dtype != FMSMO_BF16) return FMSMO_ERR_UNSUPPORTED;
  const bool sf32 = smooth && smooth_dtype == FMSMO_F32;
  if (smooth && !sf32 && smooth_dtype != x_dtype) return FMSMO_ERR_UNSUPPORTED;
  if (!fmsmo_small_linear_ok(M, N, K, sf32)) return FMSMO_ERR_UNSUPPORTED;
  if (N * ldw >= (fmsmo_decode_linear_ok(M, K) ? 1ll << 40 : 1ll << 31)) return FMSMO_ERR_UNSUPPORTED;
  if (y_dtype < 0 || y_dtype > 2 || (bias && (bias_dtype < 0 || bias_dtype > 2))) return FMSMO_ERR_UNSUPPORTED;
  if (epilogue < FMSMO_EPI_REF_F16 || epilogue > FMSMO_EPI_F32_MULADD) return FMSMO_ERR_UNSUPPORTED;
  if ((M > 1 && ldx % 8) || ldw % 16 || (((uintptr_t)x) & 15) || (((uintptr_t)w) & 15) || (smooth && (((uintptr_t)smooth) & 15)))
    return FMSMO_ERR_ALIGN;
  GemvArgs g{};
  g.b = (const uint8_t*)w; g.ldb = ldw;
  g.M = (int)M; g.N = (int)N; g.K = (int)K;
  g.w_scale = w_scale; g.w_stride = w_scale_n == 1 ? 0 : 1;
  g.bias = bias; g.bias_dtype = bias_dtype; g.epi = epilogue;
  g.y = y; g.y_dtype = y_dtype; g.ldy = ldy;
  g.x16 = (const u16*)x; g.ldx = ldx; g.smooth = (const u16*)smooth;
  g.smooth_f32 = sf32 ? 1 : 0;
  g.a_scale_out = a_scale_out;
  g.clips = clips;
  return fmsmo_decode_fused(op, x_dtype, g, (hipStream_t)stream);
}

extern "C" int fmsmo_small_linear_i8(const void* x, int x_dtype, int64_t ldx, const void* smooth, int smooth_dtype,
                                     const int8_t* w, int64_t ldw, const float* w_scale, int64_t w_scale_n, const void* bias,
                                     int bias_dtype, int epilogue, void* y, int y_dtype, int64_t ldy, float* a_scale_out,
                                     float* clips, int64_t M, int64_t N, int64_t K, fmsmo_stream_t stream) {
  return small_linear(FMSMO_OP_I8, x, x_dtype, ldx, smooth, smooth_dtype, w, ldw, w_scale, w_scale_n, bias, bias_dtype, epilogue,
                      y, y_dtype, ldy, a_scale_out, clips, M, N, K, stream);
}

extern "C" int fmsmo_small_linear_fp8(const void* x, int x_dtype, int64_t ldx, const uint8_t* w, int64_t ldw,
                                      const float* w_scale, int64_t w_scale_n, const void* bias, int bias_dtype, void* y,
                                      int y_dtype, int64_t ldy, float* a_scale_out, int64_t M, int64_t N, int64_t K,
                                      fmsmo_stream_t stream) {
  return small_linear(FMSMO_OP_E4M3, x, x_dtype, ldx, nullptr, x_dtype, w, ldw, w_scale, w_scale_n, bias, bias_dtype,
                      FMSMO_EPI_F32, y, y_dtype, ldy, a_scale_out, nullptr, M, N, K, stream);
}

// Static activations: no reduction in front of the codes, so more of them than per token, but no form of the row kernel for one long
// token.  us, quantizer + product -> one launch, N = 1024 / 4096: 1 x 2048 5.9 / 6.1 -> 4.4 / 5.0, 3072 5.9 / 6.6 -> 5.0 / 5.7, 5376 5.9 / 8.1 -> 6.3 / 7.6; 4 x 3072
// 6.5 / 7.1 -> 6.0 / 6.5, 4096 6.6 / 8.4 -> 6.9 / 8.6; 8 x 2048 6.6 / 6.6 -> 6.0 / 6.3, 3072 6.6 / 7.2 -> 7.6 / 7.8; 16 x 640 6.4 / 6.4 -> 6.0 / 6.2, 2048 6.5 / 6.5 -> 8.2 / 8.3; N =
// 12000: 4 x 1024 7.7 -> 6.9, 2048 9.3 -> 9.5, 12 x 640 7.7 -> 11.2.
extern "C" int fmsmo_small_linear_static_ok(int64_t M, int64_t N, int64_t K, float step, float zp, float clip_lo, float clip_hi) {
  if (M < 1 || M > 16 || N < 1 || K < 16 || K % 16 || N >= (1 << 30)) return 0;
  return K <= 3072 && M * ((K + UNIT - 1) / UNIT) <= 32 && (N <= 8192 || (M <= 4 && K <= 1024)) &&
         static_fmo32_ok(clip_lo, clip_hi, step, zp);
}
static int small_linear_static(const void* x, int x_dtype, int64_t ldx, float step, float zp, int sym, float clip_lo,
                               float clip_hi, float a_value, const void* a_src, int a_src_dtype, const int8_t* w, int64_t ldw,
                               const float* w_scale, int64_t w_scale_n, const void* bias, int bias_dtype, int epilogue, void* y,
                               int y_dtype, int64_t ldy, int64_t M, int64_t N, int64_t K, fmsmo_stream_t stream) {
  if (!x || !w || !w_scale || !y) return FMSMO_ERR_NULL;
  if (M <= 0 || N <= 0 || K <= 0 || (M > 1 && ldx < K) || ldw < K || ldy < N) return FMSMO_ERR_SHAPE;
  if (w_scale_n != 1 && w_scale_n != N) return FMSMO_ERR_SHAPE;
  if (x_dtype != FMSMO_F16 && x_dtype != FMSMO_BF16) return FMSMO_ERR_UNSUPPORTED;
  if (!fmsmo_small_linear_static_ok(M, N, K, step, zp, clip_lo, clip_hi)) return FMSMO_ERR_UNSUPPORTED;
  if (N * ldw >= (1ll << 31)) return FMSMO_ERR_UNSUPPORTED;
  if (y_dtype < 0 || y_dtype > 2 || (bias && (bias_dtype < 0 || bias_dtype > 2))) return FMSMO_ERR_UNSUPPORTED;
  if (epilogue < FMSMO_EPI_REF_F16 || epilogue > FMSMO_EPI_F32_MULADD) return FMSMO_ERR_UNSUPPORTED;
  if ((M > 1 && ldx % 8) || ldw % 16 || (((uintptr_t)x) & 15) || (((uintptr_t)w) & 15)) return FMSMO_ERR_ALIGN;
  GemvArgs g{};
  g.b = (const uint8_t*)w; g.ldb = ldw;
  g.M = (int)M; g.N = (int)N; g.K = (int)K;
  g.w_scale = w_scale; g.w_stride = w_scale_n == 1 ? 0 : 1;
  g.bias = bias; g.bias_dtype = bias_dtype; g.epi = epilogue;
  g.y = y; g.y_dtype = y_dtype; g.ldy = ldy;
  g.x16 = (const u16*)x; g.ldx = ldx;
  g.q_lo = clip_lo; g.q_hi = clip_hi; g.q_step = step; g.q_rcp = 1.0f / step; g.q_zp = zp; g.q_shift = 128 - (sym ? 1 : 0);
  g.a_value = a_value; g.a_src = a_src; g.a_src_dtype = a_src_dtype;
  if (!any_offsets_ok(g)) return FMSMO_ERR_UNSUPPORTED;
  return x_dtype == FMSMO_F16 ? any_launch<FMSMO_OP_I8, 1, FMSMO_F16, QUANT_STATIC>(g, (hipStream_t)stream)
                              : any_launch<FMSMO_OP_I8, 1, FMSMO_BF16, QUANT_STATIC>(g, (hipStream_t)stream);
}
extern "C" int fmsmo_small_linear_i8_static(const void* x, int x_dtype, int64_t ldx, float step, float zp, int sym, float clip_lo,
                                            float clip_hi, float a_scale, const int8_t* w, int64_t ldw, const float* w_scale,
                                            int64_t w_scale_n, const void* bias, int bias_dtype, int epilogue, void* y,
                                            int y_dtype, int64_t ldy, int64_t M, int64_t N, int64_t K, fmsmo_stream_t stream) {
  return small_linear_static(x, x_dtype, ldx, step, zp, sym, clip_lo, clip_hi, a_scale, nullptr, 0, w, ldw, w_scale, w_scale_n,
                             bias, bias_dtype, epilogue, y, y_dtype, ldy, M, N, K, stream);
}
extern "C" int fmsmo_small_linear_i8_static_scale(const void* x, int x_dtype, int64_t ldx, float step, float zp, int sym,
                                                  float clip_lo, float clip_hi, const void* a_scale, int a_scale_dtype,
                                                  const int8_t* w, int64_t ldw, const float* w_scale, int64_t w_scale_n,
                                                  const void* bias, int bias_dtype, int epilogue, void* y, int y_dtype,
                                                  int64_t ldy, int64_t M, int64_t N, int64_t K, fmsmo_stream_t stream) {
  if (!a_scale) return FMSMO_ERR_NULL;
  if (a_scale_dtype < 0 || a_scale_dtype > 2) return FMSMO_ERR_UNSUPPORTED;
  if ((uintptr_t)a_scale % (a_scale_dtype == FMSMO_F32 ? 4 : 2)) return FMSMO_ERR_ALIGN;
  return small_linear_static(x, x_dtype, ldx, step, zp, sym, clip_lo, clip_hi, 0.0f, a_scale, a_scale_dtype, w, ldw, w_scale,
                             w_scale_n, bias, bias_dtype, epilogue, y, y_dtype, ldy, M, N, K, stream);
}
