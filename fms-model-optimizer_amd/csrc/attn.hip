// Operands and products of the quantized attention matmuls (QBmmINT8Deploy): the affine int8 quantizer
// with the column sums that the zero-point correction needs, and the product whose first operand is
// quantized on its way into LDS.
//
// The static per-tensor quantizer of both operands, in the compute dtype T:
//   q = clamp( rint( rnd_T( rnd_T(x / scale) + offset ) ), -128, 127 )
#include "gemm_tile.hpp"
#include "quant_math.hpp"

#include <algorithm>
#include <type_traits>

namespace fmsmo {

// The division by the (scalar) scale without the IEEE sequence where that is exact: the 16-bit
// quotient of quant_i8_pertoken16_kernel when the scale is itself a value of T, the refined fp32
// quotient of the fp16-x / fp32-scale kernel when x is fp16; both need a scale of 2^-60 .. 2^60.
// A quotient that comes out inf or NaN (non-finite x, overflow) is redone with the IEEE division.
struct AffineDiv {
  float s, r, offset;
  bool fast;
  bool packed;  // 16-bit T, and the offset a value of T: affine_codes_packed serves
};
template <int XT, int T>
__device__ __forceinline__ AffineDiv affine_div(float scale, float offset) {
  AffineDiv d;
  d.s = scale;
  d.offset = offset;
  const float m = fabsf(scale);
  d.fast = m >= 8.6736174e-19f && m <= 1.1529215e18f;
  if constexpr (T == FMSMO_F32) {
    d.fast = d.fast && XT == FMSMO_F16;
    d.r = rcp_refined(scale);
    d.packed = d.fast;
  } else {
    d.fast = d.fast && XT == T && round_to<T>(scale) == scale;
    d.r = __builtin_amdgcn_rcpf(scale);
    // (fp16: scale <= 64 and |offset| <= 512 keep 65504 / scale + offset outside the codes; the sign of a
    // negative scale would turn the stand-in of a NaN over)
    d.packed = d.fast && round_to<T>(offset) == offset &&
               (T != FMSMO_F16 || (scale > 0.0f && scale <= 64.0f && fabsf(offset) <= 512.0f));
  }
  return d;
}
template <int T>
__device__ __forceinline__ float affine_code(float e, const AffineDiv& d) {
  float q;
  if (d.fast) {
    if constexpr (T == FMSMO_F32) q = div32_fast(e, d.s, d.r);
    else q = div16<T, false>(e, d.s, d.r);
    if (__builtin_expect(!(fabsf(q) < __builtin_inff()), 0)) q = e / d.s;
  } else {
    q = e / d.s;
  }
  const float t = round_to<T>(__fadd_rn(round_to<T>(q), d.offset));
  return fminf(fmaxf(__builtin_rintf(t), -128.0f), 127.0f);
}
// Two elements (packed as loaded) -> their codes in the low byte of each half, for 16-bit T: seven
// vector operations per element instead of about fifteen.  v_div_fixup gives infinite and NaN
// operands the IEEE quotient; fp16 adds, clamps and rounds on the pair (one rounding of the exact sum,
// the bounds are integers so clamping may come first, + 1536 rounds to nearest even and leaves the
// two's-complement byte in the mantissa), bf16 through fp32.
// (T = fp32: fp16 x and the refined quotient.)
template <int XT, int T>
__device__ __forceinline__ uint32_t affine_codes_packed(uint32_t w, const AffineDiv& d, float nz) {
  if constexpr (T == FMSMO_F16) {
    // infinite and NaN elements become +-65504 (NaN the lower bound, as the later clamp would have it: the
    // minimum hands a NaN on quieted, of which the maximum takes the other operand):
    // with |65504 / scale| beyond any code their quotient clamps to the code of the infinite one, and
    // no v_div_fixup is needed behind a finite dividend.  (As instructions of their own: the compiler
    // puts a quieting v_pk_max in front of a max of loaded values.)
    asm("v_pk_minimum3_f16 %0, %1, %2, %2" : "=v"(w) : "v"(w), "s"(0x7bff7bffu));
    asm("v_pk_max_f16 %0, %1, %2" : "=v"(w) : "v"(w), "s"(0xfbfffbffu));
  }
  const float el = cvt16<XT>((u16)(w & 0xffff)), eh = cvt16<XT>((u16)(w >> 16));
  if constexpr (T == FMSMO_F32) {
    const float tl = __builtin_amdgcn_div_fixupf(div32_fast_mix(el, d.s, d.r, nz), d.s, el) + d.offset;
    const float th = __builtin_amdgcn_div_fixupf(div32_fast_mix(eh, d.s, d.r, nz), d.s, eh) + d.offset;
    const float cl = fminf(fmaxf(tl, -128.0f), 127.0f), ch = fminf(fmaxf(th, -128.0f), 127.0f);
    return __builtin_amdgcn_perm(__float_as_uint(ch + 12582912.0f), __float_as_uint(cl + 12582912.0f), 0x0c040c00u);
  } else {
  float ql = div16_mix<T>(el, d.s, d.r, nz), qh = div16_mix<T>(eh, d.s, d.r, nz);
  if constexpr (T == FMSMO_BF16) {
    ql = __builtin_amdgcn_div_fixupf(ql, d.s, el);
    qh = __builtin_amdgcn_div_fixupf(qh, d.s, eh);
  }
  const uint32_t p = pack16<T>(ql, qh);
  if constexpr (T == FMSMO_F16) {
    hf2 h;
    __builtin_memcpy(&h, &p, 4);
    const _Float16 o = (_Float16)d.offset;
    h = h + hf2{o, o};
    h = __builtin_elementwise_min(__builtin_elementwise_max(h, hf2{(_Float16)-128.0f, (_Float16)-128.0f}),
                                  hf2{(_Float16)127.0f, (_Float16)127.0f});
    h = h + hf2{(_Float16)1536.0f, (_Float16)1536.0f};
    uint32_t r;
    __builtin_memcpy(&r, &h, 4);
    return r;
  } else {
    const uint32_t t = pack16<T>(bf16_to_f32((u16)(p & 0xffff)) + d.offset, bf16_to_f32((u16)(p >> 16)) + d.offset);
    const float lo = fminf(fmaxf(bf16_to_f32((u16)(t & 0xffff)), -128.0f), 127.0f);
    const float hi = fminf(fmaxf(bf16_to_f32((u16)(t >> 16)), -128.0f), 127.0f);
    return __builtin_amdgcn_perm(__float_as_uint(hi + 12582912.0f), __float_as_uint(lo + 12582912.0f), 0x0c040c00u);
  }
  }
}

// 16 bytes at any element boundary (rows of odd length put them there)
typedef int v4i_e2 __attribute__((ext_vector_type(4), aligned(2)));
typedef int v4i_e4 __attribute__((ext_vector_type(4), aligned(4)));

// 8 consecutive elements as loaded: one 16-byte word, two for fp32; elements from `n` on are zero
template <int XT>
struct Raw8 {
  v4i w[XT == FMSMO_F32 ? 2 : 1];
};
template <int XT, bool NT = false>
__device__ __forceinline__ Raw8<XT> load_raw8(const void* p, int n) {
  Raw8<XT> r;
  if (n >= 8) {
    if constexpr (XT == FMSMO_F32) {
      r.w[0] = *(const v4i_e4*)p;
      r.w[1] = *((const v4i_e4*)p + 1);
    } else if constexpr (NT) {
      r.w[0] = __builtin_nontemporal_load((const v4i_e2*)p);
    } else {
      r.w[0] = *(const v4i_e2*)p;
    }
  } else {
    constexpr int W = XT == FMSMO_F32 ? 8 : 4;
#pragma unroll
    for (int i = 0; i < W; ++i) {
      uint32_t v = 0;
      if constexpr (XT == FMSMO_F32) {
        if (i < n) v = ((const uint32_t*)p)[i];
      } else {
        if (2 * i < n) v = ((const u16*)p)[2 * i];
        if (2 * i + 1 < n) v |= (uint32_t)((const u16*)p)[2 * i + 1] << 16;
      }
      r.w[i >> 2][i & 3] = (int)v;
    }
  }
  return r;
}

// the eight codes as two words, codes from `n` on zero
// (ALWAYS: the host has checked what d.packed says)
template <int XT, int T, bool ALWAYS = false>
__device__ __forceinline__ uint2 affine_codes8(const Raw8<XT>& x, int n, const AffineDiv& d, float nz) {
  uint32_t o[2];
  bool done = false;
  if constexpr (XT == T ? XT != FMSMO_F32 : XT == FMSMO_F16) {
    if (ALWAYS || d.packed) {
      uint32_t c[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) c[i] = affine_codes_packed<XT, T>((uint32_t)x.w[0][i], d, nz);
      o[0] = __builtin_amdgcn_perm(c[1], c[0], 0x06040200u);
      o[1] = __builtin_amdgcn_perm(c[3], c[2], 0x06040200u);
      done = true;
    }
  }
  if (!ALWAYS && !done) {
    o[0] = o[1] = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float e;
      if constexpr (XT == FMSMO_F32) e = __int_as_float(x.w[i >> 2][i & 3]);
      else e = cvt16<XT>((u16)((uint32_t)x.w[0][i >> 1] >> ((i & 1) * 16)));
      o[i >> 2] |= ((uint32_t)(int)affine_code<T>(e, d) & 0xffu) << ((i & 3) * 8);
    }
  }
  if (n < 8) {  // (uniform except in a row's last group)
    o[0] &= n >= 4 ? ~0u : n <= 0 ? 0u : (1u << (n * 8)) - 1u;
    o[1] &= n <= 4 ? 0u : (1u << ((n - 4) * 8)) - 1u;
  }
  return make_uint2(o[0], o[1]);
}

__device__ __forceinline__ int sum_codes(uint2 o, int acc) {
  acc = __builtin_amdgcn_sdot4((int)o.x, 0x01010101, acc, false);
  return __builtin_amdgcn_sdot4((int)o.y, 0x01010101, acc, false);
}

// Sum over aligned groups of 2^lg lanes, the same in each of them: within 16 lanes by DPP modifiers of the additions
// (four rows of sums through LDS shuffles took 1.1 us of a launch of a few heads)
__device__ __forceinline__ int group_sum(int v, int lg) {
#define STEP(ctrl) v += __builtin_amdgcn_update_dpp(0, v, ctrl, 0xf, 0xf, true)
  if (lg > 0) STEP(0xb1);   // quad_perm [1,0,3,2]
  if (lg > 1) STEP(0x4e);   // quad_perm [2,3,0,1]
  if (lg > 2) STEP(0x141);  // row_half_mirror
  if (lg > 3) STEP(0x140);  // row_mirror
#undef STEP
  if (lg > 4) v += __shfl_xor(v, 16, 64);
  if (lg > 5) v += __shfl_xor(v, 32, 64);
  return v;
}

template <int XT>
__device__ __forceinline__ const void* elem_ptr(const void* x, size_t i) {
  return (const uint8_t*)x + i * (XT == FMSMO_F32 ? 4 : 2);
}

// q [batch][R][ldq] <- x [batch][R][C], columns past C zero; sums[b][r] = sum of the row's codes.
// 2^LG lanes share a row (a head of 128 elements is 16 groups of eight: 16 lanes, four rows per wave) and
// keep four groups in flight each: of four rows where the lanes hold a whole row (ROWS), else of one row.
// HBM bound.  (One 256-thread block per row, 16 threads of it with work, took 34 us for
// 32 x 2048 x 128 where this takes 8.)
struct AffineOp {
  const void* x;
  int64_t ldx, stride_x;  // elements
  float scale, offset;
  int8_t* q;
  int64_t ldq, stride_q;
  int32_t* sums;
  int R, C;
  int lg, tiles;  // row form: 2^lg lanes per row; transposing form: tiles per block
  int gx, gy;     // blocks along the rows (row form) / tile groups, column tiles (transposing form)
};
template <int XT, int T, bool ROWS>
__device__ __forceinline__ void affine_rows(const AffineOp& g, int bx, int bat) {
  constexpr int U = 4;
  const int64_t ldq = g.ldq;
  const int R = g.R, C = g.C;
  int32_t* const sums = g.sums;
  const int lanes = 1 << g.lg, l = threadIdx.x & (lanes - 1), rows = 256 >> g.lg;
  const int row0 = (ROWS ? U : 1) * bx * rows + (threadIdx.x >> g.lg);
  if (row0 >= R) return;  // whole groups of lanes
  const AffineDiv d = affine_div<XT, T>(g.scale, g.offset);
  const float nz = opaque_neg_zero();
  auto xrow = [&](int r) { return (size_t)bat * g.stride_x + (size_t)min(r, R - 1) * g.ldx; };
  auto qrow = [&](int r) { return g.q + (size_t)bat * g.stride_q + (size_t)r * ldq; };
  auto put_sum = [&](int r, int sum) {
    sum = group_sum(sum, g.lg);
    if (l == 0 && r < R) sums[(size_t)bat * R + r] = sum;
  };
  if constexpr (ROWS) {
    const int c = l * 8;
    Raw8<XT> w[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      w[u] = load_raw8<XT>(elem_ptr<XT>(g.x, xrow(row0 + u * rows) + min(c, C - 1)), C - c);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int r = row0 + u * rows;
      const uint2 o = affine_codes8<XT, T>(w[u], C - c, d, nz);
      if (r < R && c < (int)ldq) *(uint2*)(qrow(r) + c) = o;
      if (sums) put_sum(r, sum_codes(o, 0));
    }
  } else {
    int sum = 0;
    for (int c0 = l * 8; c0 < (int)ldq; c0 += U * lanes * 8) {
      Raw8<XT> w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = c0 + u * lanes * 8;
        w[u] = load_raw8<XT>(elem_ptr<XT>(g.x, xrow(row0) + min(c, C - 1)), C - c);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = c0 + u * lanes * 8;
        if (c < (int)ldq) {
          const uint2 o = affine_codes8<XT, T>(w[u], C - c, d, nz);
          *(uint2*)(qrow(row0) + c) = o;
          sum = sum_codes(o, sum);
        }
      }
    }
    if (sums) put_sum(row0, sum);
  }
}
template <int XT, int T, bool ROWS>
__global__ __launch_bounds__(256) void quant_i8_affine_kernel(AffineOp g) {
  affine_rows<XT, T, ROWS>(g, blockIdx.x, blockIdx.y);
}

// The transposing form: q [batch][C][ldq], q[c][r] = code of x[r][c], rows past R zero.  A block turns
// `tiles` tiles of 64 x 64 in LDS, the next one in flight; a thread owns 4 x 4 elements, turns them in
// registers and writes four words (rows of 76 bytes in LDS: at most two lanes per bank).
// sums[part][b][c]: the block's share of the column sums (added up where they are used: no atomics,
// nothing to clear).  A block whose rows all lie past R (ldq may be padded beyond the last 64 rows of data)
// has no part: fmsmo_affine_sum_parts counts the blocks that begin inside R.
template <int XT>
struct Raw4 {
  uint32_t w[XT == FMSMO_F32 ? 4 : 2];
};
template <int XT>
__device__ __forceinline__ Raw4<XT> load_raw4(const void* p, int n) {
  typedef int v2i_e2 __attribute__((ext_vector_type(2), aligned(2)));
  Raw4<XT> r;
  if (n >= 4) {
    if constexpr (XT == FMSMO_F32) {
      const v4i v = *(const v4i_e4*)p;
      r.w[0] = v[0], r.w[1] = v[1], r.w[2] = v[2], r.w[3] = v[3];
    } else {
      const v2i_e2 v = *(const v2i_e2*)p;
      r.w[0] = v[0], r.w[1] = v[1];
    }
  } else if constexpr (XT == FMSMO_F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) r.w[i] = i < n ? ((const uint32_t*)p)[i] : 0u;
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      uint32_t v = 0;
      if (2 * i < n) v = ((const u16*)p)[2 * i];
      if (2 * i + 1 < n) v |= (uint32_t)((const u16*)p)[2 * i + 1] << 16;
      r.w[i] = v;
    }
  }
  return r;
}
template <int XT, int T>
__device__ __forceinline__ uint32_t affine_codes4(const Raw4<XT>& x, int n, const AffineDiv& d, float nz) {
  uint32_t o = 0;
  bool done = false;
  if constexpr (XT == T ? XT != FMSMO_F32 : XT == FMSMO_F16) {
    if (d.packed) {
      o = __builtin_amdgcn_perm(affine_codes_packed<XT, T>(x.w[1], d, nz), affine_codes_packed<XT, T>(x.w[0], d, nz),
                                0x06040200u);
      done = true;
    }
  }
  if (!done) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float e;
      if constexpr (XT == FMSMO_F32) e = __uint_as_float(x.w[i]);
      else e = cvt16<XT>((u16)(x.w[i >> 1] >> ((i & 1) * 16)));
      o |= ((uint32_t)(int)affine_code<T>(e, d) & 0xffu) << (i * 8);
    }
  }
  return n >= 4 ? o : n <= 0 ? 0u : o & ((1u << (n * 8)) - 1u);
}

template <int XT, int T>
__device__ __forceinline__ void affine_turned(const AffineOp& g, int bx, int by, int bat, int batch) {
  constexpr int LDW = 19;  // words per LDS row [c][r]
  __shared__ uint32_t tile[64 * LDW];
  const int64_t ldq = g.ldq;
  const int R = g.R, C = g.C;
  const int c0 = by * 64, total = (int)(ldq / 64);
  const int t0 = bx * g.tiles, t1 = min(t0 + g.tiles, total);
  const size_t xb = (size_t)bat * g.stride_x;
  const int cl = (threadIdx.x & 15) * 4, rl = (threadIdx.x >> 4) * 4;  // this thread's 4 x 4 of a tile
  const AffineDiv d = affine_div<XT, T>(g.scale, g.offset);
  const float nz = opaque_neg_zero();
  const int oc = threadIdx.x >> 2, chunk = threadIdx.x & 3;
  const int nc = C - (c0 + cl);  // columns left from this thread's first one
  auto load = [&](int t, Raw4<XT> (&w)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = t * 64 + rl + i;
      w[i] = load_raw4<XT>(elem_ptr<XT>(g.x, xb + (size_t)min(r, R - 1) * g.ldx + min(c0 + cl, C - 1)), nc);
    }
  };
  Raw4<XT> cur[4], nxt[4];
  load(t0, cur);
  int sum = 0;
  for (int t = t0; t < t1; ++t) {
    if (t + 1 < t1) load(t + 1, nxt);
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = affine_codes4<XT, T>(cur[i], t * 64 + rl + i < R ? nc : 0, d, nz);
    // bytes [row][column] -> words of four rows of one column
    const uint32_t a = __builtin_amdgcn_perm(o[1], o[0], 0x05010400u), b = __builtin_amdgcn_perm(o[3], o[2], 0x05010400u);
    const uint32_t e = __builtin_amdgcn_perm(o[1], o[0], 0x07030602u), f = __builtin_amdgcn_perm(o[3], o[2], 0x07030602u);
    uint32_t* dst = tile + cl * LDW + (rl >> 2);
    dst[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
    dst[LDW] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    dst[2 * LDW] = __builtin_amdgcn_perm(f, e, 0x05040100u);
    dst[3 * LDW] = __builtin_amdgcn_perm(f, e, 0x07060302u);
    __syncthreads();
    const uint32_t* src = tile + oc * LDW + chunk * 4;
    const uint4 v = make_uint4(src[0], src[1], src[2], src[3]);
    if (c0 + oc < C)
      *(uint4*)((uint8_t*)g.q + (size_t)bat * g.stride_q + (size_t)(c0 + oc) * ldq + t * 64 + chunk * 16) = v;
    sum = sum_codes(make_uint2(v.x, v.y), sum);
    sum = sum_codes(make_uint2(v.z, v.w), sum);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) cur[i] = nxt[i];
  }
  if (g.sums && t0 * 64 < R) {
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    if (chunk == 0 && c0 + oc < C) g.sums[((size_t)bx * batch + bat) * C + c0 + oc] = sum;
  }
}
template <int XT, int T>
__global__ __launch_bounds__(256) void quant_i8_affine_t_kernel(AffineOp g) {
  affine_turned<XT, T>(g, blockIdx.x, blockIdx.y, blockIdx.z, gridDim.z);
}

// Both operands of a product in one launch: blocks [0, split) take the first, row by row, the others the second,
// row by row or transposing it.  A quantizer of 17 MB takes 10 us for 5 us of traffic (one burst of loads, one
// of stores and the launch); two of them behind each other, and for a few heads mostly two launches.
// us, fp16: scores of 32 heads of 2048 x 2048 x 128 (both quantizers and the product) 90 -> 83, 8 heads of 155 x 155 x 80
// 18.7 -> 12.3 (5.3 + 5.6 for the two alone).
template <int XT, int T, bool ROWS, bool TURN>
__global__ __launch_bounds__(256) void quant_i8_affine_pair_kernel(AffineOp a, AffineOp b, int split, int batch) {
  int id = blockIdx.x;
  if (id < split) {  // uniform for the whole block
    const int bat = id / a.gx;
    affine_rows<XT, T, ROWS>(a, id - bat * a.gx, bat);
    return;
  }
  id -= split;
  if constexpr (TURN) {
    const int per = b.gx * b.gy, bat = id / per, r = id - bat * per, by = r / b.gx;
    affine_turned<XT, T>(b, r - by * b.gx, by, bat, batch);
  } else {
    const int bat = id / b.gx;
    affine_rows<XT, T, ROWS>(b, id - bat * b.gx, bat);
  }
}

// sums[0][i] += sums[1 .. parts - 1][i]
__global__ __launch_bounds__(256) void add_parts_kernel(int32_t* sums, int parts, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) sums[i] = sum_parts(sums + i, n, parts);
}

// ------------------------------------------------- product with the first operand quantized on the way
// y[b] = dequant( quant(x[b]) . q2[b]^T ): probabilities x values.  x [M, K] is 16-bit and by far the largest
// operand; quantized by a kernel of its own it is read once, its codes written and read again (2 + 1 + 1
// bytes per element; 114 us for the two launches at 32 heads of 2048 x 2048 x 128, fp16).  Here a block
// reads its rows once, quantizes them in registers and writes the codes into the LDS slab the matrix
// instructions read: 2 bytes per element, 66 - 69 us (4 TB/s; bf16, whose codes take twice the vector
// operations, 113 -> 80).
// 64 x 128 tiles (all columns of a head, so that nothing is quantized twice), slabs of 128 codes, one LDS
// buffer: 24 KiB and 116 registers leave room for four blocks per compute unit, whose loads, vector
// work and matrix work overlap each other (two blocks of 128 x 128 with two buffers and loads two slabs
// ahead: 81 us; three of 128 x 128, one buffer: 76; three of 64 x 128, two buffers: 80).
// The blocks start their reductions at different slabs (rows a power of two apart would otherwise ask
// for the same memory channels at the same time).
constexpr int QA_BM = 64;
struct QaArgs {
  const void* x;
  int64_t ldx, stride_x;  // elements
  float scale, offset;
  const uint8_t* b;
  int64_t ldb, stride_b;
  const int32_t* sums;
  int parts, zero;   // zero point of the codes (offset as an integer)
  float sc;          // product of the two scales
  void* y;
  int64_t ldy;
  int batch, M, N, K;
};

template <int XT, int T>
__global__ __launch_bounds__(256, 4) void bmm_qa_kernel(QaArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int BM = QA_BM, BN = 128, BK = 128, CPR = 8;
  constexpr int NA = BM / 16, NB = 4;  // 16-byte loads per thread and slab
  __shared__ __attribute__((aligned(16))) uint8_t lds[(BM + BN) * BK];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int mt = (g.M + BM - 1) / BM;
  // contiguous tiles per XCD: the row tiles of a head share its second operand in one L2
  int tile, unused;
  tile_of_block(blockIdx.x, gridDim.x, gridDim.x, 1, 1 << 30, tile, unused);
  const int bi = tile / mt, row0 = (tile - bi * mt) * BM;
  const int ns = (g.K + BK - 1) / BK;
  const int s0 = (int)((unsigned)tile * 5u % (unsigned)ns);
  auto slab = [&](int i) {
    int s = min(i, ns - 1) + s0;
    return s >= ns ? s - ns : s;
  };

  const AffineDiv d = affine_div<XT, T>(g.scale, g.offset);
  const float nz = opaque_neg_zero();
  // x: thread -> (row tid / 16 + 16 j, 8 elements tid % 16); rows past M re-read the last one
  const int xr = tid >> 4, xc = (tid & 15) * 8;
  const u16* xbase = (const u16*)g.x + (size_t)bi * g.stride_x;
  const u16* xp[NA];
#pragma unroll
  for (int j = 0; j < NA; ++j) xp[j] = xbase + (size_t)min(row0 + xr + 16 * j, g.M - 1) * g.ldx + xc;
  // codes of the second operand: thread -> (row tid / 8 + 32 j, 16 bytes tid % 8); what lies past its
  // last row reads as zero, what lies past K meets zero codes of x
  const int br = tid >> 3, bc = tid & 7;
  const __amdgpu_buffer_rsrc_t rsrc_b = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(g.b + (int64_t)bi * g.stride_b), 0, (int)((int64_t)g.N * g.ldb), 0x00020000);
  const int vb = br * (int)g.ldb + bc * 16;
  Raw8<XT> sa[NA];
  v4i sb[NB];
  auto load = [&](int s) {
    if (s * BK + BK <= g.K) {  // uniform
#pragma unroll
      for (int j = 0; j < NA; ++j) sa[j] = load_raw8<XT, true>(xp[j] + s * BK, 8);
    } else {
      const int left = g.K - s * BK - xc;  // elements of the row from this thread's first on
#pragma unroll
      for (int j = 0; j < NA; ++j)  // (a group wholly past K is not read; its codes are zeroed below)
        sa[j] = load_raw8<XT, true>(xp[j] + (left > 0 ? s * BK : -xc), left > 0 ? left : 0);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j)
      sb[j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc_b, vb + j * 32 * (int)g.ldb, s * BK, 0));
  };
  uint8_t* wa = lds + xr * BK + (((xc >> 4) ^ swz<CPR, 1>(xr)) * 16) + (xc & 8);
  uint8_t* wb = lds + BM * BK + br * BK + ((bc ^ swz<CPR, 1>(br)) * 16);
  auto stage = [&](int s) {
    if (s * BK + BK <= g.K) {
#pragma unroll
      for (int j = 0; j < NA; ++j) *(uint2*)(wa + j * 16 * BK) = affine_codes8<XT, T, true>(sa[j], 8, d, nz);
    } else {
      const int left = g.K - s * BK - xc;
#pragma unroll
      for (int j = 0; j < NA; ++j) *(uint2*)(wa + j * 16 * BK) = affine_codes8<XT, T, true>(sa[j], left, d, nz);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) *(v4i*)(wb + j * 32 * BK) = sb[j];
  };
  const int fr = lane & 31, fg = lane >> 5, fsw = swz<CPR, 1>(fr);
  // the accumulators start from the zero-point correction, an integer per column
  const int n_base = wn * 64 + fr;
  v16i acc[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = min(n_base + j * 32, g.N - 1);
    const int z = -g.zero * sum_parts(g.sums + (size_t)bi * g.N + n, (int64_t)g.batch * g.N, g.parts);
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[j][v] = z;
  }
  load(slab(0));
  for (int i = 0; i < ns; ++i) {
    __syncthreads();  // every wave has read slab i - 1
    stage(slab(i));
    load(slab(i + 1));
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int pos = ((k * 2 + fg) ^ fsw) * 16;
      const v4i fa = *(const v4i*)(lds + (wm * 32 + fr) * BK + pos);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const v4i fb = *(const v4i*)(lds + BM * BK + (wn * 64 + j * 32 + fr) * BK + pos);
        acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, fb, acc[j], 0, 0, 0);
      }
    }
  }

  // rows m = 8 (v / 4) + 4 (lane / 32) + v % 4, columns n = 32 j + lane % 32 of the wave's 32 x 64
  const int m_base = row0 + wm * 32 + fg * 4;
  const size_t ybase = (size_t)bi * g.M * g.ldy;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int m = m_base + (v >> 2) * 8 + (v & 3);
    if (m < g.M) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n_base + j * 32;
        if (n < g.N) store_from_f32<XT>(g.y, ybase + (size_t)m * g.ldy + n, __fmul_rn((float)acc[j][v], g.sc));
      }
    }
  }
#endif
}

}  // namespace fmsmo

using namespace fmsmo;

int fmsmo_check_launch();

static bool aligned16(const void* p) { return (((uintptr_t)p) & 15) == 0; }

// Tiles of 64 rows per block of the transposing quantizer: one while that makes fewer than 1024
// blocks, then as many as keep about that number (fewer shares of the sums to add up).
static int affine_t_tiles(int64_t batch, int64_t R, int64_t C) {
  return (int)std::max<int64_t>(1, (R + 63) / 64 * ((C + 63) / 64) * batch / 1024);
}
extern "C" int fmsmo_affine_sum_parts(int64_t batch, int64_t R, int64_t C, int transpose) {
  if (!transpose || R <= 0 || C <= 0 || batch <= 0) return 1;
  const int64_t total = (R + 63) / 64, tiles = affine_t_tiles(batch, R, C);
  return (int)((total + tiles - 1) / tiles);
}

// A product adds the parts itself where that is its kernel for a reduction of 128, and for a few query rows: every block
// adds them for its columns again, which takes longer with the rows and the parts, and a launch of their own takes the host 3 us,
// by which an eager call of a few rows is bound: one query, 12 heads, scores and values, launch of their own / inside: 864 x 128
// 37.0 / 33.8 us, 587 x 80 38.6 / 34.7.  Device alone (us from a HIP graph, fp16, 8 heads, one product; 64 columns of values
// where not said): 1 row, 4 parts 10.3 / 9.8, 8 parts 11.0 / 10.6, 21 parts 14.6 / 14.5, 32 parts 17.4 / 17.7, of 128 columns 18.8 / 20.0;
// 8 rows, 4 parts 10.5 / 10.4, 32 parts 17.8 / 18.6; 16 rows, 4 parts 10.8 / 11.5, 32 parts 18.1 / 19.6; 32 rows 11.8 / 13.2,
// 19.2 / 21.4; 64 rows, 4 parts 13.5 / 16.9
extern "C" int fmsmo_affine_parts_first(int parts, int64_t M, int64_t N, int64_t K) {
  const bool inside = (K == 128 && M > 128 && N > 128) || (M <= 8 && parts <= 32);
  return parts > 1 && !inside;
}

extern "C" int fmsmo_affine_add_parts(int32_t* sums, int parts, int64_t n, fmsmo_stream_t stream) {
  if (!sums) return FMSMO_ERR_NULL;
  if (parts < 1 || n <= 0 || n > (1ll << 38)) return FMSMO_ERR_SHAPE;
  if (parts > 1)
    hipLaunchKernelGGL(add_parts_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, sums,
                       parts, n);
  return fmsmo_check_launch();
}

static int check_affine(int x_dtype, int compute_dtype, int transpose, const AffineOp& g) {
  if (g.ldx < g.C || g.stride_x < 0 || g.stride_q < 0) return FMSMO_ERR_SHAPE;
  if (x_dtype < 0 || x_dtype > 2 || compute_dtype < 0 || compute_dtype > 2) return FMSMO_ERR_UNSUPPORTED;
  if (compute_dtype != FMSMO_F32 && compute_dtype != x_dtype) return FMSMO_ERR_UNSUPPORTED;
  if (transpose) {
    if (g.ldq < g.R || g.ldq % 64 || g.stride_q % 16 || !aligned16(g.q)) return FMSMO_ERR_ALIGN;
    if (g.C > 65535 * 64ll || g.ldq > 0x7fffffff) return FMSMO_ERR_SHAPE;
  } else {
    if (g.ldq < g.C || g.ldq % 8 || g.stride_q % 8 || (((uintptr_t)g.q) & 7)) return FMSMO_ERR_ALIGN;
    if (g.ldq > 0x7fffffff) return FMSMO_ERR_SHAPE;
  }
  return (((uintptr_t)g.x) & (x_dtype == FMSMO_F32 ? 3 : 1)) ? FMSMO_ERR_ALIGN : FMSMO_OK;
}
// how an operand is laid over blocks; true: every lane group of the row form holds a whole row
static bool lay_affine(AffineOp& g, int transpose, int64_t batch) {
  if (transpose) {
    g.tiles = affine_t_tiles(batch, g.R, g.C);
    g.gx = div_up(g.ldq / 64, g.tiles);
    g.gy = div_up(g.C, 64);
    return false;
  }
  // lanes per row: one group of eight codes each, at most a wave
  g.lg = 0;
  while (g.lg < 6 && ((int64_t)8 << g.lg) < g.ldq) ++g.lg;
  const bool rows = ((int64_t)8 << g.lg) >= g.ldq;
  g.gx = div_up(g.R, (rows ? 4 : 1) * (256 >> g.lg));
  g.gy = 1;
  return rows;
}
// f<XT, T>() for the dtypes of a call (checked)
template <class F>
static void affine_dtypes(int x_dtype, int compute_dtype, F&& f) {
  typedef std::integral_constant<int, FMSMO_F16> H;
  typedef std::integral_constant<int, FMSMO_BF16> B;
  typedef std::integral_constant<int, FMSMO_F32> S;
  if (compute_dtype == FMSMO_F32) {
    if (x_dtype == FMSMO_F16) f(H{}, S{});
    else if (x_dtype == FMSMO_BF16) f(B{}, S{});
    else f(S{}, S{});
  } else if (x_dtype == FMSMO_F16) {
    f(H{}, H{});
  } else {
    f(B{}, B{});
  }
}

extern "C" int fmsmo_quant_i8_affine_sums(const void* x, int x_dtype, int64_t ldx, int64_t stride_x, float scale,
                                          float offset, int compute_dtype, int transpose, int8_t* q, int64_t ldq,
                                          int64_t stride_q, int32_t* sums, int64_t batch, int64_t R, int64_t C,
                                          fmsmo_stream_t stream) {
  if (!x || !q) return FMSMO_ERR_NULL;
  if (batch <= 0 || R <= 0 || C <= 0 || batch > 65535 || R > 0x7fffffff || C > 0x7fffffff) return FMSMO_ERR_SHAPE;
  AffineOp g{x, ldx, stride_x, scale, offset, q, ldq, stride_q, sums, (int)R, (int)C, 0, 0, 0, 0};
  const int rc = check_affine(x_dtype, compute_dtype, transpose, g);
  if (rc) return rc;
  const bool rows = lay_affine(g, transpose, batch);
  hipStream_t st = (hipStream_t)stream;
  affine_dtypes(x_dtype, compute_dtype, [&](auto xt, auto t) {
    constexpr int XT = decltype(xt)::value, T = decltype(t)::value;
    if (transpose)
      hipLaunchKernelGGL((quant_i8_affine_t_kernel<XT, T>), dim3((unsigned)g.gx, (unsigned)g.gy, (unsigned)batch), dim3(256),
                         0, st, g);
    else if (rows)
      hipLaunchKernelGGL((quant_i8_affine_kernel<XT, T, true>), dim3((unsigned)g.gx, (unsigned)batch), dim3(256), 0, st, g);
    else
      hipLaunchKernelGGL((quant_i8_affine_kernel<XT, T, false>), dim3((unsigned)g.gx, (unsigned)batch), dim3(256), 0, st, g);
  });
  return fmsmo_check_launch();
}

extern "C" int fmsmo_quant_i8_affine_pair(int x_dtype, int compute_dtype, int64_t batch, const void* a, int64_t lda,
                                          int64_t stride_a, float scale_a, float offset_a, int8_t* qa, int64_t stride_qa,
                                          int64_t M, const void* b, int64_t ldb, int64_t stride_b, float scale_b,
                                          float offset_b, int transpose_b, int8_t* qb, int64_t stride_qb, int32_t* sums_b,
                                          int64_t N, int64_t K, int64_t ldq, fmsmo_stream_t stream) {
  if (!a || !b || !qa || !qb) return FMSMO_ERR_NULL;
  if (batch <= 0 || M <= 0 || N <= 0 || K <= 0 || batch > 65535 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff)
    return FMSMO_ERR_SHAPE;
  AffineOp ga{a, lda, stride_a, scale_a, offset_a, qa, ldq, stride_qa, nullptr, (int)M, (int)K, 0, 0, 0, 0};
  AffineOp gb{b, ldb, stride_b, scale_b, offset_b, qb, ldq, stride_qb, sums_b, (int)(transpose_b ? K : N),
              (int)(transpose_b ? N : K), 0, 0, 0, 0};
  int rc = check_affine(x_dtype, compute_dtype, 0, ga);
  if (!rc) rc = check_affine(x_dtype, compute_dtype, transpose_b, gb);
  if (rc) return rc;
  const bool rows = lay_affine(ga, 0, batch);  // (the second operand's rows, not transposed, have the same length)
  lay_affine(gb, transpose_b, batch);
  const int64_t na = ga.gx * batch, nb = (int64_t)gb.gx * gb.gy * batch;
  if (na + nb >= (1ll << 31)) return FMSMO_ERR_UNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)(na + nb)), block(256);
  affine_dtypes(x_dtype, compute_dtype, [&](auto xt, auto t) {
    constexpr int XT = decltype(xt)::value, T = decltype(t)::value;
#define GO(ROWS, TURN) \
  hipLaunchKernelGGL((quant_i8_affine_pair_kernel<XT, T, ROWS, TURN>), grid, block, 0, st, ga, gb, (int)na, (int)batch)
    if (rows && transpose_b) GO(true, true);
    else if (rows) GO(true, false);
    else if (transpose_b) GO(false, true);
    else GO(false, false);
#undef GO
  });
  return fmsmo_check_launch();
}

extern "C" int fmsmo_quant_i8_affine(const void* x, int x_dtype, int64_t ldx, int64_t stride_x,
                                     float scale, float offset, int compute_dtype, int transpose,
                                     int8_t* q, int64_t ldq, int64_t stride_q, int64_t batch,
                                     int64_t R, int64_t C, fmsmo_stream_t stream) {
  return fmsmo_quant_i8_affine_sums(x, x_dtype, ldx, stride_x, scale, offset, compute_dtype, transpose, q, ldq,
                                    stride_q, nullptr, batch, R, C, stream);
}

static bool is_value_of(float v, int dtype) {
  uint32_t b;
  __builtin_memcpy(&b, &v, 4);
  if (dtype == FMSMO_F32) return true;
  if (dtype == FMSMO_BF16) return !(b & 0xffffu);
  const float a = v < 0 ? -v : v;
  if (a >= 0x1p-14f) return a <= 65504.0f && !(b & 0x1fffu);
  return a * 0x1p24f == (float)(int)(a * 0x1p24f);  // subnormal (or zero): a multiple of 2^-24
}

// Which products quantize their first operand on the way: corrected sums that stay in 32 bits
// (zero_sums_fit), all columns in one tile (nothing is
// quantized twice), whole row tiles, a reduction of two slabs or more and an eighth of the compute
// units busy (12 heads of 335 x 335 x 96, 72 tiles: 18.2 -> 11.3 us; 8 of 1501 x 1501 x 80 53 -> 29); and a
// scale and offset that the packed quotient serves.
extern "C" int fmsmo_bmm_qa_ok(int x_dtype, int compute_dtype, float scale, float offset, int64_t batch, int64_t M,
                               int64_t N, int64_t K) {
  const float a = scale < 0 ? -scale : scale;
  if (!(a >= 8.6736174e-19f && a <= 1.1529215e18f) || offset != (float)(int)offset) return 0;
  if (compute_dtype == FMSMO_F32 ? x_dtype != FMSMO_F16
                                 : (x_dtype != compute_dtype || !is_value_of(scale, compute_dtype) ||
                                    !is_value_of(offset, compute_dtype) ||
                                    (compute_dtype == FMSMO_F16 && (scale < 0.0f || a > 64.0f || offset > 512.0f || offset < -512.0f))))
    return 0;
  return zero_sums_fit((int)offset, K) && N <= 128 && K >= 256 && M >= QA_BM && batch * ((M + QA_BM - 1) / QA_BM) >= 32;
}

extern "C" int fmsmo_bmm_qa_i8(const void* x, int x_dtype, int64_t ldx, int64_t stride_x, float scale, float offset,
                               int compute_dtype, const int8_t* b, int64_t ldb, int64_t stride_b, float b_scale,
                               const int32_t* sums, int parts, void* y, int64_t ldy, int64_t batch, int64_t M, int64_t N,
                               int64_t K, fmsmo_stream_t stream) {
  if (!x || !b || !sums || !y) return FMSMO_ERR_NULL;
  if (batch <= 0 || M <= 0 || N <= 0 || K <= 0 || ldx < K || ldb < K || ldy < N || parts < 1 || stride_x < 0 ||
      stride_b < N * ldb)
    return FMSMO_ERR_SHAPE;
  if (!fmsmo_bmm_qa_ok(x_dtype, compute_dtype, scale, offset, batch, M, N, K)) return FMSMO_ERR_UNSUPPORTED;
  if (N > 128 || M >= (1 << 30) || K >= (1 << 30) || N * ldb >= (1ll << 31) || batch * div_up(M, QA_BM) >= (1ll << 31))
    return FMSMO_ERR_UNSUPPORTED;
  if ((((uintptr_t)x) & 1) || ldb % 16 || stride_b % 16 || !aligned16(b)) return FMSMO_ERR_ALIGN;
  QaArgs g{};
  g.x = x; g.ldx = ldx; g.stride_x = stride_x; g.scale = scale; g.offset = offset;
  g.b = (const uint8_t*)b; g.ldb = ldb; g.stride_b = stride_b;
  g.sums = sums; g.parts = parts; g.zero = (int)offset; g.sc = scale * b_scale;
  g.y = y; g.ldy = ldy; g.batch = (int)batch; g.M = (int)M; g.N = (int)N; g.K = (int)K;
  hipStream_t st = (hipStream_t)stream;
  dim3 grid((unsigned)(batch * div_up(M, QA_BM)));
  if (compute_dtype == FMSMO_F32)
    hipLaunchKernelGGL((bmm_qa_kernel<FMSMO_F16, FMSMO_F32>), grid, dim3(256), 0, st, g);
  else if (x_dtype == FMSMO_F16)
    hipLaunchKernelGGL((bmm_qa_kernel<FMSMO_F16, FMSMO_F16>), grid, dim3(256), 0, st, g);
  else
    hipLaunchKernelGGL((bmm_qa_kernel<FMSMO_BF16, FMSMO_BF16>), grid, dim3(256), 0, st, g);
  return fmsmo_check_launch();
}
