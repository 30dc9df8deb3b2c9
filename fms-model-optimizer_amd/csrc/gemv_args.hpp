// Operands of the decode (skinny-M) kernels and the epilogue they share.
#pragma once
#include "quant_math.hpp"

namespace fmsmo {

struct GemvArgs {
  const uint8_t* a;  // [M,K] quantized activations
  const uint8_t* b;  // [N,K] quantized weights
  int64_t lda, ldb;
  int M, N, K;
  const float* a_scale;
  const float* w_scale;
  int a_stride, w_stride;
  const void* bias;
  int bias_dtype;
  int epi;  // FMSMO_EPI_*
  void* y;
  int y_dtype;
  int64_t ldy;
  // fused decode linear: the activations arrive unquantized (fp16 / bf16) and every block
  // quantizes them itself
  const u16* x16;       // [M,K]
  int64_t ldx;
  const u16* smooth;    // [K] SmoothQuant divisors of x's dtype (fp32 when smooth_f32), or NULL
  int smooth_f32;
  int saturate;
  float* a_scale_out;   // [M] per-token scales (written by block 0), or NULL
  // static per-tensor quantizer (see fmsmo_quant_act_i8_static_t, FMSMO_SQ_FMO in fp32): clip values, step and its
  // reciprocal, zero point, 128 - sym, and the scale that the sums are dequantized with: read from a_src, or a_value
  float q_lo, q_hi, q_step, q_rcp, q_zp, a_value;
  int q_shift;
  const void* a_src;    // scalar of a_src_dtype, or NULL
  int a_src_dtype;
  float* clips;         // [2][M] the clip values they stand for, scale * 127 and its negative, or NULL
};

// block 0 of a fused kernel hands out the token scales
__device__ __forceinline__ void gemv_put_scales(const GemvArgs& g, const float* sc) {
  const int m = threadIdx.x;
  if (blockIdx.x != 0 || m >= g.M) return;
  if (g.a_scale_out) g.a_scale_out[m] = sc[m];
  if (g.clips) {
    const float a = __fmul_rn(sc[m], 127.0f);
    g.clips[m] = a;
    g.clips[g.M + m] = -a;
  }
}

// bias of output column n (no bias: -0, whose addition changes nothing, not even the sign of a zero product)
__device__ __forceinline__ float gemv_bias(const GemvArgs& g, int n) {
  if (!g.bias) return -0.f;
  return scalar_f32(g.bias, g.bias_dtype, n);
}

// y[m, n] from a sum over K, its token and weight scales and its bias
template <class AccT>
__device__ __forceinline__ void gemv_store(const GemvArgs& g, int m, int n, AccT sum, float as, float ws, float bv) {
  float out;
  if (g.epi == FMSMO_EPI_REF_F16) {
    const float sc = round_to<FMSMO_F16>(__fmul_rn(as, ws));
    out = __fadd_rn(__fmul_rn((float)sum, sc), bv);
    if (g.y_dtype != FMSMO_F32) out = round_to<FMSMO_F16>(out);
  } else if (g.epi == FMSMO_EPI_F32_MULADD) {
    out = __fadd_rn(__fmul_rn((float)sum, __fmul_rn(as, ws)), bv);
  } else {
    out = __fmaf_rn((float)sum, __fmul_rn(as, ws), bv);
  }
  const int64_t idx = (int64_t)m * g.ldy + n;
  if (g.epi == EPI_RAW_I32) ((int*)g.y)[idx] = (int)sum;
  else if (g.y_dtype == FMSMO_F16) ((u16*)g.y)[idx] = f32_to_f16(out);
  else if (g.y_dtype == FMSMO_BF16) ((u16*)g.y)[idx] = f32_to_bf16(out);
  else ((float*)g.y)[idx] = out;
}

}  // namespace fmsmo
