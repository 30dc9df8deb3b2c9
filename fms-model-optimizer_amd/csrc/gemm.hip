// Host launchers of the tiled MFMA GEMMs (int8 -> int32, int8 / e4m3 with fused dequantizing
// epilogue, grouped mixture-of-experts variant).
#include "gemm_launch.hpp"
#include <mutex>

thread_local char g_fmsmo_last_error[256] = {0};

int fmsmo_check_launch() {
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) return FMSMO_OK;
  snprintf(g_fmsmo_last_error, sizeof(g_fmsmo_last_error), "%s", hipGetErrorString(e));
  return FMSMO_ERR_LAUNCH;
}

unsigned long long*& fmsmo_clock_probe() {
  static thread_local unsigned long long* probe = nullptr;
  return probe;
}
extern "C" int fmsmo_debug_clock_probe(uint64_t* dev6) {
  if (((uintptr_t)dev6) & 7) return FMSMO_ERR_ALIGN;
  fmsmo_clock_probe() = (unsigned long long*)dev6;
  return FMSMO_OK;
}

extern "C" int fmsmo_abi_version(void) { return FMSMO_ABI_VERSION; }
extern "C" const char* fmsmo_last_error(void) { return g_fmsmo_last_error; }
extern "C" const char* fmsmo_status_str(int s) {
  switch (s) {
    case FMSMO_OK: return "ok";
    case FMSMO_ERR_NULL: return "a required pointer is NULL";
    case FMSMO_ERR_SHAPE: return "bad shape or leading dimension";
    case FMSMO_ERR_ALIGN: return "pointer, K or leading dimension not 16-byte aligned";
    case FMSMO_ERR_UNSUPPORTED: return "unsupported enum value or size";
    case FMSMO_ERR_LAUNCH: return "kernel launch failed";
    case FMSMO_ERR_SCRATCH: return "shape needs more scratch than the library's static buffer holds";
    default: return "unknown status";
  }
}


extern "C" int fmsmo_gemm_i8_i32_ws(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                                    int32_t* c, int64_t ldc, int64_t M, int64_t N, int64_t K,
                                    void* workspace, int64_t workspace_bytes, fmsmo_stream_t stream) {
  int rc = check_gemm(a, lda, b, ldb, c, ldc, M, N, K);
  if (rc) return rc;
  if (M == 0) return FMSMO_OK;
  // a few tokens: the weight-streaming decode kernels, storing their int32 sums
  if (use_decode(M, N, K, false))
    return fmsmo_gemv_dispatch(FMSMO_OP_I8, a, lda, b, ldb, nullptr, 1, nullptr, 1, nullptr, FMSMO_F32,
                               EPI_RAW_I32, c, FMSMO_F32, ldc, M, N, K, (hipStream_t)stream);
  GemmArgs g{};
  g.a = (const uint8_t*)a; g.b = (const uint8_t*)b; g.lda = lda; g.ldb = ldb;
  g.M = (int)M; g.N = (int)N; g.K = (int)K;
  // few output tiles and a long reduction: K slices into the workspace, added in a fixed order
  const SplitPlan plan = plan_split_k(M, N, K, workspace ? workspace_bytes : 0);
  if (plan.splits > 1 && workspace && workspace_bytes >= plan.ws_bytes && aligned16(workspace) &&
      plan.splits * M * lda < (1ll << 31))
    return launch_split_k_i32(plan, g, workspace, c, ldc, (hipStream_t)stream);
  EpiStoreI32 epi{c, ldc};
  launch_any<MMA_I8>(g, epi, (hipStream_t)stream);
  return fmsmo_check_launch();
}

extern "C" int fmsmo_gemm_i8_i32(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                                 int32_t* c, int64_t ldc, int64_t M, int64_t N, int64_t K,
                                 fmsmo_stream_t stream) {
  return fmsmo_gemm_i8_i32_ws(a, lda, b, ldb, c, ldc, M, N, K, nullptr, 0, stream);
}

static int gemm_i8_dq_impl(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                           const float* a_scale, int64_t a_scale_n, const float* w_scale,
                           int64_t w_scale_n, const void* bias, int bias_dtype, int epilogue,
                           void* y, int y_dtype, int64_t ldy, int64_t M, int64_t N, int64_t K,
                           void* workspace, int64_t workspace_bytes, fmsmo_stream_t stream) {
  int rc = check_gemm(a, lda, b, ldb, y, ldy, M, N, K);
  if (rc) return rc;
  rc = check_dq(a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype, y_dtype, M, N);
  if (rc) return rc;
  if (epilogue < FMSMO_EPI_REF_F16 || epilogue > FMSMO_EPI_F32_MULADD) return FMSMO_ERR_UNSUPPORTED;
  if (M == 0) return FMSMO_OK;
  if (use_decode(M, N, K, false))
    return fmsmo_gemv_dispatch(FMSMO_OP_I8, a, lda, b, ldb, a_scale, a_scale_n, w_scale, w_scale_n,
                               bias, bias_dtype, epilogue, y, y_dtype, ldy, M, N, K,
                               (hipStream_t)stream);
  GemmArgs g{};
  g.a = (const uint8_t*)a; g.b = (const uint8_t*)b; g.lda = lda; g.ldb = ldb;
  g.M = (int)M; g.N = (int)N; g.K = (int)K;
  const int as = a_scale_n == 1 ? 0 : 1, ws = w_scale_n == 1 ? 0 : 1;
  const SplitPlan plan = plan_split_k(M, N, K, workspace ? workspace_bytes : 0);
  if (plan.splits > 1 && workspace && workspace_bytes >= plan.ws_bytes && aligned16(workspace) &&
      plan.splits * M * lda < (1ll << 31)) {
    if (epilogue == FMSMO_EPI_REF_F16)
      return launch_split_k<MMA_I8, true, int>(plan, g, workspace, a_scale, as, w_scale, ws, bias,
                                               bias_dtype, y, y_dtype, ldy, (hipStream_t)stream);
    return launch_split_k<MMA_I8, false, int>(plan, g, workspace, a_scale, as, w_scale, ws, bias,
                                              bias_dtype, y, y_dtype, ldy, (hipStream_t)stream,
                                              epilogue == FMSMO_EPI_F32_MULADD);
  }
  if (epilogue == FMSMO_EPI_REF_F16)
    return launch_dq<MMA_I8, true, int>(g, a_scale, as, w_scale, ws, bias, bias_dtype, y,
                                               y_dtype, ldy, (hipStream_t)stream);
  return launch_dq<MMA_I8, false, int>(g, a_scale, as, w_scale, ws, bias, bias_dtype, y,
                                              y_dtype, ldy, (hipStream_t)stream, true,
                                              epilogue == FMSMO_EPI_F32_MULADD);
}

extern "C" int fmsmo_gemm_i8_dq(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                                const float* a_scale, int64_t a_scale_n, const float* w_scale,
                                int64_t w_scale_n, const void* bias, int bias_dtype, int epilogue,
                                void* y, int y_dtype, int64_t ldy, int64_t M, int64_t N,
                                int64_t K, fmsmo_stream_t stream) {
  return gemm_i8_dq_impl(a, lda, b, ldb, a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype,
                         epilogue, y, y_dtype, ldy, M, N, K, nullptr, 0, stream);
}

extern "C" int fmsmo_gemm_i8_dq_ws(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                                   const float* a_scale, int64_t a_scale_n, const float* w_scale,
                                   int64_t w_scale_n, const void* bias, int bias_dtype,
                                   int epilogue, void* y, int y_dtype, int64_t ldy, int64_t M,
                                   int64_t N, int64_t K, void* workspace, int64_t workspace_bytes,
                                   fmsmo_stream_t stream) {
  return gemm_i8_dq_impl(a, lda, b, ldb, a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype,
                         epilogue, y, y_dtype, ldy, M, N, K, workspace, workspace_bytes, stream);
}

// ------------------------------------------------------------- entry point that allocates nothing
// Split-K partial sums in device memory that belongs to the library's code object instead of a
// caller's workspace.  `scratch` is a host-side stand-in for the array: its device address is
// looked up once per device (each GPU that loads the library holds its own copy) and only that
// address is handed to kernels.
static __device__ __align__(256) unsigned char scratch[FMSMO_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {nullptr};

int static_scratch(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess && (dev < 0 || dev >= kMaxDevices)) e = hipErrorInvalidDevice;
  if (e == hipSuccess) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
      void* p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));  // address on the CURRENT device
      if (e == hipSuccess && !p) e = hipErrorInvalidSymbol;
      if (e == hipSuccess) g_scratch_ptr[dev] = p;
    }
    if (e == hipSuccess) *out = g_scratch_ptr[dev];
  }
  if (e != hipSuccess) {
    snprintf(g_fmsmo_last_error, sizeof(g_fmsmo_last_error), "static scratch lookup: %s",
             hipGetErrorString(e));
    return FMSMO_ERR_LAUNCH;
  }
  return FMSMO_OK;
}
}  // namespace

extern "C" int fmsmo_gemm_i8_dq_noalloc(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                                        const float* a_scale, int64_t a_scale_n,
                                        const float* w_scale, int64_t w_scale_n, const void* bias,
                                        int bias_dtype, int epilogue, void* y, int y_dtype,
                                        int64_t ldy, int64_t M, int64_t N, int64_t K,
                                        fmsmo_stream_t stream) {
  // arguments first: a rejected call touches nothing, not even the scratch lookup
  int rc0 = check_gemm(a, lda, b, ldb, y, ldy, M, N, K);
  if (rc0) return rc0;
  rc0 = check_dq(a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype, y_dtype, M, N);
  if (rc0) return rc0;
  if (epilogue < FMSMO_EPI_REF_F16 || epilogue > FMSMO_EPI_F32_MULADD) return FMSMO_ERR_UNSUPPORTED;
  if (M == 0) return FMSMO_OK;
  // the weight-streaming decode kernels use no scratch
  const bool decode = use_decode(M, N, K, false);
  // (the plan that fits the scratch, if one does: else the preferred plan's size is reported)
  int64_t need = decode ? 0 : plan_split_k(M, N, K, (int64_t)FMSMO_STATIC_SCRATCH_BYTES).ws_bytes;
  if (need > (int64_t)FMSMO_STATIC_SCRATCH_BYTES) {
    snprintf(g_fmsmo_last_error, sizeof(g_fmsmo_last_error),
             "split-K partial sums of %lld x %lld x %lld need %lld bytes, the static scratch holds %lld",
             (long long)M, (long long)N, (long long)K, (long long)need,
             (long long)FMSMO_STATIC_SCRATCH_BYTES);
    return FMSMO_ERR_SCRATCH;
  }
  void* ws = nullptr;
  if (need > 0) {
    int rc = static_scratch(&ws);
    if (rc) return rc;
  }
  // every slice's kernel stores its whole M x N block of partial sums before the reduction reads
  // it, so nothing in the scratch has to start at zero
  return gemm_i8_dq_impl(a, lda, b, ldb, a_scale, a_scale_n, w_scale, w_scale_n, bias, bias_dtype,
                         epilogue, y, y_dtype, ldy, M, N, K, ws, need, stream);
}

static bool any_takes(int64_t M, int64_t N, int64_t K, bool fp8) { return !fmsmo_gemv_batch_ok(M, K) && fmsmo_gemv_any_ok(M, N, K, fp8); }
extern "C" int64_t fmsmo_gemm_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  return any_takes(M, N, K, false) ? 0 : plan_split_k(M, N, K).ws_bytes;
}
extern "C" int64_t fmsmo_gemm_fp8_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  return any_takes(M, N, K, true) ? 0 : plan_split_k(M, N, K, 0, true).ws_bytes;
}

static int64_t gemm_tail_columns(bool fp8, int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) return 0;
  if (use_decode(M, N, K, fp8)) return 0;
  return tail_split_columns((int)M, (int)N, (int)K, fp8);
}
extern "C" int64_t fmsmo_gemm_tail_columns(int64_t M, int64_t N, int64_t K) { return gemm_tail_columns(false, M, N, K); }
extern "C" int64_t fmsmo_gemm_fp8_tail_columns(int64_t M, int64_t N, int64_t K) { return gemm_tail_columns(true, M, N, K); }

static void cut_tile_shape(bool fp8, int64_t M, int64_t N, int64_t K, int* tile_m, int* tile_n) {
  static const int bm[7] = {64, 128, 128, 128, 128, 256, 32}, bn[7] = {64, 64, 128, 192, 256, 256, 128};
  const CutTile t = cut_k_tile(M, N, K, !fp8 ? MMA_I8 : K % 64 ? MMA_FP8_F16 : MMA_FP8);
  *tile_m = bm[t];
  *tile_n = bn[t];
}
extern "C" int fmsmo_gemm_cut_tile(int fp8, int64_t M, int64_t N, int64_t K, int* tile_m, int* tile_n) {
  if (!tile_m || !tile_n) return FMSMO_ERR_NULL;
  if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff) return FMSMO_ERR_SHAPE;
  if (K % 16) return FMSMO_ERR_ALIGN;
  *tile_m = *tile_n = 0;
  if (K % 128 && !use_decode(M, N, K, fp8)) cut_tile_shape(fp8, M, N, K, tile_m, tile_n);
  return FMSMO_OK;
}

static int gemm_plan(bool fp8, int64_t M, int64_t N, int64_t K, int with_workspace, int* kernel, int* tile_m,
                     int* tile_n, int* splits) {
  if (!kernel || !tile_m || !tile_n || !splits) return FMSMO_ERR_NULL;
  if (M <= 0 || N <= 0 || K <= 0 || M > 0x7fffffff || N > 0x7fffffff || K > 0x7fffffff)
    return FMSMO_ERR_SHAPE;
  if (K % 16) return FMSMO_ERR_ALIGN;
  *tile_m = *tile_n = 0;
  *splits = 1;
  if (use_decode(M, N, K, fp8)) {
    *kernel = FMSMO_PLAN_DECODE;
    return FMSMO_OK;
  }
  // one pass of 32 x 128, 64 x 64 or 128 x 64 tiles, with or without a workspace
  if (K % 128 == 0 && use_low_tiles(M, N, K)) {
    *kernel = FMSMO_PLAN_TILE_LDS_DMA;
    *tile_m = TileLowK::BM;
    *tile_n = TileLowK::BN;
    return FMSMO_OK;
  }
  if (use_small_tiles(M, N, K) || use_tall_tiles(M, N, K)) {
    *kernel = FMSMO_PLAN_TILE_LDS_DMA;
    *tile_m = use_small_tiles(M, N, K) ? TileSmallK::BM : TileTallK::BM;
    *tile_n = TileTallK::BN;
    return FMSMO_OK;
  }
  const SplitPlan plan = with_workspace == 2 ? plan_split_k(M, N, K, (int64_t)FMSMO_STATIC_SCRATCH_BYTES, fp8)
                                             : plan_split_k(M, N, K, 0, fp8);
  if (with_workspace == 2 && plan.ws_bytes > (int64_t)FMSMO_STATIC_SCRATCH_BYTES)
    return FMSMO_ERR_SCRATCH;  // what the noalloc entry point returns for this shape
  if (with_workspace && plan.splits > 1) {
    *kernel = plan.rs ? FMSMO_PLAN_TILE_REGISTER_STAGED : FMSMO_PLAN_TILE_LDS_DMA;
    *tile_m = plan.rs ? 256 : plan.small ? TileSmallK::BM : TileMid::BM;
    *tile_n = plan.rs ? 128 : plan.tall || plan.small ? TileTallK::BN : TileMid::BN;
    *splits = plan.splits;
    return FMSMO_OK;
  }
  if (const FewRows few = a_few_rows(M, N, K)) {
    *kernel = FMSMO_PLAN_TILE_LDS_DMA;
    *tile_m = few == FEW_SMALL ? TileSmallK::BM : TileTallK::BM;
    *tile_n = TileTallK::BN;
    return FMSMO_OK;
  }
  if (K % 64) {
    *kernel = FMSMO_PLAN_GENERIC;  // (its tile: fmsmo_gemm_cut_tile)
    return FMSMO_OK;
  }
  if (K % 128) {
    *kernel = FMSMO_PLAN_TILE_LDS_DMA;
    cut_tile_shape(fp8, M, N, K, tile_m, tile_n);
    return FMSMO_OK;
  }
  const bool rs = use_register_staged(MMA_I8);
  const int bm[7] = {256, 128, 128, 256, 256, 128, 128}, bn[7] = {256, 256, 128, 192, 128, 192, 256};
  const int t = pick_tile((int)M, (int)N, (int)K, rs, fp8);
  *kernel = (rs && (t == 0 || t == 3 || t == 4)) ? FMSMO_PLAN_TILE_REGISTER_STAGED : FMSMO_PLAN_TILE_LDS_DMA;
  *tile_m = bm[t];
  *tile_n = (t == 3 && !rs) ? 256 : bn[t];
  return FMSMO_OK;
}

extern "C" int fmsmo_gemm_plan(int64_t M, int64_t N, int64_t K, int with_workspace, int* kernel, int* tile_m,
                               int* tile_n, int* splits) {
  return gemm_plan(false, M, N, K, with_workspace, kernel, tile_m, tile_n, splits);
}
extern "C" int fmsmo_gemm_fp8_plan(int64_t M, int64_t N, int64_t K, int with_workspace, int* kernel, int* tile_m,
                                   int* tile_n, int* splits) {
  if (with_workspace == 2) return FMSMO_ERR_UNSUPPORTED;  // there is no e4m3 call on the static scratch
  return gemm_plan(true, M, N, K, with_workspace, kernel, tile_m, tile_n, splits);
}

extern "C" int fmsmo_bmm_i8_dq(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                               int64_t stride_b, const float* a_scale, const float* b_scale,
                               const float* bias, void* y, int y_dtype, int64_t ldy, int64_t batch,
                               int64_t M, int64_t N, int64_t K, fmsmo_stream_t stream) {
  return launch_bmm<MMA_I8, int>(a, lda, b, ldb, stride_b, a_scale, b_scale, bias, y, y_dtype, ldy,
                                 batch, M, N, K, (hipStream_t)stream);
}


extern "C" int fmsmo_bmm_i8_zp(const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb, int64_t stride_b,
                               float scale, int zero, const int32_t* sums, int parts, void* y, int y_dtype,
                               int64_t ldy, int64_t batch, int64_t M, int64_t N, int64_t K, fmsmo_stream_t stream) {
  if (!sums) return FMSMO_ERR_NULL;
  if (parts < 1) return FMSMO_ERR_SHAPE;
  if (!zero_sums_fit(zero, K)) return FMSMO_ERR_UNSUPPORTED;
  return launch_bmm<MMA_I8, int>(a, lda, b, ldb, stride_b, nullptr, nullptr, nullptr, y, y_dtype, ldy, batch, M, N, K,
                                 (hipStream_t)stream, scale, sums, parts, zero);
}
