"""Tensor-level wrappers over the C-ABI kernels: argument checks, output allocation through
torch's caching allocator, the current HIP stream of the tensors' device.  No arithmetic happens
here; torch is only the owner of device memory and streams."""
from __future__ import annotations

import torch

from . import _lib as L

_DT = {torch.float16: L.F16, torch.bfloat16: L.BF16, torch.float32: L.F32}
_OPDT = {torch.int8: L.OP_I8, torch.float8_e4m3fn: L.OP_E4M3, torch.float16: L.OP_F16,
         torch.bfloat16: L.OP_BF16, torch.float32: L.OP_F32}
_BITS = {1: torch.uint8, 2: torch.int16, 4: torch.int32}


def _need_gpu(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            raise RuntimeError(
                "fms_mo_amd kernels run on an AMD GPU only (tensor is on %s); there is no CPU path"
                % t.device
            )


_RAW_STREAM = getattr(torch._C, "_cuda_getCurrentRawStream", None)
_CUR_DEVICE = getattr(torch._C, "_cuda_getDevice", None)


def _stream(t: torch.Tensor):
    """The current HIP stream of the tensor's device, as the integer handle the C ABI takes."""
    if _RAW_STREAM is not None:
        return _RAW_STREAM(t.get_device())
    return torch.cuda.current_stream(t.device).cuda_stream


class _NoSwitch:
    def __enter__(self):
        return self

    def __exit__(self, *exc):
        return False


_NO_SWITCH = _NoSwitch()


def _dev(t: torch.Tensor):
    """Context that makes the tensor's GPU current for a launch; nothing to do (and nothing paid:
    entering torch.cuda.device costs about a microsecond each way) when it already is."""
    idx = t.get_device()
    if _CUR_DEVICE is not None and _CUR_DEVICE() == idx:
        return _NO_SWITCH
    return torch.cuda.device(idx)


def _eager(*ts) -> bool:
    """True when the call can go straight to the implementation: plain tensors outside a compiler
    trace.  Otherwise the registered ``torch.ops.fms_mo_amd`` operator is called, whose shape-only
    twin serves tracing (going through the dispatcher costs about 3 us per call)."""
    if torch.compiler.is_compiling():
        return False
    for t in ts:
        if t is not None and type(t) is not torch.Tensor and type(t) is not torch.nn.Parameter:
            return False
    return True


def _ptr(t):
    return None if t is None else t.data_ptr()


def _dt(t: torch.Tensor) -> int:
    try:
        return _DT[t.dtype]
    except KeyError:
        raise TypeError(f"unsupported floating dtype {t.dtype}") from None


def _rows(t: torch.Tensor) -> torch.Tensor:
    """2-D, unit inner stride (row stride may be larger than the row)."""
    if t.dim() != 2:
        raise ValueError("expected a 2-D tensor")
    if t.stride(1) != 1 or (t.shape[0] > 1 and t.stride(0) < t.shape[1]):
        t = t.contiguous()
    return t


def _ld(t: torch.Tensor) -> int:
    return t.stride(0) if t.shape[0] > 1 else max(t.shape[1], t.stride(0))


def _scale_vec(s, n, device, name):
    if (type(s) is torch.Tensor and s.dtype is torch.float32 and s.dim() == 1 and s.is_cuda
            and s.is_contiguous() and not s.requires_grad and s.get_device() == device.index
            and s.numel() in (1, n)):
        return s  # the usual case: already the vector the kernels take
    if not torch.is_tensor(s):
        s = torch.tensor([float(s)], dtype=torch.float32, device=device)
    s = s.detach().to(device=device, dtype=torch.float32).reshape(-1).contiguous()
    if s.numel() not in (1, n):
        raise ValueError(f"{name} must have 1 or {n} elements, got {s.numel()}")
    return s


# ------------------------------------------------------------------------------- quantizers
def quant_act_i8_pertoken(x, smooth=None, compute_dtype=None, saturate=False):
    """(q int8 [M,K], scale fp32 [M]) -- see fmsmo_quant_act_i8_pertoken."""
    _need_gpu(x, smooth)
    x = _rows(x)
    M, K = x.shape
    if smooth is not None:
        smooth = smooth.detach().reshape(-1).contiguous()
        if smooth.numel() != K:
            raise ValueError("smooth scale must have K elements")
        if smooth.data_ptr() % 16:
            smooth = smooth.clone()
    if compute_dtype is None:
        compute_dtype = x.dtype if smooth is None else torch.promote_types(x.dtype, smooth.dtype)
    q = torch.empty((M, K), dtype=torch.int8, device=x.device)
    scale = torch.empty((M,), dtype=torch.float32, device=x.device)
    with _dev(x):
        L.call("fmsmo_quant_act_i8_pertoken", x.data_ptr(), _dt(x), _ld(x), _ptr(smooth),
               _dt(smooth) if smooth is not None else 0, _DT[compute_dtype], int(bool(saturate)),
               q.data_ptr(), K, scale.data_ptr(), M, K, _stream(x))
    return q, scale


def quant_act_i8_static(x, scale: float, zp: int, sym: int):
    _need_gpu(x)
    x = _rows(x)
    M, K = x.shape
    q = torch.empty((M, K), dtype=torch.int8, device=x.device)
    with _dev(x):
        L.call("fmsmo_quant_act_i8_static", x.data_ptr(), _dt(x), _ld(x), float(scale), int(zp),
               int(sym), q.data_ptr(), K, M, K, _stream(x))
    return q


def quant_act_i8_mulscale(x, mode, clip=None, smooth=None, meta_dtype=None):
    """(q int8 [M,K], a_scale fp32 [M] or [2]) -- see fmsmo_quant_act_i8_mulscale.  clip: device
    tensor {a_clip_val, a_clip_valn}; smooth: device tensor [K]; both of one dtype.  meta_dtype:
    dtype of the metadata vector when neither is passed (it still decides the compute dtype)."""
    _need_gpu(x, clip, smooth)
    x = _rows(x)
    M, K = x.shape
    meta = smooth if smooth is not None else clip
    if clip is not None and smooth is not None and clip.dtype != smooth.dtype:
        raise TypeError("clip and smooth must share one dtype")
    if mode != L.MS_PER_TOKEN:
        if clip is None or clip.numel() != 2:
            raise ValueError("clip must hold {a_clip_val, a_clip_valn}")
        clip = clip.detach().reshape(-1).contiguous()
    if smooth is not None:
        smooth = smooth.detach().reshape(-1).contiguous()
        if smooth.numel() != K:
            raise ValueError("smooth scale must have K elements")
        if smooth.data_ptr() % 16:
            smooth = smooth.clone()
    if meta is not None:
        meta_dtype = meta.dtype
    compute_dtype = x.dtype if meta_dtype is None else torch.promote_types(x.dtype, meta_dtype)
    q = torch.empty((M, K), dtype=torch.int8, device=x.device)
    a_scale = torch.empty((M if mode == L.MS_PER_TOKEN else 2,), dtype=torch.float32,
                          device=x.device)
    with _dev(x):
        L.call("fmsmo_quant_act_i8_mulscale", x.data_ptr(), _dt(x), _ld(x), _ptr(smooth),
               _ptr(clip), _DT[meta_dtype] if meta_dtype is not None else _dt(x), _DT[compute_dtype],
               int(mode), q.data_ptr(), K, a_scale.data_ptr(), M, K, _stream(x))
    return q, a_scale


def quant_act_fp8_pertoken(x, variant=L.FP8_LINEAR, static_scale=None):
    """(q e4m3 [M,K], scale fp32 [M] or the [1] static scale)."""
    _need_gpu(x)
    x = _rows(x)
    M, K = x.shape
    q = torch.empty((M, K), dtype=torch.float8_e4m3fn, device=x.device)
    if static_scale is not None:
        scale = _scale_vec(static_scale, 1, x.device, "static_scale")[:1].contiguous()
    else:
        scale = torch.empty((M,), dtype=torch.float32, device=x.device)
    with _dev(x):
        L.call("fmsmo_quant_act_fp8_pertoken", x.data_ptr(), _dt(x), _ld(x), int(variant),
               int(static_scale is not None), q.data_ptr(), K, scale.data_ptr(), M, K, _stream(x))
    return q, scale


def quant_act_fp8_dynamic(x, variant=L.FP8_LINEAR, per_tensor=False, scale_floor=1e-12,
                          scale_in_x_dtype=False):
    """(q e4m3 [M,K], scale fp32 [M] or [1]): the e4m3 quantizer with a dynamic scale
    max(amax / 448, scale_floor) per token or for the whole tensor, the division in fp32 or in
    x's dtype (see fmsmo_quant_act_fp8_dynamic / _tensor).  Per tensor it is two passes over x
    (abs-max, quantizer) with nothing read back to the host."""
    _need_gpu(x)
    if x.dim() != 2:
        raise ValueError("expected a 2-D tensor")
    x = _rows(x)
    M, K = x.shape
    q = torch.empty((M, K), dtype=torch.float8_e4m3fn, device=x.device)
    scale = torch.empty((1 if per_tensor else M,), dtype=torch.float32, device=x.device)
    # (fmsmo_quant_act_fp8_tensor counts 8-element chunks in 31 bits; larger tensors take column maxima)
    tensor_call = per_tensor and 0 < M * K < 1 << 34
    col_amax = absmax_cols(x) if per_tensor and not tensor_call else None
    with _dev(x):
        if tensor_call:
            parts = torch.empty((256,), dtype=torch.float32, device=x.device)
            L.call("fmsmo_quant_act_fp8_tensor", x.data_ptr(), _dt(x), _ld(x), int(variant), float(scale_floor),
                   _dt(x) if scale_in_x_dtype else L.F32, parts.data_ptr(), q.data_ptr(), K, scale.data_ptr(),
                   M, K, _stream(x))
        else:
            L.call("fmsmo_quant_act_fp8_dynamic", x.data_ptr(), _dt(x), _ld(x), int(variant),
                   int(bool(per_tensor)), _ptr(col_amax), float(scale_floor),
                   _dt(x) if scale_in_x_dtype else L.F32, q.data_ptr(), K, scale.data_ptr(), M, K, _stream(x))
    return q, scale


def quant_act_i8_static_t(x, mode, compute_dtype, scale, zp, sym=0, clip_lo=0.0, clip_hi=0.0):
    """int8 [M,K]: the static per-tensor formulas evaluated in ``compute_dtype`` (see
    fmsmo_quant_act_i8_static_t; mode is one of L.SQ_*).  All parameters are host numbers."""
    if not _COMPILING():
        q = (_H or _host()).quant_i8_static_t(x, mode, compute_dtype, scale, zp, sym, clip_lo, clip_hi)
        if q is not None:
            return q
    _need_gpu(x)
    x = _rows(x)
    M, K = x.shape
    q = torch.empty((M, K), dtype=torch.int8, device=x.device)
    with _dev(x):
        L.call("fmsmo_quant_act_i8_static_t", x.data_ptr(), _dt(x), _ld(x), int(mode),
               _DT[compute_dtype], float(scale), float(zp), int(sym), float(clip_lo), float(clip_hi),
               q.data_ptr(), K, M, K, _stream(x))
    return q


def quant_act_i8_dynamic(x, per_column, levels, zp=0, want_amax=False):
    """(q int8 [M,K], scale fp32 [1] or [K]): dynamic symmetric quantizer with one scale for the
    whole tensor or one per column, abs-max / levels in x's dtype, codes shifted by zp (see
    fmsmo_quant_act_i8_dynamic).  Two passes over x: the column abs-max, then the quantizer; nothing
    is read back to the host.  want_amax: also return the fp32 [K] column abs-max."""
    _need_gpu(x)
    x = _rows(x)
    M, K = x.shape
    col_amax = absmax_cols(x)
    q = torch.empty((M, K), dtype=torch.int8, device=x.device)
    scale = torch.empty((K if per_column else 1,), dtype=torch.float32, device=x.device)
    with _dev(x):
        L.call("fmsmo_quant_act_i8_dynamic", x.data_ptr(), _dt(x), _ld(x), col_amax.data_ptr(),
               L.DQ_PER_COLUMN if per_column else L.DQ_PER_TENSOR, int(levels), int(zp),
               q.data_ptr(), K, scale.data_ptr(), M, K, _stream(x))
    return (q, scale, col_amax) if want_amax else (q, scale)


def fake_quant_fp8(x, mode, want_values=True, want_codes=False):
    """FP8 (e4m3) emulation quantizer of QLinear on x [M,K] (see fmsmo_fake_quant_fp8; mode is one of
    L.F8E_*).  Returns (y, q, scale, inv_scale): y the fake-quantized tensor in x's dtype (None
    unless want_values), q the e4m3 codes (None unless want_codes), scale / inv_scale fp32 [1] or
    [M] (None for the saturating cast)."""
    _need_gpu(x)
    x = _rows(x)
    M, K = x.shape
    y = torch.empty((M, K), dtype=x.dtype, device=x.device) if want_values else None
    q = torch.empty((M, K), dtype=torch.float8_e4m3fn, device=x.device) if want_codes else None
    n = {L.F8E_SAT: 0, L.F8E_PER_TENSOR: 1, L.F8E_PER_ROW: M}[mode]
    scale = torch.empty((n,), dtype=torch.float32, device=x.device) if n else None
    inv = torch.empty((n,), dtype=torch.float32, device=x.device) if n else None
    col_amax = absmax_cols(x) if mode == L.F8E_PER_TENSOR else None
    with _dev(x):
        L.call("fmsmo_fake_quant_fp8", x.data_ptr(), _dt(x), _ld(x), int(mode), _ptr(col_amax),
               _ptr(y), K, _ptr(q), K, _ptr(scale), _ptr(inv), M, K, _stream(x))
    return y, q, scale, inv


# ------------------------------------------------------------------------------------ GEMMs
_WS_BYTES: dict = {}      # int8
_WS_BYTES_FP8: dict = {}  # e4m3


def _workspace(M, N, K, device, fp8=False):
    """Scratch for the split-K form of the *_dq GEMMs (None when the shape does not use one).  It
    comes from torch's caching allocator like every output, so it is also valid under graph
    capture; the library itself never allocates."""
    known, key = _WS_BYTES_FP8 if fp8 else _WS_BYTES, (M, N, K)
    nbytes = known.get(key)
    if nbytes is None:  # the policy is fixed for the life of the process: ask the library once per shape
        lib = L.load()
        nbytes = known[key] = (lib.fmsmo_gemm_fp8_workspace_bytes if fp8 else lib.fmsmo_gemm_workspace_bytes)(M, N, K)
    return torch.empty((nbytes,), dtype=torch.uint8, device=device) if nbytes > 0 else None


def gemm_plan(M, N, K, with_workspace=False, fp8=False):
    """(kernel, tile_m, tile_n, splits) the *_dq GEMMs of int8 (e4m3) operands use for a shape; no GPU
    needed (kernel is one of L.PLAN_*; see fmsmo_gemm_plan)."""
    import ctypes

    out = [ctypes.c_int(0) for _ in range(4)]
    L.call("fmsmo_gemm_fp8_plan" if fp8 else "fmsmo_gemm_plan", M, N, K, int(bool(with_workspace)),
           *[ctypes.byref(o) for o in out])
    return tuple(o.value for o in out)


def gemm_cut_tile(M, N, K, fp8=False):
    """(tile_m, tile_n) of one pass over K that is no multiple of 128 (see fmsmo_gemm_cut_tile)."""
    import ctypes

    out = [ctypes.c_int(0) for _ in range(2)]
    L.call("fmsmo_gemm_cut_tile", int(fp8), M, N, K, *[ctypes.byref(o) for o in out])
    return tuple(o.value for o in out)


def grouped_gemm_plan(experts, rows, N, K):
    """(kernel, tile_m, tile_n, bytes of K per stage) grouped_gemm_i8_dq uses for a shape; no GPU needed."""
    import ctypes

    out = [ctypes.c_int(0) for _ in range(4)]
    L.call("fmsmo_grouped_gemm_plan", experts, rows, N, K, *[ctypes.byref(o) for o in out])
    return tuple(o.value for o in out)


def clock_probe(buf):
    """Diagnostic: have block 0 of the following 256-row-tile GEMM launches store its clock
    readings into `buf` (int64 [6] on the GPU), or switch the probe off with None.  See
    fmsmo_debug_clock_probe; `core_clock_mhz` turns a filled buffer into a frequency."""
    if buf is None:
        L.call("fmsmo_debug_clock_probe", None)
        return
    _need_gpu(buf)
    if buf.dtype != torch.int64 or buf.numel() < 6 or not buf.is_contiguous():
        raise ValueError("the probe buffer must be a contiguous int64 tensor of 6 elements")
    L.call("fmsmo_debug_clock_probe", buf.data_ptr())


def stream_read(t, sink):
    """Diagnostic: one launch that only reads the bytes of the contiguous tensor `t` from device
    memory (fmsmo_debug_stream_read); `sink` is an int32 tensor of one element on the same GPU.
    Timed like a decode linear over the same weights it gives the floor the launch and the
    memory system set for that linear."""
    _need_gpu(t)
    _need_gpu(sink)
    if not t.is_contiguous() or sink.dtype != torch.int32 or sink.numel() < 1:
        raise ValueError("stream_read wants a contiguous tensor and an int32 sink")
    L.call("fmsmo_debug_stream_read", t.data_ptr(), t.numel() * t.element_size(), sink.data_ptr(), _stream(t))


def mfma_loop(data, iters, clk=None):
    """Diagnostic: the GEMM kernels' matrix instructions alone, fed from registers loaded once from
    `data` (int8 or float8_e4m3fn, contiguous; see fmsmo_debug_mfma_loop).  Returns the operations
    of one launch; `clk` (int64 [2] on the GPU) receives block 0's {core cycles, 100 MHz ticks}."""
    _need_gpu(data, clk)
    if data.dtype not in (torch.int8, torch.float8_e4m3fn) or not data.is_contiguous() or data.numel() % 4:
        raise ValueError("data must be a contiguous int8 / float8_e4m3fn tensor of a multiple of 4 elements")
    sink = torch.zeros(1, dtype=torch.float32, device=data.device)
    with _dev(data):
        L.call("fmsmo_debug_mfma_loop", _OPDT[data.dtype], data.data_ptr(), data.numel(), int(iters), _ptr(clk),
               sink.data_ptr(), _stream(data))
    return 1024.0 * iters * 2 * 16 * 2 * 32 * 32 * 64


def core_clock_mhz(buf):
    """Average core clock (MHz) over the life of the probed block: core cycles per tick of the
    constant 100 MHz counter, start of the block to the end of its epilogue."""
    c = buf.cpu().tolist()
    return (c[4] - c[0]) / ((c[5] - c[1]) / 100.0)


def _check_ab(a, w, dtype):
    _need_gpu(a, w)
    if a.dtype != dtype or w.dtype != dtype:
        raise TypeError(f"operands must be {dtype}, got {a.dtype} and {w.dtype}")
    a, w = _rows(a), _rows(w)
    if a.shape[1] != w.shape[1]:
        raise ValueError(f"K mismatch: a is {tuple(a.shape)}, w is {tuple(w.shape)} ([N,K] layout)")
    return a, w


def gemm_i8_i32(a, w):
    """int32 [M,N] = a int8 [M,K] . w int8 [N,K]^T."""
    a, w = _check_ab(a, w, torch.int8)
    M, K = a.shape
    N = w.shape[0]
    c = torch.empty((M, N), dtype=torch.int32, device=a.device)
    ws = _workspace(M, N, K, a.device)
    with _dev(a):
        if ws is not None:
            L.call("fmsmo_gemm_i8_i32_ws", a.data_ptr(), _ld(a), w.data_ptr(), _ld(w), c.data_ptr(), N,
                   M, N, K, ws.data_ptr(), ws.numel(), _stream(a))
        else:
            L.call("fmsmo_gemm_i8_i32", a.data_ptr(), _ld(a), w.data_ptr(), _ld(w), c.data_ptr(), N,
                   M, N, K, _stream(a))
    return c


def gemm_i8_dq(a, w, a_scale, w_scale, bias=None, out_dtype=torch.float16, epilogue=L.EPI_REF_F16,
               force_gemv=False):
    a, w = _check_ab(a, w, torch.int8)
    M, K = a.shape
    N = w.shape[0]
    a_scale = _scale_vec(a_scale, M, a.device, "a_scale")
    w_scale = _scale_vec(w_scale, N, a.device, "w_scale")
    if bias is not None:
        _need_gpu(bias)
        bias = bias.detach().reshape(-1).contiguous()
        if bias.numel() != N:
            raise ValueError("bias must have N elements")
    y = torch.empty((M, N), dtype=out_dtype, device=a.device)
    args = (a.data_ptr(), _ld(a), w.data_ptr(), _ld(w), a_scale.data_ptr(),
            a_scale.numel(), w_scale.data_ptr(), w_scale.numel(), _ptr(bias),
            _dt(bias) if bias is not None else 0, int(epilogue),
            y.data_ptr(), _DT[out_dtype], N, M, N, K)
    ws = None if force_gemv else _workspace(M, N, K, a.device)
    with _dev(a):
        if ws is not None:
            L.call("fmsmo_gemm_i8_dq_ws", *args, ws.data_ptr(), ws.numel(), _stream(a))
        else:
            L.call("fmsmo_gemv_i8_dq" if force_gemv else "fmsmo_gemm_i8_dq", *args, _stream(a))
    return y


def gemm_fp8_dq(a, w, a_scale, w_scale, bias=None, out_dtype=torch.bfloat16, force_gemv=False):
    a, w = _check_ab(a, w, torch.float8_e4m3fn)
    M, K = a.shape
    N = w.shape[0]
    a_scale = _scale_vec(a_scale, M, a.device, "a_scale")
    w_scale = _scale_vec(w_scale, N, a.device, "w_scale")
    if bias is not None:
        _need_gpu(bias)
        bias = bias.detach().reshape(-1).contiguous()
        if bias.numel() != N:
            raise ValueError("bias must have N elements")
    y = torch.empty((M, N), dtype=out_dtype, device=a.device)
    args = (a.data_ptr(), _ld(a), w.data_ptr(), _ld(w), a_scale.data_ptr(),
            a_scale.numel(), w_scale.data_ptr(), w_scale.numel(), _ptr(bias),
            _dt(bias) if bias is not None else 0, y.data_ptr(), _DT[out_dtype], N, M, N, K)
    ws = None if force_gemv else _workspace(M, N, K, a.device, True)
    with _dev(a):
        if ws is not None:
            L.call("fmsmo_gemm_fp8_dq_ws", *args, ws.data_ptr(), ws.numel(), _stream(a))
        else:
            L.call("fmsmo_gemv_fp8_dq" if force_gemv else "fmsmo_gemm_fp8_dq", *args, _stream(a))
    return y


def grouped_gemm_i8_dq(a, w, offsets, a_scale, w_scale, bias=None, out_dtype=torch.float16,
                       exact_ref=True):
    """a int8 [T,K] rows sorted by expert, w int8 [E,N,K], offsets int32 [E+1] (device),
    a_scale fp32 [T], w_scale fp32 [E,N], bias [E,N] or None -> [T,N]."""
    if not _COMPILING():
        y = (_H or _host()).grouped_i8(a, w, offsets, a_scale, w_scale, bias, out_dtype,
                                       L.EPI_REF_F16 if exact_ref else L.EPI_F32)
        if y is not None:
            return y
    _need_gpu(a, w, offsets)
    if a.dtype != torch.int8 or w.dtype != torch.int8 or w.dim() != 3:
        raise TypeError("a must be int8 [T,K], w int8 [E,N,K]")
    a = _rows(a)
    w = w.contiguous()
    T, K = a.shape
    E, N, K2 = w.shape
    if K2 != K or offsets.numel() != E + 1 or offsets.dtype != torch.int32:
        raise ValueError("shape mismatch (w [E,N,K], offsets int32 [E+1])")
    a_scale = _scale_vec(a_scale, T, a.device, "a_scale")
    w_scale = w_scale.detach().to(torch.float32).reshape(-1).contiguous()
    if a_scale.numel() != T or w_scale.numel() != E * N:
        raise ValueError("a_scale must be [T], w_scale [E,N]")
    if bias is not None:
        bias = bias.detach().reshape(-1).contiguous()
        if bias.numel() != E * N:
            raise ValueError("bias must be [E,N]")
    y = torch.empty((T, N), dtype=out_dtype, device=a.device)
    with _dev(a):
        L.call("fmsmo_grouped_gemm_i8_dq", a.data_ptr(), _ld(a), w.data_ptr(), K, N * K,
               offsets.contiguous().data_ptr(), E, T, a_scale.data_ptr(), w_scale.data_ptr(),
               _ptr(bias), _dt(bias) if bias is not None else 0,
               L.EPI_REF_F16 if exact_ref else L.EPI_F32, y.data_ptr(), _DT[out_dtype], N, N, K,
               _stream(a))
    return y


# ----------------------------------------------------------------------- chunked accumulation
def _chunk_workspace(a, N, chunk_size, tta):
    """(pointer, bytes, the tensor itself) of the scratch in which the slices of a cut int8 reduction are added."""
    M, K = a.shape
    nbytes = L.load().fmsmo_matmul_chunk_workspace_bytes(_OPDT[a.dtype], M, N, K, int(chunk_size), int(bool(tta)))
    if nbytes == 0:
        return None, 0, None
    ws = torch.empty((nbytes,), dtype=torch.uint8, device=a.device)
    return ws.data_ptr(), nbytes, ws


def matmul_chunk(a, w, c=None, chunk_size=64, chunk_trun_bits=0, max_acc_bits=32,
                 truncate_then_accumulate=True, clamp_acc_to_dl16=False):
    """a [M,K], w [N,K] (int8 | float8_e4m3fn | float16 | bfloat16 | float32) -> int32 / fp32 [M,N].  Floating-point
    accumulators add the rounded chunks one after the other, so a row's result does not depend on the rows beside it
    (an int32 accumulator adds them in any grouping: the entry points cut its reduction where there is a workspace)."""
    _need_gpu(a, w, c)
    if a.dtype != w.dtype or a.dtype not in _OPDT:
        raise TypeError(f"unsupported operand dtypes {a.dtype}, {w.dtype}")
    a, w = _rows(a), _rows(w)
    M, K = a.shape
    N = w.shape[0]
    if w.shape[1] != K:
        raise ValueError("K mismatch")
    esz = a.element_size()
    per16 = 16 // esz
    if K % per16 or _ld(a) % per16 or _ld(w) % per16:  # zero-pad K: contributes nothing to any chunk
        Kp = (K + 63) // 64 * 64
        a = torch.nn.functional.pad(a.view(_BITS[esz]), (0, Kp - K)).view(a.dtype)
        w = torch.nn.functional.pad(w.view(_BITS[esz]), (0, Kp - K)).view(w.dtype)
        K = Kp
    acc_dtype = torch.int32 if a.dtype == torch.int8 else torch.float32
    d = torch.empty((M, N), dtype=acc_dtype, device=a.device)
    if c is not None:
        if c.shape != (M, N):
            raise ValueError("C shape is inconsistent with A B.")
        c = c.to(acc_dtype).contiguous()
    with _dev(a):
        if a.dtype == torch.int8:
            wptr, wbytes, _ws = _chunk_workspace(a, N, chunk_size, truncate_then_accumulate and c is None)
            L.call("fmsmo_matmul_chunk_i8_ws", a.data_ptr(), _ld(a), w.data_ptr(), _ld(w), _ptr(c),
                   d.data_ptr(), N, M, N, K, int(chunk_size), int(chunk_trun_bits),
                   int(max_acc_bits), int(bool(truncate_then_accumulate)), wptr, wbytes, _stream(a))
        else:
            L.call("fmsmo_matmul_chunk_fp", a.data_ptr(), _ld(a), w.data_ptr(), _ld(w),
                   _OPDT[a.dtype], _ptr(c), d.data_ptr(), N, M, N, K, int(chunk_size),
                   int(chunk_trun_bits), int(bool(clamp_acc_to_dl16)),
                   int(bool(truncate_then_accumulate)), _stream(a))
    return d


def matmul_chunk_dq(a, w, a_scale, w_scale, bias=None, epilogue=L.EPI_SEQ_OUT, out_dtype=torch.float16,
                    chunk_size=64, chunk_trun_bits=0, max_acc_bits=32, truncate_then_accumulate=True,
                    clamp_acc_to_dl16=False):
    """y [M,N] = epilogue(chunked accumulator of a [M,K] . w [N,K]^T): the chunk-truncate matmul and
    its dequantization in one launch (see fmsmo_matmul_chunk_i8_dq / _fp_dq).  a_scale fp32 [M] or
    [1], w_scale fp32 [N] or [1], bias [N] (fp16 / bf16 / fp32) or None, epilogue one of L.EPI_*."""
    if not _COMPILING():
        y = (_H or _host()).chunk_dq(a, w, a_scale, w_scale, bias, epilogue, out_dtype, chunk_size, chunk_trun_bits, max_acc_bits,
                                     truncate_then_accumulate, clamp_acc_to_dl16)
        if y is not None:
            return y
    _need_gpu(a, w, a_scale, w_scale, bias)
    if a.dtype != w.dtype or a.dtype not in _OPDT:
        raise TypeError(f"unsupported operand dtypes {a.dtype}, {w.dtype}")
    a, w = _rows(a), _rows(w)
    M, K = a.shape
    N = w.shape[0]
    if w.shape[1] != K:
        raise ValueError("K mismatch")
    esz = a.element_size()
    per16 = 16 // esz
    if K % per16 or _ld(a) % per16 or _ld(w) % per16:  # zero-pad K: contributes nothing to any chunk
        Kp = (K + 63) // 64 * 64
        a = torch.nn.functional.pad(a.view(_BITS[esz]), (0, Kp - K)).view(a.dtype)
        w = torch.nn.functional.pad(w.view(_BITS[esz]), (0, Kp - K)).view(w.dtype)
        K = Kp
    a_scale = _scale_vec(a_scale, M, a.device, "a_scale")
    w_scale = _scale_vec(w_scale, N, a.device, "w_scale")
    if bias is not None:
        if bias.numel() != N or bias.dtype not in _DT:
            raise ValueError("bias must hold N fp16 / bf16 / fp32 values")
        bias = bias.reshape(-1).contiguous()
    y = torch.empty((M, N), dtype=out_dtype, device=a.device)
    common = (a_scale.data_ptr(), a_scale.numel(), w_scale.data_ptr(), w_scale.numel(), _ptr(bias),
              _DT[bias.dtype] if bias is not None else L.F32, int(epilogue), y.data_ptr(), _DT[out_dtype],
              N, M, N, K, int(chunk_size), int(chunk_trun_bits))
    with _dev(a):
        if a.dtype == torch.int8:
            wptr, wbytes, _ws = _chunk_workspace(a, N, chunk_size, truncate_then_accumulate)
            L.call("fmsmo_matmul_chunk_i8_dq_ws", a.data_ptr(), _ld(a), w.data_ptr(), _ld(w), *common,
                   int(max_acc_bits), int(bool(truncate_then_accumulate)), wptr, wbytes, _stream(a))
        else:
            L.call("fmsmo_matmul_chunk_fp_dq", a.data_ptr(), _ld(a), w.data_ptr(), _ld(w), _OPDT[a.dtype],
                   *common, int(bool(clamp_acc_to_dl16)), int(bool(truncate_then_accumulate)), _stream(a))
    return y


def quant_weight_i8(w, coef, smooth=None, mode="mul", want_row_sum=False):
    """Offline weight quantizer (see fmsmo_quant_weight_i8): w [N,K] fp16/bf16/fp32, coef [N] or [1]
    (``127 / clip_val`` for mode "mul", ``w_scale`` for mode "div"), smooth [K] or None.
    Returns int8 [N,K] (and the int32 row sums [N] when asked)."""
    _need_gpu(w, coef, smooth)
    if w.dim() != 2:
        raise ValueError("w must be [N, K]")
    if w.stride(1) != 1:
        w = w.contiguous()
    N, K = w.shape
    coef = coef.detach().reshape(-1).contiguous()
    if coef.numel() not in (1, N):
        raise ValueError("coef must have 1 or N elements")
    if smooth is not None:
        smooth = smooth.detach().reshape(-1).contiguous()
        if smooth.numel() != K:
            raise ValueError("smooth must have K elements")
        if smooth.data_ptr() % 16:
            smooth = smooth.clone()
    q = torch.empty((N, K), dtype=torch.int8, device=w.device)
    rs = torch.empty((N,), dtype=torch.int32, device=w.device) if want_row_sum else None
    with _dev(w):
        L.call("fmsmo_quant_weight_i8", w.data_ptr(), _dt(w), _ld(w), _ptr(smooth),
               _dt(smooth) if smooth is not None else 0, coef.data_ptr(), _dt(coef), coef.numel(),
               L.WQ_MUL if mode == "mul" else L.WQ_DIV, q.data_ptr(), K, _ptr(rs), N, K, _stream(w))
    return (q, rs) if want_row_sum else q


def absmax_cols(x, running=None):
    """Per-column abs-max of x [*, K] as fp32 [K]; with ``running`` (fp32 [K], >= 0) the result is
    the element-wise maximum of both, updated in place and returned."""
    _need_gpu(x, running)
    x = _rows(x.reshape(-1, x.shape[-1]))
    M, K = x.shape
    if running is None:
        running = torch.zeros((K,), dtype=torch.float32, device=x.device)
    elif running.dtype != torch.float32 or running.numel() != K or not running.is_contiguous():
        raise ValueError("running must be a contiguous fp32 tensor with K elements")
    with _dev(x):
        L.call("fmsmo_absmax_cols", x.data_ptr(), _dt(x), _ld(x), M, K, running.data_ptr(), _stream(x))
    return running


def deploy_vectors(clip, levels, bias, w_dtype, zp, clip_val=None, act=None, w_absmax=None, alpha=None):
    """The vectors and scalars of a deployed linear in one launch (see fmsmo_deploy_vectors): a dict with
    smooth [K] and zero_seen (None without act), w_scale, w_zp, corr, bias [N], input_scale, input_zp and the
    two clip values (None without clip_val)."""
    _need_gpu(clip, bias, act, w_absmax, alpha)
    dev, N = clip.device, clip.numel()
    f32 = dict(dtype=torch.float32, device=dev)
    i32 = dict(dtype=torch.int32, device=dev)
    o = {"w_scale": torch.empty((N,), **f32), "w_zp": torch.empty((N,), **i32), "corr": torch.empty((N,), **f32),
         "bias": torch.empty((N,), dtype=w_dtype, device=dev), "input_scale": torch.empty((), **f32),
         "input_zp": torch.empty((), **i32), "clips": None if clip_val is None else torch.empty((2,), **f32),
         "smooth": None, "zero_seen": None}
    K = 0
    if act is not None:
        K = act.numel()
        o["smooth"] = torch.empty((1, K), **f32)
        o["zero_seen"] = torch.empty(((K + 255) // 256,), **i32)
    with _dev(clip):
        L.call("fmsmo_deploy_vectors", _ptr(act), _ptr(w_absmax), _ptr(alpha), _ptr(o["smooth"]), _ptr(o["zero_seen"]), K,
               clip.data_ptr(), float(levels), _ptr(bias), _dt(bias) if bias is not None else 0,
               o["w_scale"].data_ptr(), o["w_zp"].data_ptr(), o["corr"].data_ptr(), o["bias"].data_ptr(), _DT[w_dtype], N,
               o["input_scale"].data_ptr(), o["input_zp"].data_ptr(), int(zp), _ptr(o["clips"]),
               0.0 if clip_val is None else float(clip_val), _stream(clip))
    return o


def zero_shift_bias(w, w_scale, a_meta, bias=None, offset=128.0):
    """fp32 [N] bias with the zero-point correction of asymmetric activations folded in
    (see fmsmo_zero_shift_bias).  w int8 [N,K]; w_scale fp32 [N] or [1]; a_meta fp32 [2]."""
    _need_gpu(w, w_scale, a_meta, bias)
    if w.dtype != torch.int8:
        raise TypeError("w must be int8")
    w = _rows(w)
    N, K = w.shape
    w_scale = _scale_vec(w_scale, N, w.device, "w_scale")
    if a_meta.dtype != torch.float32 or a_meta.numel() != 2:
        raise ValueError("a_meta must be fp32 {1/scale, zero point}")
    if bias is not None:
        bias = bias.detach().reshape(-1).contiguous()
        if bias.numel() != N:
            raise ValueError("bias must have N elements")
    out = torch.empty((N,), dtype=torch.float32, device=w.device)
    with _dev(w):
        L.call("fmsmo_zero_shift_bias", w.data_ptr(), _ld(w), w_scale.data_ptr(), w_scale.numel(),
               a_meta.contiguous().data_ptr(), float(offset), _ptr(bias),
               _dt(bias) if bias is not None else 0, out.data_ptr(), N, K, _stream(w))
    return out


# ---------------------------------------------------------------------------- batched matmul
def _batched3(t: torch.Tensor) -> torch.Tensor:
    """[..., R, C] -> [batch, R, C] with unit inner stride and one batch stride (a view when the
    leading dimensions collapse, a copy otherwise)."""
    t3 = t if t.dim() == 3 else t.reshape(-1, t.shape[-2], t.shape[-1])
    if t3.stride(2) != 1 or (t3.shape[1] > 1 and t3.stride(1) < t3.shape[2]):
        t3 = t3.contiguous()
    return t3


def quant_i8_affine(x, scale: float, offset: float, compute_dtype=None, transpose=False, pad_to=64, want_sums=False):
    """int8 codes of x [..., R, C] (see fmsmo_quant_i8_affine) as [batch, R, Cp] or, transposed,
    [batch, C, Rp]; the last dimension is zero-padded to a multiple of ``pad_to``.  want_sums: also
    the int32 sums of the codes along that dimension, [parts, batch, rows] to be added over the parts."""
    _need_gpu(x)
    x3 = _batched3(x)
    B, R, C = x3.shape
    compute_dtype = compute_dtype or x.dtype
    inner = R if transpose else C
    ldq = (inner + pad_to - 1) // pad_to * pad_to
    rows = C if transpose else R
    q = torch.empty((B, rows, ldq), dtype=torch.int8, device=x.device)
    sums = None
    if want_sums:
        parts = L.load().fmsmo_affine_sum_parts(B, R, C, int(bool(transpose)))
        sums = torch.empty((parts, B, rows), dtype=torch.int32, device=x.device)
    with _dev(x):
        L.call("fmsmo_quant_i8_affine_sums", x3.data_ptr(), _dt(x3), x3.stride(1) if R > 1 else C,
               x3.stride(0) if B > 1 else R * C, float(scale), float(offset), _DT[compute_dtype],
               int(bool(transpose)), q.data_ptr(), ldq, q.stride(0), _ptr(sums), B, R, C, _stream(x))
    return (q, sums) if want_sums else q


def _bmm(fn, dtype, a, b, a_scale, b_scale, bias, out_dtype):
    _need_gpu(a, b, bias)
    if a.dtype != dtype or b.dtype != dtype or a.dim() != 3 or b.dim() != 3:
        raise TypeError(f"operands must be 3-D {dtype} tensors: a [batch,M,K], b [batch,N,K]")
    a = a.contiguous()
    if b.stride(2) != 1 or b.stride(1) < b.shape[2]:
        b = b.contiguous()
    B, M, K = a.shape
    if b.shape[0] != B or b.shape[2] != K:
        raise ValueError(f"shape mismatch: a {tuple(a.shape)}, b {tuple(b.shape)} ([batch,N,K] layout)")
    N = b.shape[1]
    a_scale = _scale_vec(a_scale, 1, a.device, "a_scale")
    b_scale = _scale_vec(b_scale, 1, a.device, "b_scale")
    if bias is not None:
        bias = bias.detach().to(torch.float32).reshape(-1).contiguous()
        if bias.numel() != B * N:
            raise ValueError("bias must be [batch, N]")
    y = torch.empty((B, M, N), dtype=out_dtype, device=a.device)
    with _dev(a):
        L.call(fn, a.data_ptr(), K, b.data_ptr(), b.stride(1) if N > 1 else K,
               b.stride(0) if B > 1 else N * K, a_scale.data_ptr(), b_scale.data_ptr(), _ptr(bias),
               y.data_ptr(), _DT[out_dtype], N, B, M, N, K, _stream(a))
    return y


def bmm_i8_dq(a, b, a_scale, b_scale, bias=None, out_dtype=torch.float16):
    """y [batch,M,N] = (a [batch,M,K] . b [batch,N,K]^T) * a_scale * b_scale + bias [batch,N]."""
    return _bmm("fmsmo_bmm_i8_dq", torch.int8, a, b, a_scale, b_scale, bias, out_dtype)


def zero_sums_fit(zero, K):
    """Whether the int32 sums of bmm_i8_quantized hold (q1 - zero) . q2 whatever the codes are (K as the kernels
    see it, padded to at most 128)."""
    return (abs(int(zero)) + 128) * 128 * (-(-K // 128) * 128) < 1 << 31


def bmm_i8_quantized(m1, m2, scale1, zero1, scale2, zero2, compute_dtype):
    """y [batch, M, N] of m1's dtype = dequant(quant(m1) . quant(m2)): both operands quantized with their
    static parameters (see quant_i8_affine), the zero-point correction of m1 made from the column
    sums of m2's codes.  m1 [..., M, K], m2 [..., K, N] with equal leading dimensions.  Probabilities x
    values quantize m1 inside the product (fmsmo_bmm_qa_i8).  zero_sums_fit(zero1, K) must hold."""
    _need_gpu(m1, m2)
    M, K = m1.shape[-2:]
    if not zero_sums_fit(zero1, K):
        raise ValueError(f"the zero-point correction of K = {K} codes with zero point {zero1} may leave 32 bits")
    if not _COMPILING():
        y = (_H or _host()).bmm_quantized(m1, m2, scale1, zero1, scale2, zero2, compute_dtype)
        if y is not None:
            return y
    N = m2.shape[-1]
    a3 = _batched3(m1)
    B = a3.shape[0]
    qa = m1.dtype in (torch.float16, torch.bfloat16) and bool(L.load().fmsmo_bmm_qa_ok(
        _dt(m1), _DT[compute_dtype], scale1, zero1, B, M, N, K))
    # scores of a head dimension up to 128 run on the kernel for a reduction of exactly 128
    pad = 128 if K <= 128 and M > 128 and N > 128 else 64
    by_rows = m2.stride(-2) == 1 and m2.shape[-2] > 1  # a transposed view of a [n, k] tensor
    y = torch.empty((B, M, N), dtype=m1.dtype, device=m1.device)
    if qa:
        q2, sums = quant_i8_affine(m2.transpose(-1, -2) if by_rows else m2, scale2, zero2, compute_dtype, not by_rows, pad,
                                   want_sums=True)
        with _dev(m1):
            L.call("fmsmo_bmm_qa_i8", a3.data_ptr(), _dt(a3), a3.stride(1), a3.stride(0) if B > 1 else M * K,
                   float(scale1), float(zero1), _DT[compute_dtype], q2.data_ptr(), q2.stride(1), q2.stride(0),
                   float(scale2), sums.data_ptr(), sums.shape[0], y.data_ptr(), N, B, M, N, K, _stream(m1))
        return y
    if m1.dtype == m2.dtype and m2.numel() == B * K * N:
        # both operands' codes and the second one's sums in one launch
        b3 = _batched3(m2.transpose(-1, -2) if by_rows else m2)
        R, C = b3.shape[1:]
        Kp = (K + pad - 1) // pad * pad
        parts = L.load().fmsmo_affine_sum_parts(B, R, C, int(not by_rows))
        q1 = torch.empty((B, M, Kp), dtype=torch.int8, device=m1.device)
        q2 = torch.empty((B, N, Kp), dtype=torch.int8, device=m1.device)
        sums = torch.empty((parts, B, N), dtype=torch.int32, device=m1.device)
        with _dev(m1):
            L.call("fmsmo_quant_i8_affine_pair", _dt(a3), _DT[compute_dtype], B, a3.data_ptr(), a3.stride(1) if M > 1 else K,
                   a3.stride(0) if B > 1 else M * K, float(scale1), float(zero1), q1.data_ptr(), M * Kp, M, b3.data_ptr(),
                   b3.stride(1) if R > 1 else C, b3.stride(0) if B > 1 else R * C, float(scale2), float(zero2),
                   int(not by_rows), q2.data_ptr(), N * Kp, sums.data_ptr(), N, K, Kp, _stream(m1))
    else:
        q2, sums = quant_i8_affine(m2.transpose(-1, -2) if by_rows else m2, scale2, zero2, compute_dtype, not by_rows, pad,
                                   want_sums=True)
        q1 = quant_i8_affine(a3, scale1, zero1, compute_dtype, False, pad)
    Kp, parts = q1.shape[2], sums.shape[0]
    with _dev(m1):
        if L.load().fmsmo_affine_parts_first(parts, M, N, Kp):   # (else the product adds the parts itself)
            L.call("fmsmo_affine_add_parts", sums.data_ptr(), parts, B * N, _stream(m1))
            parts = 1
        L.call("fmsmo_bmm_i8_zp", q1.data_ptr(), Kp, q2.data_ptr(), Kp, q2.stride(0),
               _f32_product(scale1, scale2), int(zero1), sums.data_ptr(), parts, y.data_ptr(),
               _DT[m1.dtype], N, B, M, N, Kp, _stream(m1))
    return y


def _f32_product(a, b):
    """a * b rounded to fp32 (the factors are fp32 values)."""
    import struct

    return struct.unpack("f", struct.pack("f", a * b))[0]


def bmm_fp8_dq(a, b, a_scale, b_scale, bias=None, out_dtype=torch.bfloat16):
    return _bmm("fmsmo_bmm_fp8_dq", torch.float8_e4m3fn, a, b, a_scale, b_scale, bias, out_dtype)


# ------------------------------------------------------- the hot-path wrappers as torch operators
# The five wrappers every module forward ends in are registered under ``torch.ops.fms_mo_amd`` with
# shape-only twins, so that ``torch.compile`` traces a swapped model without graph breaks (the
# reference gets the same from registering its integer matmuls as ``torch.ops.fms_mo.*``,
# fms_mo/custom_ext_kernels/utils.py:642-802).  Only GPU kernels are registered: a CPU tensor that
# gets this far fails in the dispatcher.
_OPS = torch.library.Library("fms_mo_amd", "FRAGMENT")
_quant_act_i8_pertoken_impl = quant_act_i8_pertoken
_quant_act_i8_static_impl = quant_act_i8_static
_quant_act_fp8_pertoken_impl = quant_act_fp8_pertoken
_quant_act_fp8_dynamic_impl = quant_act_fp8_dynamic
_gemm_i8_dq_impl = gemm_i8_dq
_gemm_fp8_dq_impl = gemm_fp8_dq


def _register(name, schema, impl, fake):
    _OPS.define(name + schema)
    _OPS.impl(name, impl, "CUDA")
    torch.library.register_fake("fms_mo_amd::" + name)(fake)


def _rows_shape(x):
    return (x.shape[0], x.shape[1])


_register(
    "quant_act_i8_pertoken",
    "(Tensor x, Tensor? smooth, ScalarType? compute_dtype, bool saturate) -> (Tensor, Tensor)",
    lambda x, smooth, compute_dtype, saturate: _quant_act_i8_pertoken_impl(x, smooth, compute_dtype, saturate),
    lambda x, smooth, compute_dtype, saturate: (
        torch.empty(_rows_shape(x), dtype=torch.int8, device=x.device),
        torch.empty((x.shape[0],), dtype=torch.float32, device=x.device)),
)
_register(
    "quant_act_i8_static",
    "(Tensor x, float scale, int zp, int sym) -> Tensor",
    lambda x, scale, zp, sym: _quant_act_i8_static_impl(x, scale, zp, sym),
    lambda x, scale, zp, sym: torch.empty(_rows_shape(x), dtype=torch.int8, device=x.device),
)
_register(
    "quant_act_fp8_pertoken",
    "(Tensor x, int variant, Tensor? static_scale) -> (Tensor, Tensor)",
    lambda x, variant, static_scale: _quant_act_fp8_pertoken_impl(x, variant, static_scale),
    lambda x, variant, static_scale: (
        torch.empty(_rows_shape(x), dtype=torch.float8_e4m3fn, device=x.device),
        torch.empty((1 if static_scale is not None else x.shape[0],), dtype=torch.float32,
                    device=x.device)),
)
_register(
    "quant_act_fp8_dynamic",
    "(Tensor x, int variant, bool per_tensor, float scale_floor, bool scale_in_x_dtype) -> (Tensor, Tensor)",
    lambda x, variant, per_tensor, scale_floor, scale_in_x_dtype: _quant_act_fp8_dynamic_impl(
        x, variant, per_tensor, scale_floor, scale_in_x_dtype),
    lambda x, variant, per_tensor, scale_floor, scale_in_x_dtype: (
        torch.empty(_rows_shape(x), dtype=torch.float8_e4m3fn, device=x.device),
        torch.empty((1 if per_tensor else x.shape[0],), dtype=torch.float32, device=x.device)),
)
_register(
    "gemm_i8_dq",
    "(Tensor a, Tensor w, Tensor a_scale, Tensor w_scale, Tensor? bias, ScalarType out_dtype, "
    "int epilogue, bool force_gemv) -> Tensor",
    lambda a, w, a_scale, w_scale, bias, out_dtype, epilogue, force_gemv: _gemm_i8_dq_impl(
        a, w, a_scale, w_scale, bias, out_dtype, epilogue, force_gemv),
    lambda a, w, a_scale, w_scale, bias, out_dtype, epilogue, force_gemv: torch.empty(
        (a.shape[0], w.shape[0]), dtype=out_dtype, device=a.device),
)
_register(
    "gemm_fp8_dq",
    "(Tensor a, Tensor w, Tensor a_scale, Tensor w_scale, Tensor? bias, ScalarType out_dtype, "
    "bool force_gemv) -> Tensor",
    lambda a, w, a_scale, w_scale, bias, out_dtype, force_gemv: _gemm_fp8_dq_impl(
        a, w, a_scale, w_scale, bias, out_dtype, force_gemv),
    lambda a, w, a_scale, w_scale, bias, out_dtype, force_gemv: torch.empty(
        (a.shape[0], w.shape[0]), dtype=out_dtype, device=a.device),
)


def _as_scale(s, device):
    if torch.is_tensor(s):
        return s
    return torch.tensor([float(s)], dtype=torch.float32, device=device)


# An eager call of a 5 us kernel is bound by what the host does per launch: the common case -- plain,
# well-formed tensors on the current GPU, outside a compiler trace -- is checked, allocated and launched by
# the native module (csrc/host_calls.cpp), which returns None for anything else; that then goes through
# the general path (and gets its error messages there).
_COMPILING = torch.compiler.is_compiling
_H = None


def _host():
    global _H
    _H = L.host()
    return _H


def quant_act_i8_pertoken(x, smooth=None, compute_dtype=None, saturate=False):  # noqa: F811
    """(q int8 [M,K], scale fp32 [M]) -- see fmsmo_quant_act_i8_pertoken."""
    if not _COMPILING():
        r = (_H or _host()).quant_i8(x, smooth, compute_dtype, saturate)
        if r is not None:
            return r
    _need_gpu(x, smooth)
    if x.dim() != 2:
        raise ValueError("expected a 2-D tensor")
    if _eager(x, smooth):
        return _quant_act_i8_pertoken_impl(x, smooth, compute_dtype, bool(saturate))
    return torch.ops.fms_mo_amd.quant_act_i8_pertoken(x, smooth, compute_dtype, bool(saturate))


def quant_act_i8_static(x, scale: float, zp: int, sym: int):  # noqa: F811
    if not _COMPILING():
        q = (_H or _host()).quant_i8_static(x, scale, zp, sym)
        if q is not None:
            return q
    _need_gpu(x)
    if x.dim() != 2:
        raise ValueError("expected a 2-D tensor")
    if _eager(x):
        return _quant_act_i8_static_impl(x, float(scale), int(zp), int(sym))
    return torch.ops.fms_mo_amd.quant_act_i8_static(x, float(scale), int(zp), int(sym))


def quant_act_fp8_pertoken(x, variant=L.FP8_LINEAR, static_scale=None):  # noqa: F811
    """(q e4m3 [M,K], scale fp32 [M] or the [1] static scale)."""
    if static_scale is None and not _COMPILING():
        r = (_H or _host()).quant_fp8(x, variant, False, 1e-12, False)
        if r is not None:
            return r
    _need_gpu(x)
    if x.dim() != 2:
        raise ValueError("expected a 2-D tensor")
    if static_scale is not None:
        static_scale = _as_scale(static_scale, x.device)
    if _eager(x, static_scale):
        return _quant_act_fp8_pertoken_impl(x, int(variant), static_scale)
    return torch.ops.fms_mo_amd.quant_act_fp8_pertoken(x, int(variant), static_scale)


def quant_act_fp8_dynamic(x, variant=L.FP8_LINEAR, per_tensor=False, scale_floor=1e-12,  # noqa: F811
                          scale_in_x_dtype=False):
    """(q e4m3 [M,K], scale fp32 [M] or [1]), see fmsmo_quant_act_fp8_dynamic."""
    if not _COMPILING() and (per_tensor or scale_floor != 1e-12 or scale_in_x_dtype):
        r = (_H or _host()).quant_fp8(x, variant, per_tensor, scale_floor, scale_in_x_dtype)
        if r is not None:
            return r
    _need_gpu(x)
    if x.dim() != 2:
        raise ValueError("expected a 2-D tensor")
    if _eager(x):
        return _quant_act_fp8_dynamic_impl(x, int(variant), bool(per_tensor), float(scale_floor),
                                           bool(scale_in_x_dtype))
    return torch.ops.fms_mo_amd.quant_act_fp8_dynamic(x, int(variant), bool(per_tensor),
                                                      float(scale_floor), bool(scale_in_x_dtype))


def gemm_i8_dq(a, w, a_scale, w_scale, bias=None, out_dtype=torch.float16, exact_ref=True,  # noqa: F811
               force_gemv=False, epilogue=None):
    """y [M,N] = dequant(a int8 [M,K] . w int8 [N,K]^T), see fmsmo_gemm_i8_dq.  ``epilogue`` (one of
    L.EPI_*) overrides ``exact_ref`` (True = L.EPI_REF_F16, False = L.EPI_F32)."""
    if epilogue is None:
        epilogue = L.EPI_REF_F16 if exact_ref else L.EPI_F32
    if not force_gemv and not _COMPILING():
        y = (_H or _host()).gemm_dq(a, w, a_scale, w_scale, bias, out_dtype, int(epilogue))
        if y is not None:
            return y
    _need_gpu(a, w, bias)
    if _eager(a, w, bias) and (not torch.is_tensor(a_scale) or _eager(a_scale)) \
            and (not torch.is_tensor(w_scale) or _eager(w_scale)):
        return _gemm_i8_dq_impl(a, w, a_scale, w_scale, bias, out_dtype, int(epilogue), bool(force_gemv))
    return torch.ops.fms_mo_amd.gemm_i8_dq(a, w, _as_scale(a_scale, a.device), _as_scale(w_scale, a.device),
                                           bias, out_dtype, int(epilogue), bool(force_gemv))


def gemm_fp8_dq(a, w, a_scale, w_scale, bias=None, out_dtype=torch.bfloat16, force_gemv=False):  # noqa: F811
    if not force_gemv and not _COMPILING():
        y = (_H or _host()).gemm_dq(a, w, a_scale, w_scale, bias, out_dtype, 0)
        if y is not None:
            return y
    _need_gpu(a, w, bias)
    if _eager(a, w, bias) and (not torch.is_tensor(a_scale) or _eager(a_scale)) \
            and (not torch.is_tensor(w_scale) or _eager(w_scale)):
        return _gemm_fp8_dq_impl(a, w, a_scale, w_scale, bias, out_dtype, bool(force_gemv))
    return torch.ops.fms_mo_amd.gemm_fp8_dq(a, w, _as_scale(a_scale, a.device), _as_scale(w_scale, a.device),
                                            bias, out_dtype, bool(force_gemv))


# ------------------------------------------------------------------------ fused decode linear
_DECODE_OK = {}


def decode_linear_ok(x, smooth, K):
    """Can ``decode_linear_i8`` serve these activations?  fp16 / bf16, SmoothQuant divisors of the
    same dtype (or none): one token at K up to 8192 in one of the decode kernel's sizes or at
    14336 / 12800, up to four tokens at K = 4096, up to three at 14336 / 12800.  fp32 divisors
    (the quantizer then runs in fp32): K = 4096 up to two tokens, 14336 / 12800 one token."""
    if x.dim() != 2 or x.dtype not in (torch.float16, torch.bfloat16) or not x.is_cuda:
        return False
    f32s = smooth is not None and smooth.dtype == torch.float32
    if smooth is not None and ((smooth.dtype != x.dtype and not f32s) or smooth.numel() != K):
        return False
    key = (x.shape[0], K, f32s)
    if torch.compiler.is_compiling():
        # answers of earlier eager calls only (a foreign-function call cannot be traced); a shape
        # never seen eagerly takes the two-kernel path, which serves every shape
        return _DECODE_OK.get(key, False)
    if key not in _DECODE_OK:
        lib = L.load()
        ok = lib.fmsmo_decode_linear_f32s_ok if f32s else lib.fmsmo_decode_linear_ok
        _DECODE_OK[key] = bool(ok(x.shape[0], K))
    return _DECODE_OK[key]


def _decode_linear_i8_impl(x, w, w_scale, bias, smooth, out_dtype, exact_ref, saturate):
    x = _rows(x)
    w = _rows(w)
    M, K = x.shape
    N = w.shape[0]
    if w.dtype != torch.int8 or w.shape[1] != K:
        raise ValueError("w must be int8 [N, K]")
    w_scale = _scale_vec(w_scale, N, x.device, "w_scale")
    if smooth is not None:
        _need_gpu(smooth)
        smooth = smooth.detach().reshape(-1).contiguous()
        if smooth.numel() != K or smooth.dtype not in (x.dtype, torch.float32):
            raise ValueError("smooth must have K elements of x's dtype or fp32")
        if smooth.data_ptr() % 16:
            smooth = smooth.clone()
    if bias is not None:
        _need_gpu(bias)
        bias = bias.detach().reshape(-1).contiguous()
        if bias.numel() != N:
            raise ValueError("bias must have N elements")
    y = torch.empty((M, N), dtype=out_dtype, device=x.device)
    a_scale = torch.empty((M,), dtype=torch.float32, device=x.device)
    with _dev(x):
        L.call("fmsmo_decode_linear_i8", x.data_ptr(), _dt(x), _ld(x), _ptr(smooth),
               _dt(smooth) if smooth is not None else 0, int(bool(saturate)),
               w.data_ptr(), _ld(w), w_scale.data_ptr(), w_scale.numel(), _ptr(bias),
               _dt(bias) if bias is not None else 0, L.EPI_REF_F16 if exact_ref else L.EPI_F32,
               y.data_ptr(), _DT[out_dtype], N, a_scale.data_ptr(), M, N, K, _stream(x))
    return y, a_scale


_register(
    "decode_linear_i8",
    "(Tensor x, Tensor w, Tensor w_scale, Tensor? bias, Tensor? smooth, ScalarType out_dtype, "
    "bool exact_ref, bool saturate) -> (Tensor, Tensor)",
    lambda x, w, w_scale, bias, smooth, out_dtype, exact_ref, saturate: _decode_linear_i8_impl(
        x, w, w_scale, bias, smooth, out_dtype, exact_ref, saturate),
    lambda x, w, w_scale, bias, smooth, out_dtype, exact_ref, saturate: (
        torch.empty((x.shape[0], w.shape[0]), dtype=out_dtype, device=x.device),
        torch.empty((x.shape[0],), dtype=torch.float32, device=x.device)),
)


def decode_linear_i8(x, w, w_scale, bias=None, smooth=None, out_dtype=torch.float16, exact_ref=True,
                     saturate=False):
    """(y [M,N], per-token scales fp32 [M]) = quantize x per token (see quant_act_i8_pertoken) and
    multiply with the int8 weights w [N,K], in one launch; check ``decode_linear_ok`` first."""
    if not _COMPILING():
        r = (_H or _host()).decode_i8(x, w, w_scale, bias, smooth, out_dtype, L.EPI_REF_F16 if exact_ref else L.EPI_F32, saturate)
        if r is not None:
            return r
    _need_gpu(x, w, bias, smooth)
    if _eager(x, w, bias, smooth) and (not torch.is_tensor(w_scale) or _eager(w_scale)):
        return _decode_linear_i8_impl(x, w, w_scale, bias, smooth, out_dtype, bool(exact_ref), bool(saturate))
    return torch.ops.fms_mo_amd.decode_linear_i8(x, w, _as_scale(w_scale, x.device), bias, smooth,
                                                 out_dtype, bool(exact_ref), bool(saturate))


def _decode_linear_fp8_impl(x, w, w_scale, bias, out_dtype):
    x = _rows(x)
    w = _rows(w)
    M, K = x.shape
    N = w.shape[0]
    if w.dtype != torch.float8_e4m3fn or w.shape[1] != K:
        raise ValueError("w must be float8_e4m3fn [N, K]")
    w_scale = _scale_vec(w_scale, N, x.device, "w_scale")
    if bias is not None:
        _need_gpu(bias)
        bias = bias.detach().reshape(-1).contiguous()
        if bias.numel() != N:
            raise ValueError("bias must have N elements")
    y = torch.empty((M, N), dtype=out_dtype, device=x.device)
    a_scale = torch.empty((M,), dtype=torch.float32, device=x.device)
    with _dev(x):
        L.call("fmsmo_decode_linear_fp8", x.data_ptr(), _dt(x), _ld(x), w.data_ptr(), _ld(w),
               w_scale.data_ptr(), w_scale.numel(), _ptr(bias), _dt(bias) if bias is not None else 0,
               y.data_ptr(), _DT[out_dtype], N, a_scale.data_ptr(), M, N, K, _stream(x))
    return y, a_scale


_register(
    "decode_linear_fp8",
    "(Tensor x, Tensor w, Tensor w_scale, Tensor? bias, ScalarType out_dtype) -> (Tensor, Tensor)",
    lambda x, w, w_scale, bias, out_dtype: _decode_linear_fp8_impl(x, w, w_scale, bias, out_dtype),
    lambda x, w, w_scale, bias, out_dtype: (
        torch.empty((x.shape[0], w.shape[0]), dtype=out_dtype, device=x.device),
        torch.empty((x.shape[0],), dtype=torch.float32, device=x.device)),
)


def decode_linear_fp8(x, w, w_scale, bias=None, out_dtype=torch.bfloat16):
    """(y [M,N], token scales fp32 [M]): dynamic per-token e4m3 quantizer (the FP8Linear recipe) and
    the e4m3 weight-streaming matmul in one launch; check ``decode_linear_ok(x, None, K)`` first."""
    if not _COMPILING():
        r = (_H or _host()).decode_fp8(x, w, w_scale, bias, out_dtype)
        if r is not None:
            return r
    _need_gpu(x, w, bias)
    if _eager(x, w, bias) and (not torch.is_tensor(w_scale) or _eager(w_scale)):
        return _decode_linear_fp8_impl(x, w, w_scale, bias, out_dtype)
    return torch.ops.fms_mo_amd.decode_linear_fp8(x, w, _as_scale(w_scale, x.device), bias, out_dtype)
