"""Timed workloads of the quantized-linear path, through the entry points a user's program calls.

Five kinds of work:

  linear     forwards of the deployed linears of one decoder layer (or of one linear): int8 with dynamic
             per-token or static activation scales, e4m3 with dynamic per-token or per-tensor scales
  moe        the two projections of a mixture-of-experts block over tokens sorted by expert
  attention  the two quantized matmuls of attention (scores = Q.K^T, context = P.V)
  chunked    linears with a reduced-precision accumulator (chunked truncation)
  convert    calibration statistics and conversion of a trained QLinear to its deployed form

Activations are Gaussian with one input channel in a hundred scaled by 50 where SmoothQuant is on (the
distribution SmoothQuant exists for), weights N(0, 0.02), biases N(0, 0.01).
"""
import os
import sys
import types

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "fms-model-optimizer_amd"))

from fms_mo_amd import kernels  # noqa: E402
from fms_mo_amd.modules.bmm import QBmmINT8Deploy  # noqa: E402
from fms_mo_amd.modules.fp8_linear import FP8Linear  # noqa: E402
from fms_mo_amd.modules.linear import LinearFPxAcc, QLinear, QLinearINT8Deploy  # noqa: E402
from fms_mo_amd.quant.ptq import activation_stats  # noqa: E402

DEVICE = "cuda"

# decoder-layer linears as "in x out" (fused q/k/v, attention output, gate + up, down)
LLAMA_8B = "4096x6144 4096x4096 4096x28672 14336x4096"
GRANITE_8B = "4096x6144 4096x4096 4096x25600 12800x4096"


def listed():
    return [
        # the smallest call of the path: one token through one linear, issued eagerly
        {"name": "int8_decode_1", "kind": "linear", "scheme": "int8", "dtype": "float16", "smooth": "model",
         "bias": True, "tokens": 1, "shapes": "4096x4096", "graph": False},
        # a serving loop's decode step for 16 sequences, the layer's linears captured in a HIP graph
        {"name": "int8_decode_16_graph", "kind": "linear", "scheme": "int8", "dtype": "bfloat16", "smooth": "model",
         "bias": False, "tokens": 16, "shapes": LLAMA_8B, "graph": True},
        # a batch between decode and prefill (continuous batching, short prompts); statistics left in fp32 as
        # calibration produces them
        {"name": "int8_batch_100", "kind": "linear", "scheme": "int8", "dtype": "float16", "smooth": "float32",
         "bias": True, "tokens": 100, "shapes": "5120x13824", "graph": False},
        # prefill of a long prompt through a decoder layer
        {"name": "int8_prefill_4096", "kind": "linear", "scheme": "int8", "dtype": "float16", "smooth": "model",
         "bias": True, "tokens": 4096, "shapes": LLAMA_8B, "graph": False},
        # what the lowering helpers build by default: calibrated (static, asymmetric) activation range; a bf16 model
        {"name": "int8_static_1000", "kind": "linear", "scheme": "int8_static", "dtype": "bfloat16", "smooth": "none",
         "bias": True, "tokens": 1000, "shapes": "4096x6144", "graph": False},
        # e4m3 decode of three sequences through a layer, eagerly
        {"name": "fp8_decode_3", "kind": "linear", "scheme": "fp8_token", "dtype": "bfloat16", "smooth": "none",
         "bias": False, "tokens": 3, "shapes": GRANITE_8B, "graph": False},
        # e4m3 prefill of a layer
        {"name": "fp8_prefill_2048", "kind": "linear", "scheme": "fp8_token", "dtype": "bfloat16", "smooth": "none",
         "bias": False, "tokens": 2048, "shapes": GRANITE_8B, "graph": False},
        # e4m3 with one dynamic scale per tensor, a ragged number of tokens
        {"name": "fp8_tensor_777", "kind": "linear", "scheme": "fp8_tensor", "dtype": "float16", "smooth": "none",
         "bias": True, "tokens": 777, "shapes": "12800x4096", "graph": False},
        # expert block of a mixture of experts: 4096 tokens routed to two of eight experts each
        {"name": "moe_int8_8192", "kind": "moe", "dtype": "float16", "experts": 8, "rows": 8192, "hidden": 4096,
         "inter": 14336},
        # both attention matmuls of one 2048-token sequence, 32 heads
        {"name": "attention_int8_2048", "kind": "attention", "dtype": "float16", "heads": 32, "queries": 2048,
         "context": 2048, "head_dim": 128},
        # accumulator study: one expert's share of tokens through the down projection, 7 low bits dropped per chunk
        {"name": "chunked_int8_1069", "kind": "chunked", "operands": "int8", "dtype": "float16", "tokens": 1069,
         "shape": "14336x4096", "chunk": 64, "drop_bits": 7},
        # offline: statistics of a calibration batch, SmoothQuant folding, weight quantization
        {"name": "convert_gate_up", "kind": "convert", "dtype": "float16", "tokens": 2048, "shape": "4096x28672"},
    ]


def _log(rng, lo, hi, step=1):
    """An integer spread over the logarithm of lo .. hi, a multiple of step."""
    v = lo * (hi / lo) ** rng.random()
    return min(hi, max(lo, step * round(v / step)))


def _shape(rng, most):
    """In and out features of a linear: mostly multiples of 128 as models have them, else multiples of 16
    (in) and any number (out: classifier and vocabulary heads)."""
    while True:
        if rng.random() < 0.7:
            k, n = _log(rng, 512, 16384, 128), _log(rng, 256, 28672, 128)
        else:
            k, n = _log(rng, 512, 16384, 16), _log(rng, 256, 28672)
        if k * n <= most:
            return k, n


def draw(rng):
    kind = rng.choices(["linear", "moe", "attention", "chunked", "convert"], [60, 10, 10, 10, 10])[0]
    dtype = rng.choice(["float16", "bfloat16"])
    if kind == "linear":
        scheme = rng.choices(["int8", "int8_static", "fp8_token", "fp8_tensor"], [45, 15, 25, 15])[0]
        k, n = _shape(rng, 4096 * 28672)
        tokens = _log(rng, 1, 4096)
        smooth = rng.choice(["model", "float32", "none"]) if scheme == "int8" else "none"
        return {"kind": kind, "scheme": scheme, "dtype": dtype, "smooth": smooth, "bias": rng.random() < 0.5,
                "tokens": tokens, "shapes": "%dx%d" % (k, n), "graph": tokens <= 64 and rng.random() < 0.5}
    if kind == "moe":
        experts = rng.choice([4, 8, 16])
        hidden, inter = _log(rng, 1024, 4096, 128), _log(rng, 1024, 14336, 128)
        return {"kind": kind, "dtype": dtype, "experts": experts, "rows": _log(rng, 128, 8192), "hidden": hidden,
                "inter": min(inter, 4096 * 14336 * 8 // (experts * hidden) // 128 * 128)}
    if kind == "attention":
        context = _log(rng, 64, 2048)
        return {"kind": kind, "dtype": dtype, "heads": rng.choice([8, 12, 16, 32]),
                "queries": 1 if rng.random() < 0.3 else context, "context": context,
                "head_dim": rng.choice([64, 80, 96, 128])}
    if kind == "chunked":
        k, n = _shape(rng, 4096 * 14336)
        operands = rng.choice(["int8", "int8", "model", "fp8"])
        return {"kind": kind, "operands": operands, "dtype": dtype, "tokens": _log(rng, 16, 1024),
                "shape": "%dx%d" % (k, n), "chunk": rng.choice([32, 64, 128]), "drop_bits": rng.choice([4, 7, 8])}
    k, n = _shape(rng, 4096 * 28672)
    return {"kind": kind, "dtype": dtype, "tokens": _log(rng, 128, 2048), "shape": "%dx%d" % (k, n)}


def _sizes(text):
    return [tuple(int(v) for v in s.split("x")) for s in text.split()]


# ---------------------------------------------------------------------------------------- inputs
def _activations(g, m, k, dtype, outliers):
    x = torch.randn(m, k, generator=g, device=DEVICE)
    if outliers:
        x[:, torch.randperm(k, generator=g, device=DEVICE)[: max(1, k // 100)]] *= 50
    return x.to(dtype)


def _qlinear(g, k, n, dtype, bias, qa_mode, smooth=False, act_range=None):
    """A QLinear as training and calibration leave it: 16-bit weights, fp32 quantizer buffers."""
    m = QLinear(k, n, bias=bias, num_bits_feature=8, qa_mode=qa_mode, num_bits_weight=8, qw_mode="maxperCh",
                qcfg={"smoothq": smooth, "smoothq_alpha": 0.5}, device=DEVICE).to(DEVICE)
    with torch.no_grad():
        m.weight.normal_(0, 0.02, generator=g)
        m.to(dtype)
        if bias:
            m.bias.normal_(0, 0.01, generator=g)
        m.quantize_weight.float()
        m.quantize_weight.clip_val.copy_(m.weight.abs().amax(dim=1))
        m.quantize_weight.clip_valn.copy_(-m.quantize_weight.clip_val)
        if act_range is not None:
            m.quantize_feature.float()
            m.quantize_feature.clip_valn.fill_(act_range[0])
            m.quantize_feature.clip_val.fill_(act_range[1])
        if smooth:
            m.smoothq_act_scale = torch.zeros(k, device=DEVICE)
            m.smoothq_alpha = torch.full((1,), 0.5, device=DEVICE)
    return m.eval()


def _deploy(g, k, n, x, case, dtype):
    """The deployed module of the case and the activations it is given."""
    scheme = case["scheme"]
    if scheme.startswith("fp8"):
        w = 0.02 * torch.randn(n, k, generator=g, device=DEVICE)
        b = (0.01 * torch.randn(n, generator=g, device=DEVICE)).to(dtype) if case["bias"] else None
        return FP8Linear.from_float(w, b, per_channel=True, act="token" if scheme == "fp8_token" else "tensor")
    if scheme == "int8_static":
        q = _qlinear(g, k, n, dtype, case["bias"], "maxmin", act_range=(-3.0, 4.0))
        return QLinearINT8Deploy.from_fms_mo(q).to(dtype)
    smooth = case["smooth"] != "none"
    q = _qlinear(g, k, n, dtype, case["bias"], "pertokenmax", smooth)
    if smooth:
        q.set_act_scale(x.abs().amax(dim=0).float().clamp(min=1e-3))
    m = QLinearINT8Deploy.from_fms_mo(q, use_dynamic_max_act_Qfunc=-1, recalc_clipvals=False)
    return m.to(dtype) if case["smooth"] == "model" else m


def prepare(case, seed):
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = getattr(torch, case["dtype"])
    s = {"kind": case["kind"]}
    if case["kind"] == "linear":
        pairs = []
        for k, n in _sizes(case["shapes"]):
            x = _activations(g, case["tokens"], k, dtype, case["smooth"] != "none")
            pairs.append((_deploy(g, k, n, x, case, dtype), x))
        s["pairs"] = pairs
        if case["graph"]:
            # the modules read their scales once eagerly, then the launches are captured for replay
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                for m, x in pairs:
                    m(x)
            torch.cuda.current_stream().wait_stream(side)
            s["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(s["graph"]):
                s["out"] = [m(x) for m, x in pairs]
    elif case["kind"] == "moe":
        e, rows, hidden, inter = case["experts"], case["rows"], case["hidden"], case["inter"]
        # the split of a router with uniform random logits
        counts = torch.bincount(torch.randint(0, e, (rows,), generator=g, device=DEVICE), minlength=e)
        s["offsets"] = torch.cat((counts.new_zeros(1), counts.cumsum(0))).to(torch.int32)
        s["stages"] = []
        for k, n in ((hidden, 2 * inter), (inter, hidden)):
            w = torch.empty(e, n, k, dtype=torch.int8, device=DEVICE)
            for i in range(e):
                w[i] = torch.randn(n, k, generator=g, device=DEVICE).mul_(30).round_().clamp_(-127, 127)
            ws = 1e-4 + 1e-3 * torch.rand(e, n, generator=g, device=DEVICE)
            s["stages"].append((_activations(g, rows, k, dtype, False), w, ws))
        s["dtype"] = dtype
    elif case["kind"] == "attention":
        h, m, c, d = case["heads"], case["queries"], case["context"], case["head_dim"]

        def trained(lo, hi, other):
            one = lambda v: torch.tensor([v], dtype=dtype, device=DEVICE)  # noqa: E731
            return types.SimpleNamespace(
                num_bits_m1=8, num_bits_m2=8, qm1_mode="max",
                quantize_m1=types.SimpleNamespace(clip_val=one(hi), clip_valn=one(lo), num_bits=8),
                quantize_m2=types.SimpleNamespace(clip_val=one(other), num_bits=8))

        s["scores"] = QBmmINT8Deploy.from_fms_mo(trained(-4.0, 4.0, 4.0), target_device=DEVICE)
        s["context"] = QBmmINT8Deploy.from_fms_mo(trained(0.0, 1.0, 4.0), target_device=DEVICE)
        s["q"] = torch.randn(1, h, m, d, generator=g, device=DEVICE).to(dtype)
        s["k"] = torch.randn(1, h, c, d, generator=g, device=DEVICE).to(dtype)
        s["v"] = torch.randn(1, h, c, d, generator=g, device=DEVICE).to(dtype)
        s["p"] = torch.softmax(3 * torch.randn(1, h, m, c, generator=g, device=DEVICE), dim=-1).to(dtype)
    elif case["kind"] == "chunked":
        (k, n), = _sizes(case["shape"])
        s["x"] = _activations(g, case["tokens"], k, dtype, False)
        if case["operands"] == "int8":
            s["module"] = QLinearINT8Deploy.from_fms_mo(
                _qlinear(g, k, n, dtype, True, "pertokenmax"), use_int_kernel="triton", use_dynamic_max_act_Qfunc=-1,
                recalc_clipvals=False, truncate_lsb=case["drop_bits"], chunk_size=case["chunk"]).to(dtype)
        else:
            lin = torch.nn.Linear(k, n, device=DEVICE, dtype=dtype)
            with torch.no_grad():
                lin.weight.normal_(0, 0.02, generator=g)
                lin.bias.normal_(0, 0.01, generator=g)
            s["module"] = LinearFPxAcc.from_nn(lin, trun_bits=case["drop_bits"], chunk_size=case["chunk"],
                                               dynamic_fp8="per_token" if case["operands"] == "fp8" else False)
    else:
        (k, n), = _sizes(case["shape"])
        s["x"] = _activations(g, case["tokens"], k, dtype, True)
        s["qlinear"] = _qlinear(g, k, n, dtype, True, "pertokenmax", smooth=True)
    return s


# ------------------------------------------------------------------------------------------ a pass
@torch.no_grad()
def run(s):
    kind = s["kind"]
    if kind == "linear":
        if "graph" in s:
            s["graph"].replay()
            return s["out"]
        return [m(x) for m, x in s["pairs"]]
    if kind == "moe":
        out = []
        for x, w, ws in s["stages"]:
            q, scale = kernels.quant_act_i8_pertoken(x)
            out.append(kernels.grouped_gemm_i8_dq(q, w, s["offsets"], scale, ws, out_dtype=s["dtype"]))
        return out
    if kind == "attention":
        return [s["scores"](s["q"], s["k"].transpose(-1, -2)), s["context"](s["p"], s["v"])]
    if kind == "chunked":
        return s["module"](s["x"])
    q = s["qlinear"]
    stats = activation_stats("linear", s["x"], {})["linear"]
    q.set_act_scale(stats)
    m = QLinearINT8Deploy.from_fms_mo(q, use_dynamic_max_act_Qfunc=-1)
    return [stats, m.weight, m.w_scale, m.smoothq_scale, m.bias]


# ------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    byts = flops = 0
    if case["kind"] == "linear":
        for k, n in _sizes(case["shapes"]):
            byts += 2 * case["tokens"] * (k + n) + k * n + 4 * n
            flops += 2 * case["tokens"] * k * n
    elif case["kind"] == "moe":
        rows, hidden, inter = case["rows"], case["hidden"], case["inter"]
        for k, n in ((hidden, 2 * inter), (inter, hidden)):
            byts += 2 * rows * (k + n) + min(case["experts"], rows) * n * (k + 4)
            flops += 2 * rows * k * n
    elif case["kind"] == "attention":
        h, m, c, d = case["heads"], case["queries"], case["context"], case["head_dim"]
        byts = 2 * h * 2 * (m * d + c * d + m * c)
        flops = 2 * 2 * h * m * c * d
    elif case["kind"] == "chunked":
        (k, n), = _sizes(case["shape"])
        byts = 2 * case["tokens"] * (k + n) + k * n * (1 if case["operands"] == "int8" else 2) + 4 * n
        flops = 2 * case["tokens"] * k * n
    else:
        (k, n), = _sizes(case["shape"])
        byts = 2 * case["tokens"] * k + 3 * k * n + 8 * k + 4 * n
    return {"bytes": byts, "flops": flops}


def tolerance(case):
    """Four times what the path's outputs differ by from the same codes and scales in 64 bits.  Integer sums
    are exact and e4m3 sums fp32, so that is the rounding of the output dtype, 2.1e-4 (fp16) or 1.7e-3 (bf16)
    in the 2-norm; the int8 modules also form the product of the two scales in fp16, mostly a subnormal one:
    1.4e-3 (fp16), 2.2e-3 (bf16)."""
    if case["kind"] == "convert":
        # conversion on the CPU against the GPU: scales 7e-8, one weight in a million on the other side of a tie
        return {"rel": 1e-6, "differ": 1e-5}
    half = case["dtype"] == "float16"
    if case["kind"] == "moe" or case.get("scheme", case.get("operands", "")).startswith("int8"):
        return {"rel": 5.6e-3 if half else 8.8e-3}
    return {"rel": 8.4e-4 if half else 6.8e-3}
