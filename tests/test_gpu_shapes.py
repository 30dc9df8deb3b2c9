"""Kernel variants at the sizes where they can go wrong (tile edges, remainders, the ends of their
ranges), against the CPU oracle or an exact product."""
import pytest
import torch

from oracle import qlinear_oracle as O

pytestmark = pytest.mark.gpu


def gen(seed):
    return torch.Generator().manual_seed(seed)


def K():
    from fms_mo_amd import kernels

    return kernels


def make_qlinear(Kd, N, dtype, bias=True, seed=0, w_std=0.02):
    from fms_mo_amd.modules.linear import QLinear

    m = QLinear(Kd, N, bias=bias, num_bits_feature=8, qa_mode="pertokenmax", num_bits_weight=8, qw_mode="maxperCh",
                qcfg={"smoothq": False}, device="cpu")
    g = gen(seed)
    with torch.no_grad():
        m.weight.copy_(w_std * torch.randn(N, Kd, generator=g))
        if bias:
            m.bias.copy_(0.01 * torch.randn(N, generator=g))
    m.to(dtype)
    m.quantize_weight.float()
    with torch.no_grad():
        m.quantize_weight.train()
        m.quantize_weight(m.weight)
    return m.eval()


@pytest.mark.parametrize("M", [1, 5, 16, 100, 300])
@pytest.mark.parametrize("w_std", [0.02, 3e3])   # the second overflows the fp16 accumulator dtype
@pytest.mark.parametrize("kernel", ["cutlass", "triton"])
def test_deploy_module_of_a_bf16_model_rounds_to_fp16_first(dev, M, w_std, kernel):
    """acc_dtype is fp16: a bf16 model's output is the fp16 result cast to bf16 (an output beyond
    65504 becomes infinite), now inside the kernels' epilogues (decode, split K, tiles, chunks)."""
    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    Kd, N = 1024, 392
    m = make_qlinear(Kd, N, torch.bfloat16, w_std=w_std)
    x = torch.randn(M, Kd, generator=gen(M)).bfloat16()
    kw = {"truncate_lsb": 4, "chunk_size": 64} if kernel == "triton" else {}
    dep = QLinearINT8Deploy.from_fms_mo(m, use_int_kernel=kernel, use_dynamic_max_act_Qfunc=-1, recalc_clipvals=False,
                                        target_device=dev, **kw)
    y = dep(x.to(dev)).cpu()
    bufs = O.deploy_prepare(m.weight.detach(), m.bias.detach(), m.quantize_weight.clip_val)
    q_x, s_x, _ = O.quant_act_pertoken_i8(x)
    acc = O.chunk_matmul_i8(q_x, bufs["weight"], None, 64, 4, 32) if kw else O.int_gemm(q_x, bufs["weight"])
    ref = O.epilogue_ref(acc, s_x, bufs["w_scale"], bufs["bias"], torch.bfloat16)
    assert y.dtype == torch.bfloat16 and bool(torch.isinf(ref).any()) == (w_std > 1)
    assert torch.equal(y.view(torch.int16), ref.view(torch.int16))


@pytest.mark.parametrize("M,N,Kd", [
    (1, 5, 16), (3, 64, 48), (17, 65, 80), (128, 63, 112), (129, 130, 144),   # one and two stages, all but empty
    (16, 301, 1040), (300, 520, 624), (1500, 2400, 688), (257, 4099, 592),     # 128 x 64, 128 x 128, 256 x 256 tiles
    (2600, 2600, 336), (65, 640, 4160),
    (40, 100, 2064), (100, 700, 4016), (33, 250, 9344), (200, 130, 11216)])    # K slices, the last one shorter
def test_reductions_that_are_no_multiple_of_a_stage(dev, M, N, Kd):
    """K % 128 != 0 (the last stage is cut at K) and slices of unequal length: int8 exact, with and
    without a workspace; e4m3 exact on small integers.  What lies behind a row's K elements -- here
    large codes, for e4m3 NaN -- must not enter."""
    kn = K()
    g = torch.Generator(device=dev).manual_seed(M + N + Kd)
    a = torch.randint(-128, 128, (M, Kd + 16), generator=g, dtype=torch.int8, device=dev)[:, :Kd]
    w = torch.randint(-128, 128, (N, Kd + 32), generator=g, dtype=torch.int8, device=dev)[:, :Kd]
    acc = (a.double() @ w.double().t()).to(torch.int32)
    assert torch.equal(kn.gemm_i8_i32(a, w), acc)
    s_a = (torch.rand(M, 1, generator=gen(61)) * 0.05 + 1e-3).half()
    s_w = (torch.rand(N, generator=gen(62)) * 1e-3 + 1e-5).float()
    ref = O.epilogue_ref(acc.cpu(), s_a, s_w, None, torch.float16)
    y = kn.gemm_i8_dq(a, w, s_a.float().reshape(-1).to(dev), s_w.to(dev), None, out_dtype=torch.float16, exact_ref=True)
    assert torch.equal(y.cpu().view(torch.int16), ref.view(torch.int16))
    nan = torch.full((), float("nan"), device=dev)
    a8 = torch.cat((torch.randint(-4, 5, (M, Kd), generator=g, device=dev).float(), nan.expand(M, 16)), 1)
    w8 = torch.cat((torch.randint(-4, 5, (N, Kd), generator=g, device=dev).float(), nan.expand(N, 16)), 1)
    one = torch.ones(1, device=dev)
    y8 = kn.gemm_fp8_dq(a8.to(torch.float8_e4m3fn)[:, :Kd], w8.to(torch.float8_e4m3fn)[:, :Kd], one, one, None,
                        out_dtype=torch.float32)
    assert torch.equal(y8.double(), a8[:, :Kd].double() @ w8[:, :Kd].double().t())   # |sums| < 2^24: exact in fp32


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,Kd,pad", [(1, 16, 0), (3, 4096, 0), (16, 4096, 8), (17, 3856, 0), (700, 1032, 24), (4096, 512, 0)])
def test_fp8_per_tensor_quantizer_in_two_passes(dev, dtype, M, Kd, pad):
    """One scale for the tensor, with the abs-max taken inside the call (one launch up to 8192 groups of
    eight elements, partial maxima beyond; rows with a stride): bit for bit what the entry point that
    is handed the column maxima gives, for every recipe, for huge, tiny, infinite and NaN elements."""
    from fms_mo_amd import _lib as L

    kn, lib = K(), L.load()
    st = torch.cuda.current_stream().cuda_stream
    base = (torch.randn(M, Kd + pad, generator=gen(M + Kd)) * 3).to(dtype).to(dev)
    for special in (None, float("inf"), float("nan"), 0.0, 1e-20):
        x = base.clone()
        if special is not None:
            x = x * 0 if special in (0.0, 1e-20) else x
            x[M // 2, Kd // 2] = special
        x = x[:, :Kd]
        for variant, floor, in_x in ((L.FP8_LINEAR, 1e-12, False), (L.FP8_FPXACC, 1e-5, True), (L.FP8_FPXACC_DL8, 1e-5, True)):
            q, s = kn.quant_act_fp8_dynamic(x, variant, True, floor, in_x)
            amax, q2, s2 = kn.absmax_cols(x), torch.empty_like(q), torch.empty_like(s)
            dt = kn._dt(x)
            assert lib.fmsmo_quant_act_fp8_dynamic(x.data_ptr(), dt, kn._ld(x), variant, 1, amax.data_ptr(), floor,
                                                   dt if in_x else L.F32, q2.data_ptr(), Kd, s2.data_ptr(), M, Kd, st) == 0
            assert torch.equal(s.view(torch.int32), s2.view(torch.int32)), (special, variant)
            if special is not None and special != special and variant != L.FP8_LINEAR:
                continue  # a NaN abs-max: every torch code is NaN; both forms keep the floor as scale, only one clamps
            assert torch.equal(q.view(torch.uint8), q2.view(torch.uint8)), (special, variant)
