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


@pytest.mark.parametrize("how", ["assigned", "subclass"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_an_iaddmm_of_the_users_own_keeps_its_three_arguments(dev, how, dtype):
    """What it returns is cast to acc_dtype and then to the model's dtype."""
    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    class Own(QLinearINT8Deploy):
        def iaddmm_int(self, bias, m1, m2):
            return 2 * super().iaddmm_int(bias, m1, m2).float()

    cls = Own if how == "subclass" else QLinearINT8Deploy
    dep = cls.from_fms_mo(make_qlinear(256, 40, dtype), use_int_kernel="triton", use_dynamic_max_act_Qfunc=-1,
                          recalc_clipvals=False, target_device=dev, truncate_lsb=4, chunk_size=64)
    x = torch.randn(7, 256, generator=gen(7)).to(dtype).to(dev)
    plain = QLinearINT8Deploy.iaddmm_int
    if how == "assigned":
        dep.iaddmm = lambda bias, m1, m2: 2 * plain(dep, bias, m1, m2).float()
    y = dep(x)
    ref = (2 * plain(dep, dep.bias, x, dep.weight.t()).float()).half().to(dtype)
    assert y.dtype == dtype and torch.equal(y, ref)


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


@pytest.mark.parametrize("M,N,Kd", [(1, 5, 16), (17, 33, 48), (32, 64, 544), (65, 31, 1136), (96, 160, 11472)])
@pytest.mark.parametrize("odt", [torch.float32, torch.float16])
def test_e4m3_reductions_that_are_no_multiple_of_64_add_in_fp32(dev, M, N, Kd, odt):
    """2-norm error against 64 bits no larger than that of one fp32 addition after the other (products of e4m3
    elements are exact in fp32); the e4m3 matrix instruction, which keeps fewer bits, misses it by a hundred."""
    g = torch.Generator(device=dev).manual_seed(M + Kd)
    a = torch.randn(M, Kd, generator=g, device=dev).to(torch.float8_e4m3fn)
    w = torch.randn(N, Kd, generator=g, device=dev).to(torch.float8_e4m3fn)
    s_a, s_w = torch.rand(M, generator=g, device=dev) + 0.5, torch.rand(N, generator=g, device=dev) + 0.5
    bias = torch.randn(N, generator=g, device=dev)
    af, wf = a.float(), w.float()
    chain = torch.zeros(M, N, device=dev)
    for k in range(Kd):
        chain += af[:, k, None] * wf[:, k]
    exact = af.double() @ wf.double().t()
    one = torch.ones(1, device=dev)
    err = lambda y, ref: float((y.double() - ref).norm() / ref.norm())  # noqa: E731
    if odt == torch.float32:
        y = K().gemm_fp8_dq(a, w, one, one, None, out_dtype=odt)
        assert err(y, exact) <= max(err(chain, exact), 2.0 ** -25)
    ref = exact * (s_a[:, None] * s_w).double() + bias.double()
    y = K().gemm_fp8_dq(a, w, s_a, s_w, bias, out_dtype=odt)
    # (one rounding each of scale product, fma and output beyond the sum's)
    assert err(y, ref) <= 4 * err(chain, exact) + 2.0 ** (-22 if odt == torch.float32 else -11)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,Kd,pad", [(1, 16, 0), (3, 4096, 0), (16, 4096, 8), (17, 3856, 0), (700, 1032, 24), (4096, 512, 0), (3, 16384, 8),
                                      (5, 16392, 0), (900, 4096, 0)])
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
            # (a NaN abs-max: every torch code is NaN; both forms keep the floor as scale, and rows that are finite saturate)
            assert torch.equal(s.view(torch.int32), s2.view(torch.int32)), (special, variant)
            assert torch.equal(q.view(torch.uint8), q2.view(torch.uint8)), (special, variant)


def make_qbmm(dev, lo, hi, other, dtype):
    import types

    from fms_mo_amd.modules.bmm import QBmmINT8Deploy

    one = lambda v: torch.tensor([v], dtype=dtype)
    src = types.SimpleNamespace(num_bits_m1=8, num_bits_m2=8, qm1_mode="max",
                                quantize_m1=types.SimpleNamespace(clip_val=one(hi), clip_valn=one(lo), num_bits=8),
                                quantize_m2=types.SimpleNamespace(clip_val=one(other), num_bits=8))
    return QBmmINT8Deploy.from_fms_mo(src, target_device=dev)


@pytest.mark.parametrize("xdt,cdt", [(torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16),
                                     (torch.float16, torch.float32), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("transpose", [False, True])
def test_affine_codes_of_nan_are_the_lower_bound(dev, xdt, cdt, transpose):
    """Every NaN pattern, quiet and signalling, for scales of both signs (exact in 16 bits)."""
    x = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(xdt)
    x = x[torch.isnan(x)][:248].repeat(64).reshape(1, -1, 62).to(dev) if xdt == torch.bfloat16 else \
        x[torch.isnan(x)].reshape(1, -1, 62).to(dev)
    for scale in (0.03125, -0.03125, 64.0, -640.0):
        for zero in (0.0, -128.0, 100.0):
            q = K().quant_i8_affine(x, scale, zero, cdt, transpose)
            assert (q[..., :x.shape[1] if transpose else 62] == -128).all(), (scale, zero)


@pytest.mark.parametrize("xdt,sdt", [(torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16),
                                     (torch.float16, torch.float32), (torch.bfloat16, torch.float32),
                                     (torch.float32, torch.float32)])
@pytest.mark.parametrize("B,M,Kd,N,view", [
    (32, 64, 256, 64, False),     # the smallest product that quantizes m1 on the way
    (33, 130, 300, 80, False), (32, 129, 1001, 128, False), (40, 100, 383, 1, False),   # ragged rows, slabs, columns
    (2, 70, 513, 128, False), (3, 1, 77, 96, False),                                    # two launches
    (5, 200, 64, 300, True), (2, 131, 80, 129, True), (4, 1, 128, 500, True)])          # scores
def test_attention_products(dev, xdt, sdt, B, M, Kd, N, view):
    """QBmmINT8Deploy against the exact product of its own codes: integers (sums with the zero-point
    correction) times the fp32 scale product, one fp32 rounding each of sum and product, then the
    output's: at most the output's half ulp plus 2^-23.  Infinite and NaN elements of m1 quantize as in the
    stand-alone quantizer."""
    m = make_qbmm(dev, -0.7 if view else 0.0, 1.0, 3.0, sdt)
    m1 = torch.randn(B, M, Kd, generator=gen(B + M)).to(xdt)
    if not view:
        m1 = torch.softmax(m1.float() * 2, -1).to(xdt)
    m1[0, 0, 0], m1[-1, -1, -1], m1[B // 2, M // 2, Kd // 2] = float("inf"), float("nan"), -float("inf")
    m2 = torch.randn(B, N, Kd, generator=gen(N)).to(xdt).to(dev).transpose(-1, -2) if view else \
        torch.randn(B, Kd, N, generator=gen(N)).to(xdt).to(dev)
    m1 = m1.to(dev)
    y = m(m1, m2)
    q1, q2 = m.quantize_operands(m1, m2)
    s1, z1, s2, _ = m._scalars()
    exact = torch.matmul(q1[..., :Kd].double() - z1, q2[..., :Kd].double().transpose(1, 2).contiguous())
    exact = exact * float(torch.tensor(s1) * torch.tensor(s2))
    assert y.shape == exact.shape and y.dtype == xdt
    ulp = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 0.0}[xdt]
    assert ((y.double() - exact).abs() <= exact.abs() * (ulp + 2.0 ** -22) + 2.0 ** -25).all()


@pytest.mark.parametrize("Kd", [65664, 70016])  # 256 * 128 * K on either side of 2^31: 65536
def test_attention_product_whose_corrected_sum_leaves_32_bits(dev, Kd):
    """Codes 127 with zero point -128 against codes 127: 255 * 127 * K is beyond 2^31 from K = 66311 on.
    The correction in fp32 costs two roundings of terms twice the result."""
    m = make_qbmm(dev, 0.0, 1.0, 3.0, torch.float32)
    m1, m2 = torch.ones(1, 3, Kd, device=dev), torch.full((1, Kd, 5), 3.0, device=dev)
    assert ((m(m1, m2).double() / (3.0 * Kd) - 1).abs() < 2e-6).all()


@pytest.mark.parametrize("wdt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("smooth", [False, True])
@pytest.mark.parametrize("N,Kd", [(1, 8), (3, 16), (4, 2040), (5, 2048), (130, 2056), (7, 4104)])
def test_weight_quantizer_with_fp32_divisors(dev, wdt, smooth, N, Kd):
    """The short exact quotient against the IEEE one: ties (integers and halves times the divisor), codes
    past the range, infinities, NaN (code -127), zeros, and rows whose divisor leaves the range it serves."""
    g = gen(N * Kd)
    w = 0.05 * torch.randn(N, Kd, generator=g)
    c = 2.0 ** torch.randint(-12, 3, (N,), generator=g).float() * (1 + (torch.rand(N, generator=g) > 0.5) * torch.rand(N, generator=g))
    half = torch.arange(Kd) % 300 - 150
    w[::2] = 0.5 * half * c[::2, None]
    w[-1, :8] = torch.tensor([float("inf"), -float("inf"), float("nan"), 0.0, -0.0, 6e4, -6e4, 1e-7])
    if N > 4:
        c[0], c[1], c[2], c[3] = 1e-38, 0.0, -0.01, float("inf")
    w = w.to(wdt)
    s = 0.25 + 4 * torch.rand(Kd, generator=g) if smooth else None
    t = w.float() * s if smooth else w.float()
    ref = torch.nan_to_num((t / c[:, None]).round().clamp(-127, 127), nan=-127.0).to(torch.int8)
    q, rows = K().quant_weight_i8(w.to(dev), c.to(dev), s.to(dev) if smooth else None, mode="div", want_row_sum=True)
    assert torch.equal(q.cpu(), ref)
    assert torch.equal(rows.cpu(), ref.int().sum(1, dtype=torch.int32))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_conversion_in_eval_and_training_mode(dev, dtype):
    """from_fms_mo leaves the weight quantizer as a forward on the weights would, and its buffers equal those of
    the torch expressions evaluated on the same GPU."""
    import copy

    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    for train in (False, True):
        m = make_qlinear(264, 37, dtype).to(dev)
        m.smoothq, m.smoothq_alpha = True, torch.full((1,), 0.5, device=dev)
        m.smoothq_act_scale = 0.5 + torch.rand(264, generator=gen(3)).to(dev)
        m.quantize_weight.train(train)
        other = copy.deepcopy(m)
        dep = QLinearINT8Deploy.from_fms_mo(m, use_dynamic_max_act_Qfunc=-1)
        with torch.no_grad():
            other.quantize_weight(other.weight)
        a, b = m.quantize_weight, other.quantize_weight
        assert a.Niter == b.Niter and torch.equal(a.clip_val, b.clip_val) and torch.equal(a.clip_valn, b.clip_valn)
        ws = b.clip_val * 2 / torch.tensor(254.0, device=dev)
        wm = other.weight.detach().abs().max(dim=0, keepdim=True)[0].clamp(min=1e-5)
        sq = (m.smoothq_act_scale ** m.smoothq_alpha / wm ** (1.0 - m.smoothq_alpha)).clamp(min=1e-5)
        codes = ((other.weight.detach() * sq).t() / ws).round().clamp(-127, 127).t().to(torch.int8)
        assert torch.equal(dep.w_scale, ws) and torch.equal(dep.smoothq_scale, sq) and torch.equal(dep.weight, codes)
        assert dep.input_zp.dtype == torch.int32 and int(dep.input_zp) == 127 and dep.corr_term.abs().max() == 0


@pytest.mark.parametrize("M,N,Kd", [(385, 4100, 8192), (769, 4090, 12800), (1024, 2176, 9216), (641, 5000, 8320)])
def test_most_of_a_round_of_tiles_in_one_pass(dev, M, N, Kd):
    """129 .. 256 tiles of 128 x 128 and a long reduction, ragged edges included: int8 exact, e4m3 exact on
    small integers (sums below 2^24)."""
    kn = K()
    assert kn.gemm_plan(M, N, Kd, with_workspace=True)[1:] == (128, 128, 1)
    g = torch.Generator(device=dev).manual_seed(M)
    a = torch.randint(-128, 128, (M, Kd), generator=g, dtype=torch.int8, device=dev)
    w = torch.randint(-128, 128, (N, Kd), generator=g, dtype=torch.int8, device=dev)
    assert torch.equal(kn.gemm_i8_i32(a, w), (a.double() @ w.double().t()).to(torch.int32))
    a, w = a.float().div(32).round(), w.float().div(32).round()
    one = torch.ones(1, device=dev)
    y = kn.gemm_fp8_dq(a.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn), one, one, None, out_dtype=torch.float32)
    assert torch.equal(y, (a.double() @ w.double().t()).float())


@pytest.mark.parametrize("xdt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,R,C,ldq", [
    (5, 64, 300, 128), (32, 64, 2048, 128), (3, 40, 131, 128), (2, 1, 5, 64), (1, 65, 64, 128),
    (2, 130, 70, 512),            # several blocks past the data
    (32, 300, 2048, 320), (32, 250, 2048, 448), (24, 700, 2100, 1024)])   # several tiles per block
def test_column_sums_of_a_padded_transposed_operand(dev, xdt, B, R, C, ldq):
    """The sums of the transposing quantizer fill fmsmo_affine_sum_parts parts and nothing behind them, however
    far ldq is padded; rows of q past R are zero."""
    from fms_mo_amd import _lib as L

    kn, lib = K(), L.load()
    x = (2 * torch.randn(B, R, C, generator=gen(R + C))).to(xdt).to(dev)
    parts = lib.fmsmo_affine_sum_parts(B, R, C, 1)
    guard = 4 * B * C
    sums = torch.full((parts * B * C + guard,), 0x5a5a5a5a, dtype=torch.int32, device=dev)
    q = torch.full((B, C, ldq), 99, dtype=torch.int8, device=dev)
    dt = kn._dt(x)
    assert lib.fmsmo_quant_i8_affine_sums(x.data_ptr(), dt, C, R * C, 0.03125, 3.0, dt, 1, q.data_ptr(), ldq, C * ldq,
                                          sums.data_ptr(), B, R, C, torch.cuda.current_stream().cuda_stream) == 0
    ref = (x / 0.03125 + 3.0).round().clamp(-128, 127).to(torch.int8).transpose(1, 2)
    assert torch.equal(q[..., :R], ref) and not q[..., R:].any()
    assert torch.equal(sums[:parts * B * C].view(parts, B, C).sum(0), ref.sum(-1, dtype=torch.int32))
    assert (sums[parts * B * C:] == 0x5a5a5a5a).all()


@pytest.mark.parametrize("xdt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Kd", [16, 40, 64, 72, 128])
def test_attention_scores_of_a_stored_second_operand(dev, xdt, Kd):
    """Scores whose second operand is stored [k, n]: its codes are padded to the 128 of the kernel for short
    reductions, beyond the data's last 64 rows for head dimensions up to 64."""
    m = make_qbmm(dev, -0.7, 1.0, 3.0, xdt)
    m1 = torch.randn(3, 140, Kd, generator=gen(Kd)).to(xdt).to(dev)
    m2 = torch.randn(3, Kd, 300, generator=gen(Kd + 1)).to(xdt).to(dev)
    y = m(m1, m2)
    assert torch.equal(y, m(m1, m2.transpose(1, 2).contiguous().transpose(1, 2)))
    q1, q2 = m.quantize_operands(m1, m2)
    s1, z1, s2, _ = m._scalars()
    exact = torch.matmul(q1[..., :Kd].double() - z1, q2[..., :Kd].double().transpose(1, 2).contiguous()) * (s1 * s2)
    ulp = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[xdt]
    assert ((y.double() - exact).abs() <= exact.abs() * (ulp + 2.0 ** -22) + 2.0 ** -25).all()


@pytest.mark.parametrize("odt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,M,Kd,N,ldy", [
    (3, 1, 640, 100, 100), (2, 130, 1024, 64, 70), (2, 300, 1024, 100, 100), (2, 129, 512, 129, 129),
    (2, 140, 192, 300, 300), (2, 140, 128, 300, 300), (2, 140, 128, 300, 312)])
def test_zero_point_product_with_one_or_several_parts(dev, odt, B, M, Kd, N, ldy):
    """fmsmo_bmm_i8_zp with the sums of the second operand in parts and added up first: the same bits, and the
    exact integer times the scale rounded twice (fp32, output).  Output rows may be further apart than N."""
    from fms_mo_amd import _lib as L

    lib, st = L.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev).manual_seed(M + N)
    a = torch.randint(-128, 128, (B, M, Kd), generator=g, dtype=torch.int8, device=dev)
    w = torch.randint(-128, 128, (B, N, Kd), generator=g, dtype=torch.int8, device=dev)
    whole = w.sum(-1, dtype=torch.int32)
    parts = torch.randint(-9999, 9999, (11, B, N), generator=g, dtype=torch.int32, device=dev)
    parts[4] += whole - parts.sum(0, dtype=torch.int32)
    scale, zero, ys = 0.0371, -77, []
    for add in (False, True):
        if add:
            assert lib.fmsmo_affine_add_parts(parts.data_ptr(), 11, B * N, st) == 0
            assert torch.equal(parts[0], whole)
        y = torch.full((B, M, ldy), 7.0, dtype=odt, device=dev)
        assert lib.fmsmo_bmm_i8_zp(a.data_ptr(), Kd, w.data_ptr(), Kd, N * Kd, scale, zero, parts.data_ptr(),
                                   1 if add else 11, y.data_ptr(), K()._DT[odt], ldy, B, M, N, Kd, st) == 0
        assert (y[..., N:] == 7.0).all()
        ys.append(y[..., :N])
    acc = torch.matmul(a.double() - zero, w.double().transpose(1, 2).contiguous())
    ref = (acc.float() * torch.tensor(scale, dtype=torch.float32, device=dev)).to(odt)   # |acc| < 2^31, one rounding each
    assert torch.equal(ys[0], ys[1]) and torch.equal(ys[0], ref)


@pytest.mark.parametrize("M,Kd,N", [(70, 130, 140), (140, 80, 200)])
def test_attention_operands_are_copied_once(dev, monkeypatch, M, Kd, N):
    """m1 [batch, heads, rows, k] that lies as [batch, rows, heads, k] is made contiguous once."""
    kn = K()
    m = make_qbmm(dev, -1.0, 1.0, 3.0, torch.float32)
    m1 = torch.randn(2, M, 3, Kd, generator=gen(M)).to(dev).transpose(1, 2)
    m2 = torch.randn(2, 3, Kd, N, generator=gen(N)).to(dev)
    ref = m(m1.contiguous(), m2)
    copies, batched3 = [], kn._batched3

    def spy(t):
        out = batched3(t)
        copies.extend([t.shape] if out.data_ptr() != t.data_ptr() else [])
        return out

    monkeypatch.setattr(kn, "_batched3", spy)
    assert torch.equal(m(m1, m2), ref)
    assert copies == [m1.shape]


@pytest.mark.parametrize("M,N,Kd", [(33, 250, 9472), (40, 100, 4016), (65, 1000, 4096), (200, 1024, 1536)])
def test_a_workspace_with_room_for_fewer_slices_is_used(dev, M, N, Kd):
    """Slices of unequal length (K = 74 x 128 and K % 128 != 0) and of equal length: with room for fewer slices than
    the plan would take the call makes fewer, within the room; with room for one it leaves the workspace alone."""
    from fms_mo_amd import _lib as L

    st = torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=dev).manual_seed(M)
    a = torch.randint(-128, 128, (M, Kd), generator=g, dtype=torch.int8, device=dev)
    w = torch.randint(-128, 128, (N, Kd), generator=g, dtype=torch.int8, device=dev)
    ref = (a.double() @ w.double().t()).to(torch.int32)
    full = L.load().fmsmo_gemm_workspace_bytes(M, N, Kd) // (M * N * 4)
    assert full > 2
    for room in (1, 2, full - 1, full):
        ws = torch.full((room * M * N + 64,), 0x55555555, dtype=torch.int32, device=dev)
        c = torch.empty((M, N), dtype=torch.int32, device=dev)
        L.call("fmsmo_gemm_i8_i32_ws", a.data_ptr(), Kd, w.data_ptr(), Kd, c.data_ptr(), N, M, N, Kd,
               ws.data_ptr(), room * M * N * 4 + 16, st)
        assert torch.equal(c, ref)
        assert bool((ws[:2 * M * N] != 0x55555555).any()) == (room > 1), room
        assert (ws[room * M * N:] == 0x55555555).all()


@pytest.mark.parametrize("Kd", [16, 64, 272, 1000])          # shorter than a stage, one stage, cut last stages
@pytest.mark.parametrize("M,N", [(1, 1), (65, 131), (128, 128), (130, 260)])
@pytest.mark.parametrize("dtype", [torch.int8, torch.float8_e4m3fn, torch.float16, torch.float32])
def test_chunked_products_at_the_edges_of_tiles_and_of_the_reduction(dev, M, N, Kd, dtype):
    """Integer-valued operands whose partial sums stay below 2^24: every chunk sum and every sum of rounded
    chunks is exact in fp32 whatever its order, so the result is bit-pinned for all operand types."""
    if dtype == torch.float32:
        Kd = Kd // 4 * 4
    elif Kd % 16:
        Kd = Kd // 16 * 16
    a = torch.randint(-6, 7, (M, Kd), generator=gen(M + Kd)).float().to(dtype)
    w = torch.randint(-6, 7, (N, Kd), generator=gen(N + Kd + 1)).float().to(dtype)
    for cs, t in ((32, 3), (64, 5), (128, 4)):
        if dtype == torch.int8:
            ref = O.chunk_matmul_i8(a, w, None, cs, t, 32)
        else:
            ref = O.chunk_matmul_fp(a.float(), w.float(), None, cs, t)
        d = K().matmul_chunk(a.to(dev), w.to(dev), None, chunk_size=cs, chunk_trun_bits=t)
        assert torch.equal(d.cpu(), ref), (cs, t)
        one = torch.ones(1, device=dev)
        y = K().matmul_chunk_dq(a.to(dev), w.to(dev), one, one, None, 1, torch.float32, chunk_size=cs, chunk_trun_bits=t)
        assert torch.equal(y.cpu(), ref.float()), (cs, t)


@pytest.mark.parametrize("tta,dl16,bits", [(True, False, 14), (True, True, 32), (False, False, 32), (False, True, 32), (False, False, 14)])
@pytest.mark.parametrize("M,N,Kd", [(1, 1, 16), (65, 131, 272), (130, 260, 1024)])   # K below, past and at the end of a stage
@pytest.mark.parametrize("dtype", [torch.int8, torch.float8_e4m3fn, torch.float16, torch.float32])
def test_chunked_products_clamped_or_with_a_rounded_running_sum(dev, M, N, Kd, dtype, tta, dl16, bits):
    """What is done at the end of a chunk beside the common configuration, with and without an initial accumulator, bits to
    round or none: integer-valued operands whose sums stay below 2^24, exact in fp32 in any order (as in the test above)."""
    a = torch.randint(-6, 7, (M, Kd), generator=gen(M + Kd)).float().to(dtype)
    w = torch.randint(-6, 7, (N, Kd), generator=gen(N + Kd + 1)).float().to(dtype)
    c0 = torch.randint(-999, 999, (M, N), generator=gen(5)).to(torch.int32 if dtype == torch.int8 else torch.float32)
    for cs, t in ((32, 3), (64, 0), (256, 5)):
        for c in (None, c0):
            if dtype == torch.int8:
                ref = O.chunk_matmul_i8(a, w, c, cs, t, bits, tta)
            else:
                ref = O.chunk_matmul_fp(a.float(), w.float(), c, cs, t, dl16, tta)
            d = K().matmul_chunk(a.to(dev), w.to(dev), None if c is None else c.to(dev), chunk_size=cs, chunk_trun_bits=t,
                                 max_acc_bits=bits, truncate_then_accumulate=tta, clamp_acc_to_dl16=dl16)
            assert torch.equal(d.cpu(), ref), (cs, t, c is not None)


@pytest.mark.parametrize("M,N", [(1030, 2050), (1024, 2048), (65, 129)])   # 561 and 512 tiles of 64 x 64, ragged ones
@pytest.mark.parametrize("Kd", [272, 256])
@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, torch.float16, torch.bfloat16, torch.float32])
def test_chunked_products_in_floating_point_on_either_tile(dev, M, N, Kd, dtype):
    """Both sides of the line between 64 x 64 and 128 x 128 tiles, every schedule and the DL16 clamp, an initial accumulator:
    integer-valued operands, exact in fp32 in any order (as in the test above).  On real values a row has the same bits on
    either tile."""
    a = torch.randint(-6, 7, (M, Kd), generator=gen(M + Kd)).float().to(dtype)
    w = torch.randint(-6, 7, (N, Kd), generator=gen(N + Kd + 1)).float().to(dtype)
    c = torch.randint(-999, 999, (M, N), generator=gen(5)).float()
    esz = a.element_size()
    for cs, t, dl16, c0 in ((64 // esz, 4, False, None), (128 // esz, 0, False, c), (256 // esz, 5, True, None), (64 // esz, 3, True, c)):
        cs = max(cs, 32 if esz == 1 else 16)
        ref = O.chunk_matmul_fp(a.float(), w.float(), c0, cs, t, dl16)
        d = K().matmul_chunk(a.to(dev), w.to(dev), None if c0 is None else c0.to(dev), chunk_size=cs, chunk_trun_bits=t,
                             clamp_acc_to_dl16=dl16)
        assert torch.equal(d.cpu(), ref), (cs, t, dl16)
    a, w = (torch.randn(s, Kd, generator=gen(s)).to(dtype).to(dev) for s in (1030, 2050))
    for dl16 in (False, True):
        big = K().matmul_chunk(a, w, None, chunk_size=64, chunk_trun_bits=5, clamp_acc_to_dl16=dl16)
        assert torch.equal(K().matmul_chunk(a[:M], w[:N], None, chunk_size=64, chunk_trun_bits=5, clamp_acc_to_dl16=dl16), big[:M, :N])


@pytest.mark.parametrize("M,N,Kd,cs", [(16, 130, 8192, 64), (129, 100, 4112, 128), (40, 600, 4096 + 48, 32),
                                       (1100, 4096, 6144, 64),     # 288 tiles: whole ones and cut ones in one launch
                                       (70, 260, 6000, 4096)])     # few, long chunks
@pytest.mark.parametrize("dtype", [torch.int8, torch.float8_e4m3fn, torch.float16])
def test_chunked_products_whose_reduction_is_cut(dev, M, N, Kd, cs, dtype):
    """The sums of the slices against the uncut launch (no workspace) and, where it is quick, the oracle: integer-valued
    operands, whose rounded chunks add up exactly in fp32 in any grouping (as in the test above)."""
    from fms_mo_amd import _lib as L

    lib = L.load()
    a = torch.randint(-6, 7, (M, Kd), generator=gen(M + Kd)).float().to(dtype).to(dev)
    w = torch.randint(-6, 7, (N, Kd), generator=gen(N + Kd + 1)).float().to(dtype).to(dev)
    op, esz, t = K()._OPDT[dtype], a.element_size(), 5
    nbytes = lib.fmsmo_matmul_chunk_workspace_bytes(op, M, N, Kd, cs, 1)
    if cs < 4096:
        assert nbytes > 0
    acc = torch.int32 if dtype == torch.int8 else torch.float32

    def run(limit):
        d = torch.full((M, N), -7, dtype=acc, device=dev)
        ws = torch.full((max(limit, 16),), 0x5a, dtype=torch.uint8, device=dev)
        tail = (32, 1) if dtype == torch.int8 else (0, 1)
        head = (a.data_ptr(), Kd, w.data_ptr(), Kd) + (() if dtype == torch.int8 else (op,))
        L.call("fmsmo_matmul_chunk_i8_ws" if dtype == torch.int8 else "fmsmo_matmul_chunk_fp_ws", *head, None, d.data_ptr(), N,
               M, N, Kd, cs, t, *tail, ws.data_ptr() if limit else None, limit, torch.cuda.current_stream().cuda_stream)
        return d

    whole = run(0)
    for limit in {nbytes, nbytes // 2, nbytes - 16}:
        if limit > 0:
            assert torch.equal(run(limit), whole), limit
    if dtype == torch.int8 and nbytes:   # a size below zero is no room
        d, ws = torch.empty((M, N), dtype=acc, device=dev), torch.full((nbytes,), 0x5a, dtype=torch.uint8, device=dev)
        L.call("fmsmo_matmul_chunk_i8_ws", a.data_ptr(), Kd, w.data_ptr(), Kd, None, d.data_ptr(), N, M, N, Kd, cs, t, 32, 1,
               ws.data_ptr(), -1, torch.cuda.current_stream().cuda_stream)
        assert torch.equal(d, whole) and bool((ws == 0x5a).all())
    if N < 1000:
        ref = (O.chunk_matmul_i8(a.cpu(), w.cpu(), None, cs, t, 32) if dtype == torch.int8
               else O.chunk_matmul_fp(a.cpu().float(), w.cpu().float(), None, cs, t))
        assert torch.equal(whole.cpu(), ref)


@pytest.mark.parametrize("dtype", [torch.float8_e4m3fn, torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,Kd,cs", [(130, 8192, 64), (600, 4096 + 48, 32)])
def test_chunked_rows_do_not_depend_on_the_rows_beside_them(dev, dtype, N, Kd, cs):
    """Real-valued operands, whose rounded chunks do not add up exactly: every row has the bits of the launch without a
    workspace, which adds its chunks one after the other, whatever the number of rows."""
    from fms_mo_amd import _lib as L

    a = torch.randn(300, Kd, generator=gen(Kd)).to(dtype).to(dev)
    w = torch.randn(N, Kd, generator=gen(N)).to(dtype).to(dev)
    d = torch.empty((300, N), device=dev)
    L.call("fmsmo_matmul_chunk_fp", a.data_ptr(), Kd, w.data_ptr(), Kd, K()._OPDT[dtype], None, d.data_ptr(), N, 300, N, Kd,
           cs, 5, 0, 1, torch.cuda.current_stream().cuda_stream)
    one = torch.ones(1, device=dev)
    for M in (1, 16, 129, 300):
        assert torch.equal(K().matmul_chunk(a[:M], w, None, chunk_size=cs, chunk_trun_bits=5), d[:M]), M
        for a_scale in (one, 1.0 * one.expand(M).contiguous(), one.reshape(1, 1)):   # native call (twice), general path
            y = K().matmul_chunk_dq(a[:M], w, a_scale, one, None, 1, torch.float32, chunk_size=cs, chunk_trun_bits=5)
            assert torch.equal(y, d[:M]), M


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Kd,N,bias,stats", [(264, 37, True, "some"), (256, 256, False, "some"), (520, 300, True, "zero"),
                                             (8, 1, False, "none"), (512, 257, True, "extreme")])
def test_vectors_of_a_converted_linear(dev, dtype, Kd, N, bias, stats):
    """One launch for the vectors against the torch expressions on the same GPU: ends of 256-channel groups, a
    statistic of zero (SmoothQuant is left out), no statistics at all, statistics and weights at both ends of the range."""
    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    m = make_qlinear(Kd, N, dtype, bias=bias).to(dev)
    if stats != "none":
        m.smoothq, m.smoothq_alpha = True, torch.full((1,), 0.4, device=dev)
        m.smoothq_act_scale = 0.5 + torch.rand(Kd, generator=gen(3)).to(dev)
    if stats == "zero":
        m.smoothq_act_scale[Kd - 1] = 0
    if stats == "extreme":
        with torch.no_grad():
            m.weight[:, :4] = 0
            m.weight[:, 4:8] = 6e4
        m.smoothq_act_scale[2], m.smoothq_act_scale[3] = 1e-30, 1e30
        m.smoothq_act_scale[6], m.smoothq_act_scale[7] = 1e-30, float("nan")
    dep = QLinearINT8Deploy.from_fms_mo(m, use_dynamic_max_act_Qfunc=-1, recalc_clipvals=False)
    cv, w = m.quantize_weight.clip_val, m.weight.detach()
    ws = cv * 2 / torch.tensor(254.0, device=dev)
    if stats in ("none", "zero"):
        sq = torch.ones(1, device=dev, dtype=dtype)
    else:
        wm = w.abs().max(dim=0, keepdim=True)[0].clamp(min=1e-5)
        sq = (m.smoothq_act_scale ** m.smoothq_alpha / wm ** (1.0 - m.smoothq_alpha)).clamp(min=1e-5)
    codes = torch.nan_to_num(((w * sq).t() / ws).round().clamp(-127, 127).t(), nan=-127.0).to(torch.int8)
    assert dep.smoothq_scale.dtype == sq.dtype and torch.equal(torch.nan_to_num(dep.smoothq_scale), torch.nan_to_num(sq))
    assert torch.equal(dep.w_scale, ws) and torch.equal(dep.weight, codes)
    b = m.bias.detach().float() if bias else torch.zeros(N, device=dev)
    assert dep.bias.dtype == dtype and torch.equal(dep.bias, b.to(dtype)) and torch.equal(dep.corr_term, torch.zeros_like(ws))
    assert torch.equal(dep.w_zp, torch.zeros(N, dtype=torch.int32, device=dev)) and int(dep.input_zp) == 127
    assert list(dep.state_dict()) == ["weight", "input_scale", "input_zp", "w_scale", "w_zp", "smoothq_scale", "corr_term", "bias"]
    assert float(dep.input_scale) == 1 and [float(v) for v in dep.cvs[:2]] == [8.0, -8.0]


def test_conversion_broadcasts_a_bias_of_one_element_and_refuses_another_length(dev):
    """The kernel for the vectors reads one bias per output channel: other lengths are left to the torch expressions."""
    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    m = make_qlinear(256, 96, torch.float16, bias=True).to(dev)
    for n in (1, 7, 95, 97):
        m.bias = torch.nn.Parameter(torch.full((n,), 0.25, device=dev).half())
        if n == 1:
            dep = QLinearINT8Deploy.from_fms_mo(m, use_dynamic_max_act_Qfunc=-1, recalc_clipvals=False)
            assert torch.equal(dep.bias, torch.full((96,), 0.25, device=dev).half())
        else:
            with pytest.raises(RuntimeError):
                QLinearINT8Deploy.from_fms_mo(m, use_dynamic_max_act_Qfunc=-1, recalc_clipvals=False)


@pytest.mark.parametrize("counts,N,Kd,tile", [
    ([3, 0, 1, 5], 130, 256, (64, 64, 128)),                                     # a few rows per expert
    ([0] * 40 + [1, 2, 33] + [0] * 30 + [64, 1], 72, 384, (64, 64, 128)),        # more groups than lanes, most of them empty
    ([43, 64, 65, 0], 200, 1024, (64, 64, 128)),
    ([180, 256, 100, 129, 181], 1100, 640, (64, 64, 128)),
    ([41, 0, 60, 63], 8203, 256, (32, 128, 128)),                                # whole and ragged tiles of 32 rows
    ([1, 31, 32, 33, 2, 0, 9, 10, 64, 65, 1, 7, 8, 0, 0, 12], 8190, 384, (32, 128, 128)),
    ([20] * 69 + [65], 4097, 384, (32, 128, 128)),                               # more groups than lanes
    ([40] * 64 + [0, 7, 128, 1, 1, 3], 4100, 384, (128, 128, 64)),
    ([0, 40, 60], 1100, 192, (128, 128, 64)),                                    # reduction of whole 64-byte stages only
    ([350, 300, 257, 384, 1], 2500, 4096, (128, 128, 128)),
    ([1, 128, 129, 42], 8200, 256, (128, 128, 64)),
    ([513, 0, 700, 2000], 8200, 512, (256, 256, 128)),
    ([10, 200, 127], 300, 192, (128, 128, 64)),
    ([2049, 0, 1800, 255], 8200, 1216, (256, 256, 64))])
@pytest.mark.parametrize("exact_ref,out_dtype", [(True, torch.float16), (False, torch.float32)])
def test_grouped_products_in_every_tile(dev, counts, N, Kd, tile, exact_ref, out_dtype):
    """Bit-identical to one product per expert (integer sums, the same epilogue), rows of no expert untouched."""
    from fms_mo_amd import _lib as L

    kn = K()
    E, lead, T = len(counts), 3, sum(counts) + 5     # three rows in front of the first expert's, two behind the last one's
    for rows in (T - 5, T):
        assert kn.grouped_gemm_plan(E, rows, N, Kd)[1:] == tile
    g = torch.Generator(device=dev).manual_seed(N)
    a = torch.randint(-128, 128, (T, Kd), generator=g, dtype=torch.int8, device=dev)
    w = torch.randint(-128, 128, (E, N, Kd), generator=g, dtype=torch.int8, device=dev)
    sa, sw = torch.rand(T, generator=g, device=dev) * 1e-3, torch.rand(E, N, generator=g, device=dev) * 1e-2
    b = torch.randn(E, N, generator=g, device=dev)
    off = torch.tensor([lead] + counts, device=dev).cumsum(0).to(torch.int32)
    y = torch.full((T + 1, N), -7.0, device=dev, dtype=out_dtype)
    L.call("fmsmo_grouped_gemm_i8_dq", a.data_ptr(), Kd, w.data_ptr(), Kd, N * Kd, off.data_ptr(), E, T, sa.data_ptr(), sw.data_ptr(),
           b.data_ptr(), L.F32, L.EPI_REF_F16 if exact_ref else L.EPI_F32, y.data_ptr(), kn._DT[out_dtype], N, N, Kd,
           torch.cuda.current_stream().cuda_stream)
    inner = kn.grouped_gemm_i8_dq(a[lead:-2], w, off - lead, sa[lead:-2], sw, b, out_dtype=out_dtype, exact_ref=exact_ref)
    assert torch.equal(inner, y[lead:-3]) and (y[:lead] == -7).all() and (y[-3:] == -7).all()
    lo = lead
    for e, c in enumerate(counts):
        if c:
            ref = kn.gemm_i8_dq(a[lo:lo + c], w[e], sa[lo:lo + c], sw[e], b[e], out_dtype=out_dtype, exact_ref=exact_ref)
            assert torch.equal(y[lo:lo + c], ref), e
        lo += c


@pytest.mark.parametrize("M,N,Kd,slices", [
    (17, 12290, 1024, 1), (33, 8200, 4096, 1), (64, 28600, 2048, 1),       # up to 64 tokens, many columns
    (65, 1000, 1920, 1), (100, 5000, 128, 1), (129, 2050, 3072, 1), (257, 1030, 8064, 1),   # up to one block per unit
    (700, 1500, 1536, 1), (4033, 500, 1024, 1), (1, 64, 256, 0),           # up to two; (a decode launch beside them)
    (100, 1000, 2176, 4), (70, 300, 4736, 4), (128, 1024, 14336, 8), (90, 60, 12416, 8)])   # slices, the last one shorter
def test_small_tiles(dev, M, N, Kd, slices):
    """64 x 64 tiles at the ends of the ranges that take them, ragged edges included: int8 exact, e4m3 exact on small
    integers (sums below 2^24), rows and columns past the end untouched."""
    kn = K()
    for fp8 in (False, True):
        plan = kn.gemm_plan(M, N, Kd, with_workspace=True, fp8=fp8)
        if slices:
            assert plan[1:3] == (64, 64) and plan[3] == slices, plan
    g = torch.Generator(device=dev).manual_seed(M + N)
    a = torch.randint(-128, 128, (M, Kd), generator=g, dtype=torch.int8, device=dev)
    w = torch.randint(-128, 128, (N, Kd), generator=g, dtype=torch.int8, device=dev)
    assert torch.equal(kn.gemm_i8_i32(a, w), (a.double() @ w.double().t()).to(torch.int32))
    a, w = a.float().div(32).round(), w.float().div(32).round()
    ref = (a.double() @ w.double().t()).float()
    one = torch.ones(1, device=dev)
    y = kn.gemm_fp8_dq(a.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn), one, one, None, out_dtype=torch.float32)
    assert torch.equal(y, ref)
    sa, sw = torch.rand(M, generator=g, device=dev), torch.rand(N, generator=g, device=dev)
    y = kn.gemm_i8_dq(a.to(torch.int8), w.to(torch.int8), sa, sw, None, out_dtype=torch.float32, exact_ref=False)
    torch.testing.assert_close(y, ref * (sa[:, None] * sw[None, :]), rtol=1e-6, atol=0)


@pytest.mark.parametrize("M,N,Kd,tile", [
    (1025, 900, 8192, (64, 64)), (1030, 70, 8320, (64, 64)),            # above 1024 rows: up to a round of 64 x 64 tiles,
    (1300, 1279, 2176, (128, 64)), (2700, 641, 14336, (128, 64)),       # then of 128 x 64 ones, however long the reduction
    (2000, 2559, 512, (128, 128)), (1400, 25590, 640, (128, 128)),                      # short ones
    (1000, 6143, 2048, (128, 192)), (385, 8193, 1408, (128, 192)), (3900, 1930, 1536, (128, 256)),  # one round, more than of
    (1200, 2999, 6016, (128, 128)), (1200, 2999, 6144, (128, 128)),     # 128 x 128; eight waves, int8 from 6144 on four
    (1100, 1601, 6016, (128, 64)), (1100, 1601, 6144, (128, 64))])
def test_tiles_of_many_rows_and_of_short_reductions(dev, M, N, Kd, tile):
    """Ragged edges of the tiles that such launches take: int8 exact, e4m3 exact on small integers (sums below 2^24)."""
    kn = K()
    assert kn.gemm_plan(M, N, Kd, with_workspace=True)[1:] == (*tile, 1)
    g = torch.Generator(device=dev).manual_seed(M + N)
    a = torch.randint(-128, 128, (M, Kd), generator=g, dtype=torch.int8, device=dev)
    w = torch.randint(-128, 128, (N, Kd), generator=g, dtype=torch.int8, device=dev)
    assert torch.equal(kn.gemm_i8_i32(a, w), (a.double() @ w.double().t()).to(torch.int32))
    a, w = a.float().div(32).round(), w.float().div(32).round()
    one = torch.ones(1, device=dev)
    y = kn.gemm_fp8_dq(a.to(torch.float8_e4m3fn), w.to(torch.float8_e4m3fn), one, one, None, out_dtype=torch.float32)
    assert torch.equal(y, (a.double() @ w.double().t()).float())


@pytest.mark.parametrize("dtype,compute", [(torch.float16, torch.float16), (torch.bfloat16, torch.bfloat16),
                                           (torch.float16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("M,N,Kd,pad", [(1, 1, 1, 64), (5, 63, 8, 64), (130, 129, 128, 128), (64, 200, 65, 64), (3, 70, 1030, 64),
                                        (257, 80, 512, 64)])
@pytest.mark.parametrize("turned", [False, True])
def test_both_operands_of_a_product_quantized_in_one_launch(dev, dtype, compute, M, N, Kd, pad, turned):
    """Codes and sums of the pair against the two launches it stands for, rows of a wider tensor included."""
    from fms_mo_amd import _lib as L

    kn, B = K(), 3
    a = torch.randn(B, M, Kd + 3, generator=gen(M)).to(dtype).to(dev)[:, :, :Kd]
    b = torch.randn(B, Kd if turned else N, (N if turned else Kd) + 5, generator=gen(N)).to(dtype).to(dev)
    b = b[:, :, :N if turned else Kd]
    b[0, 0, 0] = float("inf")
    q1 = kn.quant_i8_affine(a, 0.03125, 3, compute, False, pad)
    q2, sums = kn.quant_i8_affine(b, 0.02, -7, compute, turned, pad, want_sums=True)
    ld = q1.shape[2]
    p1, p2, s2 = torch.full_like(q1, 99), torch.full_like(q2, 99), torch.full_like(sums, 99)
    L.call("fmsmo_quant_i8_affine_pair", kn._DT[dtype], kn._DT[compute], B, a.data_ptr(), a.stride(1), a.stride(0), 0.03125, 3.0,
           p1.data_ptr(), p1.stride(0), M, b.data_ptr(), b.stride(1), b.stride(0), 0.02, -7.0, int(turned), p2.data_ptr(),
           p2.stride(0), s2.data_ptr(), N, Kd, ld, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(p1, q1) and torch.equal(p2, q2) and torch.equal(s2, sums)
    assert torch.equal(sums.sum(0, dtype=torch.int32), q2.sum(2, dtype=torch.int32))
