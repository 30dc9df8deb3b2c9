"""Products of a few tokens with any K (csrc/gemv_any.hip): against exact integer sums and 64-bit floating point, and the form with
the quantizer inside against quantizer and product as two calls."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def gen(seed):
    return torch.Generator().manual_seed(seed)


# (M, N, K): tiles of 16 tokens and their edges, half groups and single rows of weights, one 16-byte chunk of K up to many turns of
# the waves, the limits of the 8- and 16-wave launches (K = 1024 | 1040; N = 4096 | 4097; N = 8200 at K = 768 and 784 goes to the tiles;
# the 4-wave launches are those of WIDE below)
SHAPES = [(1, 1, 16), (2, 7, 48), (3, 8, 128), (5, 9, 144), (16, 23, 528), (4, 1000, 640), (15, 8200, 768), (15, 8200, 784),
          (16, 4097, 1024), (16, 4096, 1040), (3, 300, 4224), (12, 700, 6032), (9, 520, 2432), (6, 9000, 6144), (2, 260, 7808),
          (1, 2060, 3072), (2, 2060, 9216), (1, 2060, 9232), (17, 40, 272), (24, 4096, 1168), (32, 513, 4080), (25, 100, 2240), (33, 65, 1008),
          (40, 1100, 2304), (64, 2056, 1920), (64, 31, 976)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_int8_sums_are_exact(dev, M, N, K):
    from fms_mo_amd import kernels as kn

    a = torch.randint(-128, 128, (M, K + 32), generator=gen(1), dtype=torch.int8)[:, 16:K + 16]  # rows of another stride
    w = torch.randint(-128, 128, (N, K), generator=gen(2), dtype=torch.int8)
    want = a.double() @ w.double().t()  # below 2^53: exact
    ad = torch.empty(M, K + 32, dtype=torch.int8, device=dev)[:, 16:K + 16]
    ad.copy_(a)
    assert torch.equal(kn.gemm_i8_i32(ad, w.to(dev)).cpu().double(), want)
    s, sw = torch.rand(M, generator=gen(3)) + 0.5, torch.rand(N, generator=gen(4)) * 1e-3
    b = torch.randn(N, generator=gen(5))
    y = kn.gemm_i8_dq(ad, w.to(dev), s.to(dev), sw.to(dev), b.to(dev), out_dtype=torch.float32, exact_ref=False)
    # two roundings of the scales' product and the fused multiply-add, 2^-24 each, and the sum's conversion
    want = want * (s[:, None] * sw).double() + b.double()
    bound = 4 * 2.0 ** -24 * (want.abs() + b.abs().double() + 1e-6)
    assert bool(((y.cpu().double() - want).abs() <= bound).all())


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_e4m3_sums(dev, M, N, K):
    from fms_mo_amd import kernels as kn

    a = torch.randn(M, K, generator=gen(6)).to(torch.float8_e4m3fn)
    w = torch.randn(N, K, generator=gen(7)).to(torch.float8_e4m3fn)
    one = torch.ones(1, device=dev)
    y = kn.gemm_fp8_dq(a.to(dev), w.to(dev), one, one, out_dtype=torch.float32).cpu().double()
    want, scale = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    # K % 64 != 0: sums as fp32 additions keep them, at most one rounding of 2^-24 of the magnitudes so far per addition and
    # lane, of which a chain has K / 32 + 16; else the e4m3 instruction, which drops what lies 2^-13 or more below the largest
    # product of the 32 that it adds at a time
    per = 2.0 ** -24 * (K / 32 + 16) if K % 64 else 2.0 ** -13
    assert bool(((y - want).abs() <= per * scale + 1e-30).all())


FUSED = [(1, 1, 16), (1, 9, 528), (1, 300, 1040), (1, 4100, 3088), (1, 264, 5376), (1, 72, 7168), (1, 520, 9232), (1, 64, 12288),
         (2, 40, 6144), (3, 1000, 4080), (4, 24, 3072), (4, 2100, 640), (2, 8192, 1024), (8, 520, 512), (7, 17, 496), (4, 4200, 768)]


@pytest.mark.parametrize("M,N,K", FUSED)
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("smooth", ["none", "same", "float32"])
def test_int8_with_its_quantizer(dev, M, N, K, dt, smooth):
    """Codes, scales, clip values and results of the two calls bit for bit, with rows off the quantizer's fast path among them."""
    from fms_mo_amd import _lib as L
    from fms_mo_amd import kernels as kn

    lib = L.load()
    if not lib.fmsmo_small_linear_ok(M, N, K, int(smooth == "float32")):
        assert smooth == "float32"
        pytest.skip("left to the two calls")
    x = torch.randn(M, K, generator=gen(11))
    x[:, 3] *= 40
    if M >= 3:
        x[1] = 0.0
        x[2] *= 1e-30
    if M >= 4:
        x[3, K // 2] = float("inf")
    if M >= 7:
        x[4, 1], x[5, 0] = float("nan"), 6e4
    sm = None
    if smooth != "none":
        sm = torch.rand(K, generator=gen(12)) * 3 + 0.2
        if K == 640:
            sm[7] = 1e-30 if dt == torch.bfloat16 or smooth == "float32" else 0.0  # outside the fast quotient's range
        sm = sm.to(dt if smooth == "same" else torch.float32).to(dev)
    x = x.to(dt).to(dev)
    w = torch.randint(-127, 128, (N, K), generator=gen(13), dtype=torch.int8).to(dev)
    sw, b = (torch.rand(N, generator=gen(14)) * 1e-3).to(dev), torch.randn(N, generator=gen(15)).to(dt).to(dev)
    q, s = kn.quant_act_i8_pertoken(x, sm, compute_dtype=torch.float32 if smooth == "float32" else None)
    for epi, out in ((L.EPI_REF_F16, torch.float16), (L.EPI_F32, torch.float32)):
        want = kn.gemm_i8_dq(q, w, s, sw, b, out_dtype=out, exact_ref=epi == L.EPI_REF_F16)
        y = torch.empty(M, N, dtype=out, device=dev)
        sc, clips = torch.empty(M, device=dev), torch.empty(2, M, device=dev)
        L.call("fmsmo_small_linear_i8", x.data_ptr(), kn._dt(x), K, None if sm is None else sm.data_ptr(),
               0 if sm is None else kn._dt(sm), w.data_ptr(), K, sw.data_ptr(), N, b.data_ptr(), kn._dt(b), epi, y.data_ptr(),
               kn._DT[out], N, sc.data_ptr(), clips.data_ptr(), M, N, K, torch.cuda.current_stream().cuda_stream)
        bits = torch.int16 if out == torch.float16 else torch.int32
        assert torch.equal(sc.view(torch.int32), s.reshape(-1).view(torch.int32))
        assert torch.equal(y.view(bits), want.view(bits))
        assert torch.equal(clips.nan_to_num(7.0), torch.stack((s.reshape(-1) * 127, -(s.reshape(-1) * 127))).nan_to_num(7.0))


@pytest.mark.parametrize("M,N,K", FUSED)
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_e4m3_with_its_quantizer(dev, M, N, K, dt):
    from fms_mo_amd import _lib as L
    from fms_mo_amd import kernels as kn

    x = 2 * torch.randn(M, K, generator=gen(21))
    if M >= 3:
        x[1] = 0.0
    if M >= 4:
        x[3, K // 2] = float("inf")
    x = x.to(dt).to(dev)
    q, s = kn.quant_act_fp8_pertoken(x, L.FP8_LINEAR)
    w = torch.randn(N, K, generator=gen(22)).to(torch.float8_e4m3fn).to(dev)
    sw, b = (torch.rand(N, generator=gen(23)) * 0.01).to(dev), torch.randn(N, generator=gen(24)).to(dt).to(dev)

    def both(w, sw, b):
        y, sc = torch.empty(M, N, device=dev), torch.empty(M, device=dev)
        L.call("fmsmo_small_linear_fp8", x.data_ptr(), kn._dt(x), K, w.data_ptr(), K, sw.data_ptr(), N,
               None if b is None else b.data_ptr(), 0 if b is None else kn._dt(b), y.data_ptr(), 2, N, sc.data_ptr(), M, N, K,
               torch.cuda.current_stream().cuda_stream)
        assert torch.equal(sc.view(torch.int32), s.reshape(-1).view(torch.int32))
        return y, kn.gemm_fp8_dq(q, w, s, sw, b, out_dtype=torch.float32)

    eye = torch.zeros(N, K)
    eye[torch.arange(min(N, K)), torch.arange(min(N, K))] = 1
    y, want = both(eye.to(torch.float8_e4m3fn).to(dev), torch.ones(N, device=dev), None)  # the codes themselves
    assert torch.equal(y.nan_to_num(7.0, 8.0, 9.0), want.nan_to_num(7.0, 8.0, 9.0))
    y, want = both(w, sw, b)
    fin = torch.isfinite(want)
    assert torch.equal(torch.isfinite(y), fin)
    # the same products, added in another order: both within 2^-13 (see test_e4m3_sums) of the magnitudes' sum
    mag = (q.float().abs() @ w.float().abs().t()) * (s.reshape(-1, 1) * sw) + b.float().abs()
    assert bool(((y - want).abs() <= 2 * 2.0 ** -13 * mag)[fin].all())


@pytest.mark.parametrize("K,smooth", [(640, False), (1040, True), (4224, False)])
def test_forward_of_a_small_linear(dev, K, smooth):
    """The deployed module's forward: the same output, input_scale and clip values as by the general path."""
    import types

    from fms_mo_amd import _lib, kernels
    from fms_mo_amd.modules.linear import QLinear, QLinearINT8Deploy

    q = QLinear(K, 200, bias=True, num_bits_feature=8, qa_mode="pertokenmax", num_bits_weight=8, qw_mode="maxperCh",
                qcfg={"smoothq": smooth, "smoothq_alpha": 0.5}, device=dev).to(dev).half()
    q.quantize_weight.float()
    with torch.no_grad():
        q.quantize_weight.clip_val.copy_(q.weight.abs().amax(dim=1))
    if smooth:
        q.smoothq_act_scale = torch.rand(K, device=dev) + 0.1
        q.smoothq_alpha = torch.full((1,), 0.5, device=dev)
    m = QLinearINT8Deploy.from_fms_mo(q.eval(), use_dynamic_max_act_Qfunc=-1, recalc_clipvals=False).half()
    x = torch.randn(2, K, generator=gen(31)).half().to(dev)
    m(x)  # (the scales' host-side facts are found out)
    y, s, c = m(x), m.input_scale, [t.clone() for t in m.cvs[:2]]
    host, h = _lib._host, kernels._H
    stub = types.SimpleNamespace(**{n: (lambda *a: None) for n in dir(_lib.host()) if not n.startswith("_")})
    try:
        _lib._host = kernels._H = stub
        want = m(x)
        assert torch.equal(y, want) and torch.equal(s, m.input_scale)
        if not smooth:
            assert all(torch.equal(a.reshape(-1), b.reshape(-1)) for a, b in zip(c, m.cvs[:2]))
    finally:
        _lib._host, kernels._H = host, h


def test_what_is_left_to_the_two_calls():
    from fms_mo_amd import _lib as L

    lib = L.load()
    assert lib.fmsmo_small_linear_ok(1, 4096, 5376, 0) and not lib.fmsmo_small_linear_ok(1, 4096, 16400, 0)
    assert not lib.fmsmo_small_linear_ok(1, 4096, 5377, 0) and not lib.fmsmo_small_linear_ok(9, 64, 512, 0)
    assert not lib.fmsmo_small_linear_ok(2, 8200, 1024, 0) and lib.fmsmo_small_linear_ok(2, 8200, 4096, 0)
    assert not lib.fmsmo_small_linear_ok(1, 4096, 2048, 1) and lib.fmsmo_small_linear_ok(1, 4096, 4096, 1)


PARAMS = [(7 / 255, -109.0, 0, -3.0, 4.0), (0.0123, 0.0, 1, -1.5, 1.5), (2.0 ** -20, -0.5, 0, -0.25, 0.5), (300.0, 3.25, 1, -6e4, 6e4)]


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("par", PARAMS)
def test_static_codes_in_fp32(dev, dt, par):
    """The kernel with the short division (contiguous rows) against the one with the IEEE division (rows of another stride), on every
    16-bit pattern, and both against torch on the CPU."""
    from fms_mo_amd import _lib as L
    from fms_mo_amd import kernels as kn

    step, zp, sym, lo, hi = par
    x = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(dt).reshape(64, 1024)
    wide = torch.zeros(64, 1032, dtype=dt, device=dev)
    wide[:, :1024] = x.to(dev)
    args = (L.SQ_FMO, torch.float32, step, zp, sym, lo, hi)
    q = kn.quant_act_i8_static_t(x.to(dev), *args)
    assert torch.equal(q, kn.quant_act_i8_static_t(wide[:, :1024], *args))
    f = torch.tensor
    t = x.float().clamp(lo, hi) / f(step) - f(zp)
    ok = ~torch.isnan(x.float())  # (the kernels take NaN for the lower clip value)
    want = (torch.round(t) - (128 - sym)).nan_to_num(0).to(torch.int32).to(torch.int8)
    assert torch.equal(q.cpu()[ok], want[ok])


@pytest.mark.parametrize("M,N,K", [(1, 1, 16), (1, 100, 2064), (3, 23, 528), (4, 9000, 1024), (8, 300, 2048), (16, 4100, 640), (2, 72, 3072)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_int8_with_the_static_quantizer(dev, M, N, K, dt):
    from fms_mo_amd import _lib as L
    from fms_mo_amd import kernels as kn

    x = (3 * torch.randn(M, K, generator=gen(41))).to(dt).to(dev)
    x[0, 1], x[0, K - 1], x[M - 1, 3] = float("inf"), -float("inf"), float("nan")
    w = torch.randint(-127, 128, (N, K), generator=gen(42), dtype=torch.int8).to(dev)
    sw, b = (torch.rand(N, generator=gen(43)) * 1e-3).to(dev), torch.randn(N, generator=gen(44)).to(dt).to(dev)
    for step, zp, sym, lo, hi in PARAMS[:2]:
        assert L.load().fmsmo_small_linear_static_ok(M, N, K, step, zp, lo, hi)
        q = kn.quant_act_i8_static_t(x, L.SQ_FMO, torch.float32, step, zp, sym, lo, hi)
        want = kn.gemm_i8_dq(q, w, torch.tensor([0.0274], device=dev), sw, b, out_dtype=torch.float16, exact_ref=True)
        y = torch.empty(M, N, dtype=torch.float16, device=dev)
        L.call("fmsmo_small_linear_i8_static", x.data_ptr(), kn._dt(x), K, step, zp, sym, lo, hi, 0.0274, w.data_ptr(), K,
               sw.data_ptr(), N, b.data_ptr(), kn._dt(b), L.EPI_REF_F16, y.data_ptr(), 0, N, M, N, K,
               torch.cuda.current_stream().cuda_stream)
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("M,K", [(2, 640), (50, 1040), (3, 4096)])
@pytest.mark.parametrize("bias", [True, False])
def test_forward_of_a_static_linear(dev, M, K, bias, monkeypatch):
    """The native forward against the general one, before and after the module's parameters are written to."""
    import types

    from fms_mo_amd import _lib, kernels
    from fms_mo_amd.modules.linear import QLinear, QLinearINT8Deploy

    q = QLinear(K, 200, bias=bias, num_bits_feature=8, qa_mode="maxmin", num_bits_weight=8, qw_mode="maxperCh",
                qcfg={"smoothq": False}, device=dev).to(dev).bfloat16()
    q.quantize_weight.float(), q.quantize_feature.float()
    with torch.no_grad():
        q.quantize_weight.clip_val.copy_(q.weight.abs().amax(dim=1))
        q.quantize_feature.clip_valn.fill_(-3.0), q.quantize_feature.clip_val.fill_(4.0)
    m = QLinearINT8Deploy.from_fms_mo(q.eval()).bfloat16()
    x = torch.randn(M, K, generator=gen(51)).bfloat16().to(dev)
    stub = types.SimpleNamespace(**{n: (lambda *a: None) for n in dir(_lib.host()) if not n.startswith("_")})

    def general():
        with monkeypatch.context() as c:
            c.setattr(_lib, "_host", stub), c.setattr(kernels, "_H", stub)
            return m(x)

    m(x)  # (the parameters are read)
    assert _lib.host().deploy_i8(m.__dict__, x, QLinearINT8Deploy, __import__("fms_mo_amd.modules.linear", fromlist=["x"])._OWN_METHODS) is not None
    assert torch.equal(m(x), general())
    m.input_scale.mul_(2)
    assert torch.equal(m(x), general())
    m.cvs[0] = m.cvs[0] * 0.5
    assert torch.equal(m(x), general())
    m.quant_stepsize = m.quant_stepsize * 3
    assert torch.equal(m(x), general()) and torch.equal(m(x), general())
    m.qa_fmo_mo_qfunc = lambda t: torch.zeros(t.shape, dtype=torch.int8, device=t.device)
    assert torch.equal(m(x), general())


# More than 8192 columns: the launches of four waves (K <= 768), of two blocks and one per compute unit with several row groups each, and
# of gemv_short_kernel with two and four groups to a block (K <= 512; more than 16384 and 32768 columns)
WIDE = [(1, 8200, 640), (1, 8201, 720), (2, 8200, 640), (2, 9001, 768), (2, 8200, 784), (5, 11003, 2816), (10, 16391, 2432), (16, 8999, 1664),
        (1, 8193, 9232), (4, 8200, 9216), (1, 16400, 272), (16, 20001, 512), (7, 17001, 16), (1, 32790, 496)]


@pytest.mark.parametrize("M,N,K", WIDE)
def test_sums_over_many_columns(dev, M, N, K):
    from fms_mo_amd import _lib as L
    from fms_mo_amd import kernels as kn

    for fp8 in (False, True):
        assert kn.gemm_plan(M, N, K, fp8=fp8)[0] == L.PLAN_DECODE
    test_int8_sums_are_exact(dev, M, N, K)
    test_e4m3_sums(dev, M, N, K)


@pytest.mark.parametrize("M,N,K", [(3, 8200, 640), (16, 8201, 768)])
def test_the_entry_point_of_the_decode_products_takes_four_waves_too(dev, M, N, K):
    """fmsmo_gemv_i8_dq has no tiles to go to."""
    from fms_mo_amd import _lib as L

    a = torch.randint(-128, 128, (M, K), generator=gen(1), dtype=torch.int8)
    w = torch.randint(-128, 128, (N, K), generator=gen(2), dtype=torch.int8)
    ad, wd, one, y = a.to(dev), w.to(dev), torch.ones(1, device=dev), torch.empty(M, N, device=dev)
    L.call("fmsmo_gemv_i8_dq", ad.data_ptr(), K, wd.data_ptr(), K, one.data_ptr(), 1, one.data_ptr(), 1, None, 0, L.EPI_F32, y.data_ptr(), 2, N,
           M, N, K, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(y.cpu().double(), a.double() @ w.double().t())  # below 2^24: exact


@pytest.mark.parametrize("M,N,K", [(1, 8200, 640), (1, 8201, 720), (1, 9000, 16)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_e4m3_with_its_quantizer_over_many_columns(dev, M, N, K, dt):
    test_e4m3_with_its_quantizer(dev, M, N, K, dt)


@pytest.mark.parametrize("M,N,K", [(4, 9000, 640), (1, 8201, 400), (3, 8195, 768)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_int8_with_the_static_quantizer_over_many_columns(dev, M, N, K, dt):
    test_int8_with_the_static_quantizer(dev, M, N, K, dt)


@pytest.mark.parametrize("M,N,K", [(3, 8200, 640), (10, 9001, 2688), (10, 8207, 6016), (11, 8201, 2560), (11, 8201, 2688), (3, 1048605, 640)])
def test_a_group_of_rows_per_block(dev, M, N, K):
    """More than 8192 columns: a block per 16 of them, at the ends of the range, up to 65536 blocks, which own two groups in the last one's case."""
    from fms_mo_amd import _lib as L

    g = torch.Generator(device=dev).manual_seed(M + K)
    a = torch.randint(-64, 64, (M, K), generator=g, dtype=torch.int8, device=dev)
    w = torch.randint(-32, 32, (N, K), generator=g, dtype=torch.int8, device=dev)
    one, y = torch.ones(1, device=dev), torch.empty(M, N, device=dev)
    L.call("fmsmo_gemv_i8_dq", a.data_ptr(), K, w.data_ptr(), K, one.data_ptr(), 1, one.data_ptr(), 1, None, 0, L.EPI_F32, y.data_ptr(), 2, N,
           M, N, K, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(y.double(), a.double() @ w.double().t())  # sums below 2^24: exact
