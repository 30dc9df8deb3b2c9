"""The native host calls against the general Python path they stand in for, over the forms that either takes."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def general(monkeypatch):
    """Switches the native calls off (every one answers None) inside a with block."""
    import contextlib

    from fms_mo_amd import _lib, kernels

    names = [n for n in dir(_lib.host()) if not n.startswith("_")]
    stub = types.SimpleNamespace(**{n: (lambda *a: None) for n in names})

    @contextlib.contextmanager
    def off():
        with monkeypatch.context() as m:
            m.setattr(_lib, "_host", stub)
            m.setattr(kernels, "_H", stub)
            yield

    return off


def same(a, b):
    if isinstance(a, (list, tuple)):
        return len(a) == len(b) and all(same(x, y) for x, y in zip(a, b))
    return a.dtype == b.dtype and a.shape == b.shape and torch.equal(a.reshape(-1).contiguous().view(torch.uint8), b.reshape(-1).contiguous().view(torch.uint8))


def forms(Kd, dtype, dev):
    g = torch.Generator(device=dev).manual_seed(5)
    x = lambda *s: torch.randn(*s, generator=g, device=dev).to(dtype)  # noqa: E731
    yield "matrix", x(3, Kd)
    yield "vector", x(Kd)
    yield "three dimensions", x(2, 3, Kd)
    yield "rows of a wider matrix", x(40, Kd + 16)[:, :Kd]
    yield "columns", x(Kd, 6).t()
    yield "strided batch", x(4, 5, Kd)[:, ::2]
    yield "one row of many", x(9, Kd)[4:5]
    yield "needs a gradient", x(20, Kd).requires_grad_()
    yield "many rows", x(200, Kd)
    yield "inference", x(7, Kd)


def qlinear(Kd, N, dtype, bias, dev, smooth):
    from fms_mo_amd.modules.linear import QLinear

    m = QLinear(Kd, N, bias=bias, num_bits_feature=8, qa_mode="pertokenmax", num_bits_weight=8, qw_mode="maxperCh",
                qcfg={"smoothq": smooth}, device=dev)
    with torch.no_grad():
        m.weight.normal_(0, 0.02)
        if bias:
            m.bias.normal_(0, 0.01)
    m.to(dtype)
    m.quantize_weight.float()
    with torch.no_grad():
        m.quantize_weight.clip_val.copy_(m.weight.abs().amax(dim=1))
    if smooth:
        m.smoothq_act_scale = 0.5 + torch.rand(Kd, device=dev)
        m.smoothq_alpha = torch.full((1,), 0.5, device=dev)
    return m.to(dev).eval()


@pytest.mark.parametrize("Kd", [512, 4096])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("smooth,half", [(False, False), (True, False), (True, True)])
def test_deployed_linear(dev, general, Kd, dtype, smooth, half):
    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    m = QLinearINT8Deploy.from_fms_mo(qlinear(Kd, 130, dtype, bool(half), dev, smooth), use_dynamic_max_act_Qfunc=-1)
    if half:
        m = m.to(dtype)
    for name, x in forms(Kd, dtype, dev):
        with torch.inference_mode(name == "inference"):
            y, s, cvs = m(x), m.input_scale, [c.clone() for c in m.cvs[:2]]
            with general():
                y2, s2 = m(x), m.input_scale
                assert same(y, y2) and same(s, s2) and not y.requires_grad, name
                assert same(cvs, [c.reshape(a.shape) for c, a in zip(m.cvs[:2], cvs)]), name


def test_deployed_linear_follows_its_buffers_and_overrides(dev, general):
    """Written, replaced and cast scales, an iaddmm or quantizer of the user's own, a subclass: never a stale answer."""
    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    x = torch.randn(50, 512, device=dev).half()
    m = QLinearINT8Deploy.from_fms_mo(qlinear(512, 64, torch.float16, True, dev, True), use_dynamic_max_act_Qfunc=-1)

    def check():
        y = m(x)
        with general():
            assert same(y, m(x))
        return y

    y0 = check()
    m.w_scale.mul_(2)
    assert not torch.equal(y0, check())
    m.w_scale = m.w_scale.half()
    check()
    m.smoothq_scale = torch.ones(1, device=dev, dtype=torch.float16)   # SmoothQuant off
    check()
    m.iaddmm = lambda bias, a, b: torch.zeros(a.shape[0], b.shape[1], device=a.device, dtype=torch.float16)
    assert not check().any()
    m.set_matmul_op()
    assert check().any()
    m._quantize = lambda a: torch.zeros(a.shape, dtype=torch.int8, device=a.device)
    m(x)
    del m._quantize

    class Own(QLinearINT8Deploy):
        def iaddmm_int(self, bias, m1, m2, out_dtype=None):
            return super().iaddmm_int(bias, m1, m2, out_dtype) * 0

    m.__class__ = Own
    m.set_matmul_op()
    assert not check().any()


@pytest.mark.parametrize("act", ["token", "tensor"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_fp8_linear(dev, general, act, dtype):
    from fms_mo_amd.modules.fp8_linear import FP8Linear

    g = torch.Generator(device=dev).manual_seed(6)
    for Kd, bias, per_channel in ((512, True, True), (4096, False, False)):
        b = torch.randn(130, generator=g, device=dev).to(dtype) if bias else None
        m = FP8Linear.from_float(0.02 * torch.randn(130, Kd, generator=g, device=dev), b, per_channel=per_channel, act=act)
        for name, x in forms(Kd, dtype, dev):
            with torch.inference_mode(name == "inference"):
                y = m(x)
                with general():
                    assert same(y, m(x)), name
    m.dynamic_scale_floor, m.dynamic_scale_in_input_dtype = 1e-5, True
    y = m(x)
    with general():
        assert same(y, m(x))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,C,D", [(1, 70, 64), (200, 200, 80), (257, 257, 128), (300, 300, 128)])
def test_attention_products(dev, general, dtype, M, C, D):
    from fms_mo_amd import kernels

    g = torch.Generator(device=dev).manual_seed(7)
    x = lambda *s: torch.randn(*s, generator=g, device=dev).to(dtype)  # noqa: E731
    cases = [(x(1, 3, M, D), x(1, 3, C, D).transpose(-1, -2)), (torch.softmax(x(1, 3, M, C).float(), -1).to(dtype), x(1, 3, C, D)),
             (x(3, M, 2 * D)[..., :D], x(3, C, D).transpose(-1, -2)), (x(3, M, C), x(3, C, 2 * D)[..., ::2]),
             (x(3, M, D), x(3, D, 1))]
    for m1, m2 in cases:
        args = (m1, m2, 0.03, 3, 0.05, 0, dtype)
        y = kernels.bmm_i8_quantized(*args)
        with general():
            assert same(y, kernels.bmm_i8_quantized(*args))


def test_wrappers_take_and_refuse_what_they_did(dev, general):
    from fms_mo_amd import _lib as L
    from fms_mo_amd import kernels as K

    x = torch.randn(40, 256, device=dev).half()
    w8 = torch.randint(-127, 128, (70, 256), device=dev, dtype=torch.int8)
    wf = torch.randn(70, 256, device=dev).to(torch.float8_e4m3fn)
    ws, b = torch.rand(70, device=dev), torch.randn(70, device=dev).half()
    q, s = K.quant_act_i8_pertoken(x)
    qf, sf = K.quant_act_fp8_pertoken(x)
    calls = [lambda: K.quant_act_i8_pertoken(x, torch.rand(1, 256, device=dev).half().add(0.5).fill_(2)),
             lambda: K.quant_act_i8_pertoken(x, None, torch.float32), lambda: K.quant_act_i8_static(x, 0.1, 3.0, 0),
             lambda: K.quant_act_i8_static_t(x, L.SQ_RAW, torch.float16, 0.1, 3, 1), lambda: K.quant_act_fp8_pertoken(x),
             lambda: K.quant_act_fp8_dynamic(x, L.FP8_FPXACC, True, 1e-5, True), lambda: K.quant_act_fp8_dynamic(x),
             lambda: K.gemm_i8_dq(q, w8, s, ws, b), lambda: K.gemm_i8_dq(q, w8, 0.5, ws, None, torch.float32, exact_ref=False),
             lambda: K.gemm_fp8_dq(qf, wf, sf, ws, b), lambda: K.gemm_fp8_dq(qf, wf, sf, ws.reshape(-1, 1), b),
             lambda: K.matmul_chunk_dq(q, w8, s, ws, b, chunk_size=64, chunk_trun_bits=4),
             lambda: K.matmul_chunk_dq(q[:, :200], w8[:, :200], s, ws, None, chunk_size=32, chunk_trun_bits=4),
             lambda: K.matmul_chunk_dq(qf, wf, sf, ws, b, out_dtype=torch.bfloat16, chunk_size=64, chunk_trun_bits=4),
             lambda: K.grouped_gemm_i8_dq(q, torch.stack([w8, w8]), torch.tensor([0, 11, 40], device=dev, dtype=torch.int32), s,
                                          torch.stack([ws, ws]), torch.stack([b, b]))]
    for i, call in enumerate(calls):
        r = call()
        with general():
            assert same(r, call()), i
    refused = [lambda: K.quant_act_i8_pertoken(x[0]), lambda: K.quant_act_i8_pertoken(x.cpu()), lambda: K.gemm_i8_dq(q, w8[:, :128], s, ws),
               lambda: K.gemm_i8_dq(q, w8, s[:7], ws), lambda: K.gemm_i8_dq(q, w8, s, ws, b[:5]), lambda: K.gemm_i8_dq(q, wf, s, ws),
               lambda: K.matmul_chunk_dq(q, w8, s, ws, chunk_size=48, chunk_trun_bits=4), lambda: K.quant_act_fp8_pertoken(x.double()),
               lambda: K.grouped_gemm_i8_dq(q, w8, torch.zeros(2, device=dev, dtype=torch.int32), s, ws)]
    for i, call in enumerate(refused):
        with pytest.raises(Exception) as here:
            call()
        with general():
            with pytest.raises(Exception) as there:
                call()
        assert type(here.value) is type(there.value) and str(here.value) == str(there.value), i


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Kd", [8, 4096, 40000])
def test_clip_values_come_with_the_scales(dev, general, dtype, Kd):
    """+- scale * 127 of every row, also of rows that take the quantizer's IEEE branch (infinite, NaN, zero)."""
    from fms_mo_amd import _lib as L

    x = torch.randn(70, Kd, device=dev).to(dtype)
    x[3], x[5, 0], x[6, Kd - 1] = 0, float("inf"), float("nan")
    q, s, c0, c1 = L.host().quant_i8_clips(x)
    with general():
        from fms_mo_amd import kernels

        q2, s2 = kernels.quant_act_i8_pertoken(x)
    rows = torch.ones(70, dtype=torch.bool)
    rows[6] = False   # (codes of a row with a NaN are not specified)
    assert torch.equal(q[rows], q2[rows]) and same(s.reshape(-1)[rows], s2[rows])
    assert same(c0[rows], (s2.reshape(-1, 1) * 127)[rows]) and same(c1[rows], -(s2.reshape(-1, 1) * 127)[rows])


def test_graph_capture_and_streams(dev):
    """The calls of a forward on a side stream, captured and replayed several times, against the eager result."""
    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    mods = [QLinearINT8Deploy.from_fms_mo(qlinear(512, 130, torch.float16, True, dev, s), use_dynamic_max_act_Qfunc=-1)
            for s in (False, True)]
    x = torch.randn(30, 512, device=dev).half()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for m in mods:
            m(x)
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = [m(x) for m in mods]
    for i in range(3):
        x.normal_()
        want = [m(x) for m in mods]
        g.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want)), i


def test_scales_in_the_memory_of_the_ones_before(dev, general):
    """A 16-bit weight scale and a SmoothQuant divisor dropped and allocated anew, with other values and no forward in
    between, as a trip through host memory leaves them: the address and the version may be those of the old ones."""
    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    x = torch.randn(50, 512, device=dev).half()
    m = QLinearINT8Deploy.from_fms_mo(qlinear(512, 64, torch.float16, True, dev, True), use_dynamic_max_act_Qfunc=-1).half()

    def replace(name, values):
        old = m._buffers[name].data_ptr()
        m._buffers[name] = None
        tried = []
        while not tried or (tried[-1].data_ptr() != old and len(tried) < 64):
            tried.append(values.to(dev))
        m._buffers[name] = tried[-1]

    scale, divisors = m.w_scale.cpu(), m.smoothq_scale.cpu()
    replace("w_scale", scale)
    replace("smoothq_scale", divisors)
    for i in range(1, 4):
        y0 = m(x)
        replace("w_scale", scale * 2**i)
        replace("smoothq_scale", divisors * 3 if i != 2 else torch.ones_like(divisors))
        y = m(x)
        with general():
            for k in [k for k in m.__dict__ if k.startswith(("_ws_", "_sq_"))]:   # nothing kept
                del m.__dict__[k]
            assert same(y, m(x)) and not torch.equal(y, y0), i


@pytest.mark.parametrize("kind", ["smooth", "plain", "e4m3"])
def test_operands_replaced_while_a_launch_runs(dev, kind):
    """Another thread may replace a module's tensors between the two launches of its forward: here the quantizer's entry
    point does so itself, drops them and writes over memory of their sizes.  The forward ends with those it began with."""
    import ctypes

    from fms_mo_amd import _lib as L
    from fms_mo_amd.modules.fp8_linear import FP8Linear
    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    x = torch.randn(50, 512, device=dev).half()
    if kind == "e4m3":
        m = FP8Linear.from_float(0.02 * torch.randn(128, 512, device=dev), torch.randn(128, device=dev).half(), per_channel=True)
        name = "fmsmo_quant_act_fp8_pertoken"
    else:
        m = QLinearINT8Deploy.from_fms_mo(qlinear(512, 128, torch.float16, True, dev, kind == "smooth"),
                                          use_dynamic_max_act_Qfunc=-1).half()
        name = "fmsmo_quant_act_i8_pertoken" + ("" if kind == "smooth" else "_clips")
    want, host, lib, seen, junk = m(x), L.host(), L.load(), [], []
    addresses = {n: ctypes.cast(getattr(lib, n), ctypes.c_void_p).value for n in host.entries()}

    def replace(*args):
        rc = getattr(lib, name)(*args)
        for held in (m._parameters, m._buffers):
            for n in [n for n, t in held.items() if t is not None and t.dim() > 0]:
                sizes, dtype = held[n].shape, held[n].dtype
                held[n] = None
                junk.extend(torch.full(sizes, 3.0, device=dev).to(dtype) for _ in range(2))
        m.__dict__.pop("_ws_kept", None), m.__dict__.pop("_sq_kept", None)
        junk.extend(torch.full((128,), 7.0, device=dev) for _ in range(2))
        seen.append(rc)
        return rc

    call = ctypes.CFUNCTYPE(ctypes.c_int, *L.SIGNATURES[name])(replace)
    host.bind({**addresses, name: ctypes.cast(call, ctypes.c_void_p).value}, L.raise_status)
    try:
        y = m(x)
    finally:
        host.bind(addresses, L.raise_status)
    assert seen == [0] and same(y, want)


def on_another_gpu(t):
    """A tensor that says it lies on the next GPU (its memory is that of `t`: it is for checks, not for launches)."""
    import ctypes

    class Exchange(ctypes.Structure):   # DLManagedTensor
        _fields_ = [("data", ctypes.c_void_p), ("device_type", ctypes.c_int32), ("device", ctypes.c_int32), ("ndim", ctypes.c_int32),
                    ("code", ctypes.c_uint8), ("bits", ctypes.c_uint8), ("lanes", ctypes.c_uint16), ("shape", ctypes.c_void_p),
                    ("strides", ctypes.c_void_p), ("offset", ctypes.c_uint64), ("context", ctypes.c_void_p), ("deleter", ctypes.c_void_p)]

    raw = t.view(torch.uint8) if t.dtype == torch.float8_e4m3fn else t
    sizes = (ctypes.c_int64 * t.dim())(*t.shape)
    steps = (ctypes.c_int64 * t.dim())(*t.stride())
    code = 0 if raw.dtype in (torch.int8, torch.int32) else 1 if raw.dtype == torch.uint8 else 4 if raw.dtype == torch.bfloat16 else 2
    x = Exchange(t.data_ptr(), 10, t.get_device() + 1, t.dim(), code, 8 * t.element_size(), 1, ctypes.addressof(sizes),
                 ctypes.addressof(steps), 0, None, None)
    new = ctypes.pythonapi.PyCapsule_New
    new.restype, new.argtypes = ctypes.py_object, [ctypes.c_void_p, ctypes.c_char_p, ctypes.c_void_p]
    out = torch.utils.dlpack.from_dlpack(new(ctypes.addressof(x), b"dltensor", None)).view(t.dtype)
    out._keep = (t, x, sizes, steps)
    assert out.get_device() == t.get_device() + 1 and out.shape == t.shape
    return out


def test_native_calls_leave_tensors_of_another_gpu_to_the_general_path(dev):
    from fms_mo_amd import _lib as L

    h, half = L.host(), torch.float16
    x, xb = torch.randn(4, 128, device=dev).half(), torch.randn(1, 2, 8, 64, device=dev).half()
    q, w = torch.ones(4, 128, device=dev, dtype=torch.int8), torch.ones(32, 128, device=dev, dtype=torch.int8)
    qf, wf = q.half().to(torch.float8_e4m3fn), w.half().to(torch.float8_e4m3fn)
    s, ws, b, sm = torch.ones(4, device=dev), torch.ones(32, device=dev), torch.ones(32, device=dev).half(), torch.ones(128, device=dev).half()
    off, w3 = torch.tensor([0, 4], device=dev, dtype=torch.int32), w[None].contiguous()
    calls = [(h.quant_i8, x, sm, None, False), (h.quant_i8_clips, x), (h.quant_i8_static, x, 0.1, 3, 0),
             (h.quant_i8_static_t, x, L.SQ_RAW, half, 0.1, 3, 1, 0.0, 0.0), (h.quant_fp8, x, L.FP8_LINEAR, False, 1e-12, False),
             (h.gemm_dq, q, w, s, ws, b, half, L.EPI_F32), (h.gemm_dq, qf, wf, s, ws, b, half, 0),
             (h.decode_i8, x, w, ws, b, sm, half, L.EPI_F32, False), (h.decode_fp8, x, wf, ws, b, half),
             (h.grouped_i8, q, w3, off, s, ws[None], b[None], half, L.EPI_F32),
             (h.chunk_dq, q, w, s, ws, b, L.EPI_SEQ_OUT, half, 64, 4, 32, True, False),
             (h.bmm_quantized, xb, xb.transpose(-1, -2), 0.1, 0, 0.1, 0, half),
             (h.fp8_linear, {"weight": wf, "weight_scale": ws, "bias": b}, True, x, False, 1e-12, False)]
    for f, *args in calls:
        for i, a in enumerate(args):
            if torch.is_tensor(a):
                assert f(*args[:i], on_another_gpu(a), *args[i + 1:]) is None, (f.__name__, i)
            elif isinstance(a, dict):
                for k in a:
                    assert f(*args[:i], {**a, k: on_another_gpu(a[k])}, *args[i + 1:]) is None, (f.__name__, k)
    from fms_mo_amd.modules import linear

    x = torch.randn(50, 512, device=dev).half()
    m = linear.QLinearINT8Deploy.from_fms_mo(qlinear(512, 64, half, True, dev, True), use_dynamic_max_act_Qfunc=-1)
    m(x)
    call = lambda: h.deploy_i8(m.__dict__, x, type(m), linear._OWN_METHODS)  # noqa: E731
    for held, n in ((m._parameters, "weight"), (m._buffers, "w_scale"), (m._buffers, "smoothq_scale"), (m._buffers, "bias")):
        assert call() is not None
        own, held[n] = held[n], on_another_gpu(held[n].detach())
        assert call() is None, n
        held[n] = own


@pytest.mark.parametrize("smooth,tokens", [(False, 50), (True, 50), (True, 1)])
def test_methods_replaced_on_the_class_or_the_module_are_called(dev, monkeypatch, smooth, tokens):
    """Every method that the forward in Python goes through, replaced where a user would: on the class, on one module."""
    from fms_mo_amd.modules.linear import QLinearINT8Deploy

    x = torch.randn(tokens, 4096, device=dev).half()
    m = QLinearINT8Deploy.from_fms_mo(qlinear(4096, 64, torch.float16, True, dev, smooth), use_dynamic_max_act_Qfunc=-1)
    want = m(x)
    names = ["_smoothq_active", "_w_scale_f32", "_set_input_scale"] + ["_quantize", "qa_dynamic_max_qfunc"] * (not smooth)
    for name in names:
        own, calls = getattr(QLinearINT8Deploy, name), []

        def spy(self, *args):
            calls.append(name)
            return own(self, *args)

        with monkeypatch.context() as p:
            p.setattr(QLinearINT8Deploy, name, spy)
            assert same(m(x), want) and calls, name
        calls.clear()
        m.__dict__[name] = lambda *args: spy(m, *args)
        assert same(m(x), want) and calls, name
        del m.__dict__[name]
        calls.clear()
        assert same(m(x), want) and not calls
