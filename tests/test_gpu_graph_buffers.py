"""Captured forwards of the deployed modules and the buffers they read: a replay follows a buffer that was written to in place, whatever
eager calls in between found out and let go of."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def static_linear(dev, K, dtype):
    from fms_mo_amd.modules.linear import QLinear, QLinearINT8Deploy

    q = QLinear(K, 200, bias=True, num_bits_feature=8, qa_mode="maxmin", num_bits_weight=8, qw_mode="maxperCh",
                qcfg={"smoothq": False}, device=dev).to(dev).to(dtype)
    q.quantize_weight.float(), q.quantize_feature.float()
    with torch.no_grad():
        q.quantize_weight.clip_val.copy_(q.weight.abs().amax(dim=1))
        q.quantize_feature.clip_valn.fill_(-3.0), q.quantize_feature.clip_val.fill_(4.0)
    return QLinearINT8Deploy.from_fms_mo(q.eval()).to(dtype)


def captured(m, x):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        m(x)  # (what the host keeps of the buffers is read before the capture)
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y = m(x)
    return g, y


def fill_freed_memory(dev):
    return [torch.full((n,), 1e30, device=dev) for n in (1, 2, 64, 200, 256) for _ in range(64)]


@pytest.mark.parametrize("M,K", [(2, 640), (50, 1040), (300, 1024)])  # quantizer inside the product; in front of it
@pytest.mark.parametrize("dtype,scale_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                               (torch.bfloat16, torch.float32)])
def test_replay_of_a_static_forward_reads_the_scale_of_the_module(dev, M, K, dtype, scale_dtype):
    m = static_linear(dev, K, dtype)
    m._buffers["input_scale"] = m.input_scale.to(scale_dtype)
    g = torch.Generator().manual_seed(M)
    x = torch.randn(M, K, generator=g).to(dtype).to(dev)
    want = m(x)
    graph, y = captured(m, x)
    graph.replay()
    assert torch.equal(y, want)
    m.input_scale.mul_(2)
    graph.replay()
    want = m(x)
    assert torch.equal(y, want)
    for i in range(3):
        m(x.half() if dtype == torch.bfloat16 else x.bfloat16())  # parameters for another dtype of x ...
        m.cvs[0] = m.cvs[0].clone()                               # ... and of another clip value, of the same number
        m(x)
        held = fill_freed_memory(dev)
        m.input_scale.mul_(0.5)
        graph.replay()
        assert torch.equal(y, m(x)), i
        del held


@pytest.mark.parametrize("M", [1, 40])
def test_replay_of_a_dynamic_forward_follows_the_scale_of_the_weights(dev, M):
    """w_scale of 16 bits: the fp32 copy that the products read."""
    from fms_mo_amd.modules.linear import QLinear, QLinearINT8Deploy

    q = QLinear(1024, 300, bias=True, num_bits_feature=8, qa_mode="pertokenmax", num_bits_weight=8, qw_mode="maxperCh",
                qcfg={"smoothq": False}, device=dev).to(dev).half()
    q.quantize_weight.float()
    with torch.no_grad():
        q.quantize_weight.clip_val.copy_(q.weight.abs().amax(dim=1))
    m = QLinearINT8Deploy.from_fms_mo(q.eval(), use_dynamic_max_act_Qfunc=-1, recalc_clipvals=False).half()
    x = torch.randn(M, 1024, generator=torch.Generator().manual_seed(M)).half().to(dev)
    graph, y = captured(m, x)
    for i in range(3):
        m.w_scale.mul_(2)
        want = m(x)
        held = fill_freed_memory(dev)
        graph.replay()
        assert torch.equal(y, want) and torch.equal(m(x), want), i
        del held
    m.w_scale.mul_(0.25)
    late = torch.cuda.CUDAGraph()
    with torch.cuda.graph(late):  # the buffer changed since the last eager call: converted inside the graph, kept by nobody
        z = m(x)
    want = m(x)
    assert torch.equal(want, m(x)) and not torch.equal(want, y)
    late.replay()
    assert torch.equal(z, want)


@pytest.mark.parametrize("M,N,K,smooth", [(1, 640, 9216, False), (2, 256, 6144, False), (4, 1024, 2048, True), (6, 4112, 256, True)])
def test_replay_of_what_is_one_launch_eagerly_and_two_in_a_graph(dev, M, N, K, smooth):
    """The same bits and the same scales either way."""
    from fms_mo_amd import _lib as L
    from fms_mo_amd.modules.linear import QLinear, QLinearINT8Deploy

    assert L.load().fmsmo_small_linear_better(0, M, N, K, 0) == 2
    q = QLinear(K, N, bias=True, num_bits_feature=8, qa_mode="pertokenmax", num_bits_weight=8, qw_mode="maxperCh",
                qcfg={"smoothq": smooth, "smoothq_alpha": 0.5}, device=dev).to(dev).half()
    q.quantize_weight.float()
    with torch.no_grad():
        q.quantize_weight.clip_val.copy_(q.weight.abs().amax(dim=1))
    if smooth:
        q.smoothq_act_scale = torch.rand(K, device=dev) + 0.1
        q.smoothq_alpha = torch.full((1,), 0.5, device=dev)
    m = QLinearINT8Deploy.from_fms_mo(q.eval(), use_dynamic_max_act_Qfunc=-1, recalc_clipvals=False).half()
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(M)).half().to(dev)
    graph, y = captured(m, x)
    scale = m.input_scale
    graph.replay()
    want = m(x)
    assert torch.equal(y, want) and torch.equal(scale, m.input_scale)
    x.mul_(1.5)
    graph.replay()
    want = m(x)
    assert torch.equal(y, want) and torch.equal(scale, m.input_scale)
