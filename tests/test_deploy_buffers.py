"""What a linear finds out about its tensors is asked again when another one takes their place."""
import copy
import io
import types

import pytest
import torch

from fms_mo_amd.modules.linear import QLinear, QLinearINT8Deploy


def deployed(dynamic=-1, **kwargs):
    q = QLinear(64, 64, bias=True, num_bits_feature=8, qa_mode="pertokenmax" if dynamic else "maxmin", num_bits_weight=8,
                qw_mode="maxperCh", qcfg={"smoothq": False}, device="cpu")
    with torch.no_grad():
        q.weight.normal_(0, 0.02)
        q.quantize_weight.clip_val.copy_(q.weight.abs().amax(dim=1))
        if not dynamic:
            q.quantize_feature.clip_valn.fill_(-3.0)
            q.quantize_feature.clip_val.fill_(4.0)
    m = QLinearINT8Deploy.from_fms_mo(q.eval(), use_dynamic_max_act_Qfunc=dynamic, recalc_clipvals=False, **kwargs)
    m.w_scale = m.w_scale.half()
    m.smoothq_scale = torch.full((1, 64), 2.0).half()
    return m


QUESTIONS = {
    "w_scale": (-1, lambda m: m._w_scale_f32().tolist(), lambda m: m.w_scale.float().tolist(), 0.5),
    "smoothq_scale": (-1, lambda m: m._smoothq_active(), lambda m: bool((m.smoothq_scale != 1).all()), 0.5),
    "input_scale": (False, lambda m: m._static_params(torch.float16)["scale"], lambda m: float(m.input_scale), 0.5),
}


def in_the_place_of(m, name, values):
    """Drops the buffer and puts a new one with these values in, of version 0 and where the old one lay if the allocator
    will have it."""
    old = m._buffers[name]
    dtype, address = old.dtype, old.data_ptr()
    m._buffers[name] = old = None
    tried = []
    for _ in range(64):
        tried.append(torch.empty(values.shape, dtype=dtype))
        if tried[-1].data_ptr() == address:
            break
    tried[-1].numpy()[...] = values.numpy()   # (counts no version, as a copy to a new tensor does not)
    m._buffers[name] = tried[-1]


@pytest.mark.parametrize("name", list(QUESTIONS))
def test_a_buffer_in_the_memory_of_the_one_before(name):
    dynamic, ask, want, factor = QUESTIONS[name]
    m = deployed(dynamic)
    in_the_place_of(m, name, m._buffers[name].clone())
    for _ in range(8):
        assert ask(m) == want(m)
        in_the_place_of(m, name, m._buffers[name].float().mul(factor).to(m._buffers[name].dtype))
        assert ask(m) == want(m)
        m._buffers[name].data = m._buffers[name].data * 3
        assert ask(m) == want(m)
        m._buffers[name].fill_(1)
        assert ask(m) == want(m)
        in_the_place_of(m, name, torch.full_like(m._buffers[name], 2))


def test_the_copy_of_the_weight_scale_stays_where_it_is():
    """A captured graph may hold its address: a change of the buffer is written to the copy, not to another one."""
    m = deployed()
    kept = m._w_scale_f32()
    for change in (lambda: m.w_scale.mul_(0.5), lambda: in_the_place_of(m, "w_scale", m.w_scale.clone() * 2),
                   lambda: setattr(m, "w_scale", m.w_scale.bfloat16())):
        change()
        with torch.inference_mode():
            assert m._w_scale_f32() is kept
        assert kept.tolist() == m.w_scale.float().tolist() and not kept.is_inference()
    m.w_scale = m.w_scale.float()
    assert m._w_scale_f32().data_ptr() == m.w_scale.data_ptr() != kept.data_ptr()
    was = m.w_scale
    m.w_scale = (was * 2).half()       # (another tensor's memory is never written to)
    before = was.clone()
    assert m._w_scale_f32().tolist() == m.w_scale.float().tolist() and torch.equal(was, before)


def test_copies_and_pickles_ask_for_themselves():
    m = deployed()
    m._w_scale_f32(), m._smoothq_active()
    buf = io.BytesIO()
    torch.save(m, buf)
    buf.seek(0)
    for c in (copy.deepcopy(m), torch.load(buf, weights_only=False)):
        assert not c._ws_kept and not c._sq_kept
        c.w_scale.mul_(2)
        assert c._w_scale_f32().tolist() == c.w_scale.float().tolist() != m._w_scale_f32().tolist()
        assert c._smoothq_active() is m._smoothq_active() is True


def test_quantized_weights_and_smoothquant_scale_of_a_weight_in_the_memory_of_the_one_before():
    """The eval-mode caches of a QLinear: another weight, another statistic, another clip value of version 0 where the old
    one lay; what was quantized for the old weight is not kept for the new one."""
    m = QLinear(64, 48, bias=False, num_bits_feature=8, qa_mode="pertokenmax", num_bits_weight=8, qw_mode="max",
                qcfg={"smoothq": True}, device="cpu").eval()
    with torch.no_grad():
        m.weight.normal_(0, 0.02)
        m.quantize_weight.clip_val.fill_(0.1)
        m.smoothq_act_scale.copy_(torch.rand(64) + 0.5)
    x = torch.zeros(1, 64)

    def check():
        scale = m._cached_smoothq_scale(x)
        q, s = m._int_weights(scale)
        fresh = copy.deepcopy(m)
        assert not fresh._wcache and not fresh._sqcache
        scale2 = fresh._cached_smoothq_scale(x)
        q2, s2 = fresh._int_weights(scale2)
        assert torch.equal(scale, scale2) and torch.equal(q, q2) and torch.equal(s, s2)
        assert m._int_weights(m._cached_smoothq_scale(x))[0] is q      # asked once
        return q

    def replace(held, name, values, wrap=lambda t: t):
        address, held[name] = held[name].data_ptr(), None
        tried = [torch.empty(values.shape)]
        while tried[-1].data_ptr() != address and len(tried) < 64:
            tried.append(torch.empty(values.shape))
        tried[-1].numpy()[...] = values.numpy()
        held[name] = wrap(tried[-1])

    for i in range(6):
        q = check()
        replace(m._parameters, "weight", torch.randn(48, 64) * 0.02, lambda t: torch.nn.Parameter(t))
        assert not torch.equal(check(), q)
        replace(m._buffers, "smoothq_act_scale", torch.rand(64) + 0.5)
        check()
        with torch.no_grad():
            m.weight.mul_(0.5)
        check()


def test_attention_scalars_assigned_twice_through_data():
    """Two assignments with no forward in between: the second may lie where the first buffer lay, in the same tensor."""
    from fms_mo_amd.modules.bmm import QBmmINT8Deploy

    one = lambda v: torch.tensor([v])  # noqa: E731
    src = types.SimpleNamespace(num_bits_m1=8, num_bits_m2=8, qm1_mode="max",
                                quantize_m1=types.SimpleNamespace(clip_val=one(4.0), clip_valn=one(-4.0), num_bits=8),
                                quantize_m2=types.SimpleNamespace(clip_val=one(4.0), num_bits=8))
    m = QBmmINT8Deploy.from_fms_mo(src, target_device="cpu")
    m.m2_scale.data = one(1.0)
    for i in range(100):
        assert m._scalars()[2] == float(m.m2_scale)
        address = m.m2_scale.data_ptr()
        m.m2_scale.data = torch.empty(1)
        tried = []
        while not tried or (tried[-1].data_ptr() != address and len(tried) < 200):
            tried.append(torch.empty(1))
        tried[-1].numpy()[...] = 20.0 + i
        m.m2_scale.data = tried[-1]
        del tried
        assert m._scalars()[2] == 20.0 + i
