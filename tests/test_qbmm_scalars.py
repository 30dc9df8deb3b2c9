"""QBmmINT8Deploy reads its four scalars again when their buffers change."""
import copy
import io
import types

import pytest
import torch

from fms_mo_amd.modules.bmm import QBmmINT8Deploy


def make(hi=1.0, lo=0.0, other=3.0, dtype=torch.float32):
    one = lambda v: torch.tensor([v], dtype=dtype)
    src = types.SimpleNamespace(num_bits_m1=8, num_bits_m2=8, qm1_mode="max",
                                quantize_m1=types.SimpleNamespace(clip_val=one(hi), clip_valn=one(lo), num_bits=8),
                                quantize_m2=types.SimpleNamespace(clip_val=one(other), num_bits=8))
    return QBmmINT8Deploy.from_fms_mo(src, target_device="cpu")


def want(m):
    return float(m.m1_scale), int(m.m1_zp) - 128, float(m.m2_scale), int(m.m2_zp)


def changes():
    yield "load", lambda m: m.load_state_dict(make(2.0, -1.0, 5.0).state_dict())
    yield "assign", lambda m: m.load_state_dict(make(2.0, -1.0, 5.0).state_dict(), assign=True)
    yield "copy", lambda m: m.m1_scale.copy_(torch.tensor([0.25]))
    yield "zp", lambda m: m.m1_zp.fill_(77)
    yield "m2", lambda m: m.m2_scale.mul_(3)
    yield "m2_zp", lambda m: m.m2_zp.add_(1)
    yield "setattr", lambda m: setattr(m, "m2_scale", torch.tensor([0.5]))
    yield "data", lambda m: setattr(m.m1_scale, "data", torch.tensor([0.75]))
    yield "half", lambda m: m.half()


@pytest.mark.parametrize("name,change", list(changes()))
def test_scalars_follow_their_buffers(name, change):
    m = make()
    before = m._scalars()
    assert before == want(m) and m._scalars() is before   # read once
    with torch.no_grad():
        change(m)
    assert m._scalars() == want(m) != before


def test_scalars_of_copies_and_of_inference_tensors():
    m = make()
    m._scalars()
    c = copy.deepcopy(m)
    buf = io.BytesIO()
    torch.save(m, buf)
    buf.seek(0)
    d = torch.load(buf, weights_only=False)
    for other in (c, d):
        with torch.no_grad():
            other.m1_scale.mul_(2)
        assert other._scalars() == want(other) and m._scalars() == want(m) != want(other)
    with torch.inference_mode():
        i = make()
        assert i._scalars() == want(i)


def test_copies_do_not_take_the_scalars_of_the_module_they_came_from():
    """Its buffers' memory, written to and given to the copy, has the addresses and versions of its finding."""
    m = copy.deepcopy(make())   # (a copy's buffers begin at version 1, those of a copy of it too)
    m._scalars()
    memory = [m._buffers[n].detach() for n in ("m1_scale", "m1_zp", "m2_scale", "m2_zp")]
    c = copy.deepcopy(m)
    memory[2].fill_(9.0)
    for n, t in zip(("m1_scale", "m1_zp", "m2_scale", "m2_zp"), memory):
        c._buffers[n].data = t
    assert c._scalars() == want(c) and c._scalars()[2] == 9.0
