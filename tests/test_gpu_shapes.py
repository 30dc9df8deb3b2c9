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
