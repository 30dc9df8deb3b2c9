"""e4m3 products of one and two tokens add in fp32: sums that the scaled e4m3 matrix instruction, which drops what lies 2^-13 or more
below the largest product of those it adds at a time, does not keep."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# every kernel that serves one or two tokens of these rows: whole rows, streamed in 128-byte steps with and without the quantizer
SHAPES = [(1, n, 1024) for n in (72, 4100, 8200)] + [(1, 8200, 3968)] + \
         [(1, n, k) for k in (10368, 11008, 12928, 13824, 15872) for n in (72, 2056, 4104)] + [(1, 8200, 11008)] + \
         [(2, n, k) for k in (1152, 1920, 3200, 3584, 4608, 4992, 7296, 8064, 9216, 11008, 13824) for n in (72, 4104)] + \
         [(2, n, k) for k in (1152, 3200, 4608, 8064) for n in (8200, 16400)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_small_products_beside_large_ones(dev, M, N, K):
    """Products of 2^7 of either sign and of 2^-8: every partial sum is a multiple of 2^-8 below 2^16, exact in fp32 in any order."""
    from fms_mo_amd import _lib as L
    from fms_mo_amd import kernels as kn
    from fms_mo_amd.modules.fp8_linear import FP8Linear

    x = torch.full((M, K), 2.0 ** -4)
    x[:, 5::32] = 16.0
    x[:, K // 2] = 448.0  # the largest, against a weight of 0: the token's scale is 1, the codes are x
    w = torch.full((N, K), 2.0 ** -4)
    sign = 1.0 - 2.0 * (torch.arange(K // 32)[None, :] + torch.arange(N)[:, None] // 3).remainder(2).float()
    w[:, 5::32] = 8.0 * sign
    w[:, 7::32] *= (1.0 + torch.arange(N).remainder(7).float())[:, None]
    w[:, K // 2] = 0.0
    x, w = x.to(torch.bfloat16).to(dev), w.to(torch.float8_e4m3fn).to(dev)
    want = (x[:1].double() @ w.double().t()).expand(M, N).float()
    q, s = kn.quant_act_fp8_pertoken(x, L.FP8_LINEAR)
    one = torch.ones(N, device=dev)
    assert torch.equal(s.reshape(-1), one[:M])
    assert torch.equal(kn.gemm_fp8_dq(q, w, s, one, out_dtype=torch.float32), want)
    if L.load().fmsmo_small_linear_ok(M, N, K, 0):
        y = torch.empty(M, N, device=dev)
        L.call("fmsmo_small_linear_fp8", x.data_ptr(), kn._dt(x), K, w.data_ptr(), K, one.data_ptr(), N, None, 0, y.data_ptr(), 2, N,
               None, M, N, K, torch.cuda.current_stream().cuda_stream)
        assert torch.equal(y, want)
    m = FP8Linear(K, N, False, {"weights": {"strategy": "channel", "symmetric": True, "dynamic": False},
                                "input_activations": {"strategy": "token", "symmetric": True, "dynamic": True}}).to(dev)
    m.weight.data = w
    assert torch.equal(m(x), want.to(torch.bfloat16))
