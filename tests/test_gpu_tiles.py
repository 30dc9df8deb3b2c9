"""Tile shapes of the products (csrc/gemm_launch.hpp), each at ragged edges: against exact sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def check(dev, M, N, K):
    """int8 exact; e4m3 on small integers, whose sums stay below 2^24: exact in fp32."""
    from fms_mo_amd import kernels as kn

    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a = torch.randint(-128, 128, (M, K + 16), generator=g, dtype=torch.int8, device=dev)[:, :K]
    w = torch.randint(-128, 128, (N, K + 32), generator=g, dtype=torch.int8, device=dev)[:, :K]
    acc = a.double() @ w.double().t()
    assert torch.equal(kn.gemm_i8_i32(a, w).double(), acc)
    one = torch.ones(1, device=dev)
    assert torch.equal(kn.gemm_i8_dq(a, w, one, one, None, out_dtype=torch.float32, exact_ref=False).double(), acc)
    # NaN behind the rows' K elements must not enter
    nan = torch.full((), float("nan"), device=dev)
    a8 = torch.cat((torch.randint(-4, 5, (M, K), generator=g, device=dev).float(), nan.expand(M, 16)), 1).to(torch.float8_e4m3fn)[:, :K]
    w8 = torch.cat((torch.randint(-4, 5, (N, K), generator=g, device=dev).float(), nan.expand(N, 16)), 1).to(torch.float8_e4m3fn)[:, :K]
    y = kn.gemm_fp8_dq(a8, w8, one, one, None, out_dtype=torch.float32)
    assert torch.equal(y.double(), a8.double() @ w8.double().t())


@pytest.mark.parametrize("M,N,K", [
    (65, 33, 528), (129, 4100, 1088), (200, 5000, 976), (193, 4801, 1088),         # 64 x 64, 128 x 64
    (1025, 2050, 528), (1000, 2060, 704), (1300, 6000, 528), (1290, 3990, 704),     # 128 x 128, 128 x 192
    (1210, 5142, 848), (1234, 5861, 832), (4000, 4090, 1040), (4010, 4080, 1088)])  # 128 x 256, 256 x 256 (int8)
def test_last_stage_cut_at_k(dev, M, N, K):
    from fms_mo_amd import kernels as kn

    tile = {65: (64, 64), 193: (128, 64), 1000: (128, 128), 1290: (128, 192), 1234: (128, 256), 4010: (256, 256)}.get(M)
    if tile and K % 64 == 0:
        assert kn.gemm_plan(M, N, K)[1:3] == tile
    check(dev, M, N, K)


@pytest.mark.parametrize("M,N,K,tile", [
    (2733, 3200, 1024, (128, 192)), (3367, 2941, 768, (128, 192)), (2050, 2310, 896, (128, 192)), (3627, 5389, 256, (128, 256))])
def test_short_reductions_in_tiles_of_128_rows(dev, M, N, K, tile):
    from fms_mo_amd import kernels as kn

    assert kn.gemm_plan(M, N, K)[1:3] == tile
    check(dev, M, N, K)


@pytest.mark.parametrize("M,N,K,tile", [
    (2, 8200, 272, None), (13, 8300, 640, (64, 64)), (16, 16384, 640, (64, 64)),                    # a few tokens, many columns
    (5, 17001, 528, None), (3, 16500, 704, (32, 128)), (16, 20000, 640, (32, 128)), (32, 16450, 1152, (32, 128)), (17, 16387, 1024, (32, 128))])
def test_a_few_rows_over_many_columns(dev, M, N, K, tile):
    from fms_mo_amd import kernels as kn

    if tile:
        assert kn.gemm_plan(M, N, K)[1:3] == tile
    check(dev, M, N, K)


@pytest.mark.parametrize("counts,N,K,tile", [
    ([0, 3, 90, 1, 65, 41, 0, 6], 4270, 2048, (64, 128)),
    ([1, 63, 64, 65, 0, 5, 128, 129, 40, 0, 2, 70, 90, 30, 7, 33], 2102, 1664, (64, 128)),
    ([129, 1, 697], 4145, 1664, (128, 256)), ([128, 257, 255, 256, 0, 300], 2721, 1152, (128, 256)),
    ([569, 0, 129], 1989, 2304, (128, 128))])
def test_grouped_tiles_of_eight_waves(dev, counts, N, K, tile):
    """int8: exact; experts without rows, with one, and on either side of a tile."""
    from fms_mo_amd import kernels as kn

    E, T = len(counts), sum(counts)
    assert kn.grouped_gemm_plan(E, T, N, K)[1:3] == tile
    g = torch.Generator(device=dev).manual_seed(N)
    a = torch.randint(-128, 128, (T, K), generator=g, dtype=torch.int8, device=dev)
    w = torch.randint(-128, 128, (E, N, K), generator=g, dtype=torch.int8, device=dev)
    off = torch.tensor([0] + counts, device=dev).cumsum(0).to(torch.int32)
    y = kn.grouped_gemm_i8_dq(a, w, off, torch.ones(T, device=dev), torch.ones(E, N, device=dev), None, out_dtype=torch.float32,
                              exact_ref=False)
    lo = 0
    for e, c in enumerate(counts):  # (integer sums, rounded once to fp32)
        want = (a[lo:lo + c].double() @ w[e].double().t()).float()
        assert torch.equal(y[lo:lo + c], want), e
        lo += c


@pytest.mark.parametrize("M,N,K,tile", [
    (100, 1100, 2176, (64, 64)), (64, 8461, 2816, (64, 64)), (128, 8190, 4224, (64, 64)), (200, 700, 3968, (64, 64)),
    (65, 8300, 2816, (128, 64)), (100, 8924, 8320, (128, 64)), (130, 5470, 4224, (128, 64)), (100, 16000, 9344, (128, 64))])
def test_a_few_hundred_rows_in_one_pass(dev, M, N, K, tile):
    from fms_mo_amd import kernels as kn

    for fp8 in (False, True):
        assert kn.gemm_plan(M, N, K, with_workspace=True, fp8=fp8)[1:] == (*tile, 1)
    check(dev, M, N, K)
