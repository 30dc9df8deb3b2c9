"""Where a dispatch has its lines, without a GPU: shapes on either side that were measured with the weights coming from memory."""
import pytest

from fms_mo_amd import _lib as L
from fms_mo_amd import kernels


@pytest.mark.parametrize("fp8,M,N,K,smooth_f32,better", [
    (0, 1, 640, 8192, 0, 1), (0, 1, 640, 8208, 0, 2), (0, 1, 2064, 8208, 0, 0), (1, 1, 1024, 11008, 0, 0), (1, 1, 4096, 10240, 0, 1),
    (1, 1, 7168, 4352, 0, 0), (1, 1, 4096, 4352, 0, 1), (1, 1, 11008, 6144, 0, 1), (1, 1, 11008, 7168, 0, 0),
    (0, 2, 6144, 4224, 0, 0), (0, 2, 6144, 3072, 0, 2), (0, 2, 4096, 4224, 0, 1), (0, 2, 1024, 6144, 0, 2), (1, 2, 6144, 4224, 0, 1),
    (1, 2, 6144, 6144, 0, 0), (0, 3, 6144, 3072, 0, 0), (1, 3, 6144, 3072, 0, 1), (0, 4, 6144, 1152, 0, 2), (0, 4, 4096, 3072, 0, 1),
    (0, 4, 4096, 2048, 0, 2), (1, 4, 6144, 3072, 0, 0), (0, 6, 6144, 256, 0, 2), (0, 6, 4096, 256, 0, 1), (1, 8, 8192, 512, 0, 1),
    (0, 2, 6144, 512, 1, 2), (0, 2, 6144, 1024, 1, 1), (0, 1, 6144, 1024, 1, 1), (0, 1, 6144, 512, 1, 2), (0, 6, 2048, 256, 1, 2),
    (0, 1, 28672, 4096, 1, 1), (0, 3, 4096, 14336, 0, 1), (1, 1, 8192, 8192, 0, 1),   # shapes of the streaming kernel and of whole rows
    (0, 9, 64, 512, 0, 0), (0, 1, 4096, 16400, 0, 0), (0, 1, 4096, 5377, 0, 0)])      # not taken at all
def test_one_launch_only_where_it_is_the_better_one(fp8, M, N, K, smooth_f32, better):
    assert L.load().fmsmo_small_linear_better(fp8, M, N, K, smooth_f32) == better


@pytest.mark.parametrize("M,N,K,decode", [
    (5, 11008, 2816, True), (3, 10240, 2560, True), (16, 9088, 1664, True), (2, 12288, 640, True), (13, 8320, 640, False),
    (12, 14336, 896, False), (5, 9216, 768, True), (10, 24576, 2432, True), (10, 24576, 2176, False), (12, 24576, 2432, False), (16, 16384, 2816, True),
    (5, 18944, 1616, True), (16, 9216, 3600, False), (10, 9216, 3600, True), (1, 28672, 528, True), (16, 24576, 5248, True)])
def test_a_few_tokens_over_many_columns(M, N, K, decode):
    for fp8 in (False, True):
        assert (kernels.gemm_plan(M, N, K, fp8=fp8)[0] == L.PLAN_DECODE) is decode
        assert K % 64 or kernels._workspace(M, N, K, "cpu", fp8) is None


@pytest.mark.parametrize("M,N,K,splits", [
    (40, 2176, 3968, 3), (40, 4096, 3072, 3), (32, 6784, 3584, 2), (64, 4096, 3584, 3), (80, 2176, 3328, 3), (128, 4096, 3968, 3), (80, 5504, 6912, 2),
    (64, 8192, 2560, 1), (64, 2176, 2560, 1), (64, 11008, 3584, 1), (128, 4096, 3328, 1), (128, 5504, 4608, 1), (200, 700, 3968, 1)])
def test_slices_where_one_pass_has_too_few_loads_in_flight(M, N, K, splits):
    for fp8 in (False, True):
        plan = kernels.gemm_plan(M, N, K, with_workspace=True, fp8=fp8)
        assert plan[3] == splits and (splits > 1 or plan[1:3] == (64, 64))
        ws = kernels._workspace(M, N, K, "cpu", fp8)
        assert (0 if ws is None else ws.numel()) == (splits * M * N * 4 if splits > 1 else 0)


@pytest.mark.parametrize("experts,rows,N,K,tile", [
    (4, 239, 3712, 10240, (64, 64)), (4, 558, 1792, 9344, (64, 64)), (16, 557, 2048, 11520, (64, 64)),     # 112 .. 256 larger tiles
    (16, 932, 4096, 7168, (128, 128)), (4, 541, 4864, 2688, (64, 128)),                                    # long rows, short ones
    (8, 1643, 1152, 1792, (128, 128)), (4, 1807, 1280, 6272, (128, 128)), (16, 2479, 1280, 9600, (64, 128)),   # more of them, or whole rounds
    (16, 5405, 2048, 1280, (128, 256))])
def test_grouped_tiles_that_leave_half_the_chip_idle(experts, rows, N, K, tile):
    assert kernels.grouped_gemm_plan(experts, rows, N, K)[1:3] == tile


@pytest.mark.parametrize("M,N,K,i8,e4m3", [   # the sizes of test_gpu_tiles.test_last_stage_cut_at_k, and of a few rows over many columns
    (65, 33, 528, (64, 64), (64, 64)), (129, 4100, 1088, (64, 64), (64, 64)), (200, 5000, 976, (128, 64), (128, 64)),
    (193, 4801, 1088, (128, 64), (128, 64)), (1025, 2050, 528, (128, 128), (128, 128)), (1000, 2060, 704, (128, 128), (128, 128)),
    (1300, 6000, 528, (128, 192), (128, 192)), (1290, 3990, 704, (128, 192), (128, 192)), (1210, 5142, 848, (128, 256), (128, 256)),
    (1234, 5861, 832, (128, 256), (128, 256)), (4000, 4090, 1040, (256, 256), (128, 256)), (4010, 4080, 1088, (256, 256), (128, 256)),
    (5, 17001, 528, (32, 128), (32, 128)), (32, 16450, 1136, (32, 128), (32, 128)),
    (1, 17001, 528, (0, 0), (0, 0)), (4010, 4080, 1024, (0, 0), (0, 0))])                # decode kernel; whole stages
def test_tiles_whose_last_stage_is_cut_at_k(M, N, K, i8, e4m3):
    for fp8, tile in ((False, i8), (True, e4m3)):
        assert kernels.gemm_cut_tile(M, N, K, fp8) == tile
        assert K % 64 or K % 128 == 0 or kernels.gemm_plan(M, N, K, fp8=fp8)[1:3] == tile
    with pytest.raises(L.FmsMoHipError):
        kernels.gemm_cut_tile(0, N, K)


@pytest.mark.parametrize("experts,rows,N,K,tile", [
    (16, 406, 5760, 4864, (32, 128)), (16, 386, 4352, 6656, (32, 128)), (16, 590, 4480, 6528, (32, 128)),   # a third tile on a part of the units
    (8, 398, 7424, 5376, (64, 128)), (16, 469, 7168, 4096, (64, 128)), (16, 622, 5632, 5120, (64, 128))])   # two at most, or more rows or columns
def test_grouped_tiles_of_experts_with_few_rows(experts, rows, N, K, tile):
    assert kernels.grouped_gemm_plan(experts, rows, N, K)[1:3] == tile


@pytest.mark.parametrize("M,N,K,splits", [
    (41, 3467, 3120, 3), (44, 1673, 3424, 3), (123, 2739, 3504, 3), (109, 866, 3264, 1), (226, 1395, 3424, 1), (47, 2369, 2960, 2), (56, 3671, 2544, 2), (35, 3278, 2448, 1),
    (47, 2090, 2704, 1), (128, 1601, 3600, 3)])
def test_slices_of_int8_reductions_that_are_cut_at_k(M, N, K, splits):
    assert kernels.gemm_plan(M, N, K, with_workspace=True)[3] == splits
    ws = kernels._workspace(M, N, K, "cpu", False)
    assert (0 if ws is None else ws.numel()) == (splits * M * N * 4 if splits > 1 else 0)
