"""Rules that the host evaluates for a launch, without a GPU."""
import contextlib
import ctypes
import os

import pytest
import torch

from fms_mo_amd import _lib as L
from fms_mo_amd import kernels


@pytest.mark.parametrize("zero", [0, 1, -1, 127, -128, 255, -256, 30000, -(1 << 31)])
def test_zero_point_products_refuse_what_leaves_32_bits(zero):
    """|q1 - zero| <= |zero| + 128 and |q2| <= 128: from (|zero| + 128) * 128 * K >= 2^31 on the corrected sum may
    wrap.  The entry points refuse that before they look at a pointer's contents, the wrapper before it launches."""
    lib = L.load()
    last = ((1 << 31) - 1) // ((abs(zero) + 128) * 128)   # largest K that fits
    buf = (ctypes.c_int8 * 64)()
    p = (ctypes.addressof(buf) + 15) // 16 * 16

    def zp(K):   # (a stride between the entries of b that is refused behind the rule: nothing is ever launched)
        return lib.fmsmo_bmm_i8_zp(p, K, p, K, 0, 1.0, zero, p, 1, p, L.F16, 1, 1, 1, 1, K, None)

    SHAPE, UNSUPPORTED = 2, 4
    top = last // 64 * 64
    assert zp(top + 64) == UNSUPPORTED and (top == 0 or zp(top) == SHAPE)
    assert kernels.zero_sums_fit(zero, last // 128 * 128) and not kernels.zero_sums_fit(zero, last + 1)
    if abs(zero) <= 512:
        assert lib.fmsmo_bmm_qa_ok(L.F16, L.F16, 0.5, float(zero), 32, 64, 64, last) == 1
    assert lib.fmsmo_bmm_qa_ok(L.F16, L.F32, 0.5, float(zero), 32, 64, 64, max(256, last + 1)) == 0


def test_e4m3_plan_and_workspace_are_those_of_the_e4m3_calls():
    """129 .. 256 tiles of 128 x 128 and a long reduction: e4m3 runs in one pass throughout, int8 from 224 tiles on; the
    workspace that is asked for (and allocated) is that of the operand type."""
    if any(os.environ.get(k) for k in ("FMSMO_TILE", "FMSMO_RS", "FMSMO_SPLIT_K", "FMSMO_TALL")):
        pytest.skip("tuning overrides are set")
    lib, rs, dma = L.load(), L.PLAN_TILE_REGISTER_STAGED, L.PLAN_TILE_LDS_DMA
    for M, N, K, i8, fp8 in ((640, 4096, 14336, (rs, 256, 128, 2), (dma, 128, 128, 1)),      # 160 tiles
                             (640, 5120, 13824, (rs, 256, 128, 2), (dma, 128, 128, 1)),      # 200
                             (777, 4096, 12800, (dma, 128, 128, 1), (dma, 128, 128, 1)),     # 224
                             (512, 4096, 14336, (rs, 256, 128, 4), (rs, 256, 128, 4)),       # 128: slices for both
                             (40, 100, 4016, (dma, 128, 64, 3), (dma, 128, 64, 3))):         # the last slice shorter
        for fp8_call, want, size in ((False, i8, lib.fmsmo_gemm_workspace_bytes),
                                     (True, fp8, lib.fmsmo_gemm_fp8_workspace_bytes)):
            plan = kernels.gemm_plan(M, N, K, with_workspace=True, fp8=fp8_call)
            nbytes = want[3] * M * N * 4 if want[3] > 1 else 0
            ws = kernels._workspace(M, N, K, "cpu", fp8_call)
            assert plan == want and size(M, N, K) == nbytes and (ws.numel() if ws is not None else 0) == nbytes, (M, N, K)
    out = [ctypes.byref(ctypes.c_int()) for _ in range(4)]
    assert lib.fmsmo_gemm_fp8_plan(640, 4096, 14336, 2, *out) == 4   # no e4m3 call on the static scratch: refused


def test_fp8_per_tensor_quantizer_of_a_huge_tensor(monkeypatch):
    """From 2^31 groups of eight elements on, more than the two-pass call counts, the column maxima serve as
    before.  (The calls are recorded, not made, and the 32 GiB have no storage.)"""
    names = []
    monkeypatch.setattr(kernels.L, "call", lambda name, *args: names.append((name, args)))
    monkeypatch.setattr(kernels, "_need_gpu", lambda *t: None)
    monkeypatch.setattr(kernels, "_dev", lambda t: contextlib.nullcontext())
    monkeypatch.setattr(kernels, "_stream", lambda t: None)
    for rows, want in ((1 << 20, ["fmsmo_absmax_cols", "fmsmo_quant_act_fp8_dynamic"]),
                       ((1 << 20) - 1, ["fmsmo_quant_act_fp8_tensor"])):
        kernels._quant_act_fp8_dynamic_impl(torch.empty(rows, 1 << 14, dtype=torch.float16, device="meta"), per_tensor=True)
        assert [n for n, _ in names] == want
        assert want[-1] != "fmsmo_quant_act_fp8_dynamic" or (names[-1][1][4] == 1 and names[-1][1][5] is not None)
        names.clear()


def test_chunked_products_ask_for_a_workspace_only_where_they_may_be_cut():
    lib = L.load()
    need = lib.fmsmo_matmul_chunk_workspace_bytes
    assert need(L.OP_I8, 16, 4096, 14336, 64, 1) == 256 * 65536      # 32 tiles, eight slices each
    assert need(L.OP_I8, 1069, 4096, 14336, 64, 1) == 256 * 65536    # 256 whole tiles and 32 cut ones
    assert need(L.OP_I8, 16, 4096, 14336, 64, 0) == 0                # the running accumulator itself is rounded
    assert need(L.OP_I8, 1024, 4096, 14336, 64, 1) == 0              # one whole round
    assert need(L.OP_I8, 16, 4096, 14336, 16384, 1) == 0             # one chunk
    assert need(L.OP_F16, 16, 4096, 4096, 8, 1) == 0 and need(9, 16, 4096, 4096, 64, 1) == 0
    assert need(L.OP_I8, 0, 4096, 4096, 64, 1) == 0 and need(L.OP_I8, 1 << 30, 4096, 4096, 64, 1) == 0


def test_a_grouped_launch_of_a_few_tiles_takes_small_ones():
    """Never 256 x 256, which leave all but a dozen compute units idle, nor anything that is no whole number of stages."""
    for E in (1, 4, 7, 64):
        for rows in (1, 9, 164, 949):
            for N in (1, 59, 256, 300):
                for Kd in (64, 128, 192, 256, 448, 1472, 4096):
                    _, tm, tn, stage = kernels.grouped_gemm_plan(E, rows, N, Kd)
                    assert (tm, tn) != (256, 256) and Kd % stage == 0, (E, rows, N, Kd)
    assert kernels.grouped_gemm_plan(8, 8192, 28672, 4096) == (L.PLAN_TILE_REGISTER_STAGED, 256, 256, 128)
    assert kernels.grouped_gemm_plan(4, 4104, 8200, 1216) == (L.PLAN_TILE_LDS_DMA, 256, 256, 64)
    # tens of thousands of experts: no launch of more than 2^32 threads (one block per possible tile)
    for E, rows, N, Kd in ((1 << 16, 1 << 16, 16384, 128), (1 << 18, 100, 8192, 128), (1 << 20, 1 << 20, 2048, 128)):
        kernel, tm, tn, _ = kernels.grouped_gemm_plan(E, rows, N, Kd)
        assert kernel == L.PLAN_TILE_REGISTER_STAGED or (-(-rows // tm) + E) * -(-N // tn) * 256 < 1 << 32, (E, rows, N)
    for bad in ((0, 8, 8, 64), (1, 0, 8, 64), (1, 8, 8, 96)):
        with pytest.raises(L.FmsMoHipError):
            kernels.grouped_gemm_plan(*bad)


def test_the_columns_cut_off_a_last_round_are_those_of_the_operand_type():
    """int8 takes 128 x 128 tiles up to K = 1280 where that pays, e4m3 up to 640 and by another margin: a launch that does
    has no round of 256 x 256 tiles to cut."""
    if any(os.environ.get(k) for k in ("FMSMO_TILE", "FMSMO_RS", "FMSMO_TAIL_SPLIT")):
        pytest.skip("tuning overrides are set")
    i8, fp8 = L.load().fmsmo_gemm_tail_columns, L.load().fmsmo_gemm_fp8_tail_columns
    assert (i8(1700, 20992, 640), fp8(1700, 20992, 640)) == (0, 2304)
    assert kernels.gemm_plan(1700, 20992, 640)[1:3] == (128, 128) and kernels.gemm_plan(1700, 20992, 640, fp8=True)[1:3] == (256, 256)
    assert i8(2048, 25600, 4096) == fp8(2048, 25600, 4096) == 1024
    assert fp8(4096, 28672, 4096) == fp8(16, 25600, 4096) == fp8(0, 25600, 4096) == 0


def test_parts_of_column_sums_are_added_first_but_for_a_few_rows_and_the_kernel_of_128():
    first = L.load().fmsmo_affine_parts_first
    assert not first(1, 1000, 64, 256) and not first(4, 1, 64, 256) and not first(8, 8, 64, 256) and not first(32, 8, 128, 2048)
    assert first(4, 9, 64, 256) and first(33, 1, 64, 2112) and first(32, 64, 128, 2048) and first(2, 128, 300, 128)
    assert not first(2, 129, 129, 128) and first(2, 129, 128, 128) and first(2, 300, 300, 192)
