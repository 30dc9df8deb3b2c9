"""Rules that the host evaluates for a launch, without a GPU."""
import ctypes

import pytest

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
