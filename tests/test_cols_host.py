"""Which projections of few rows take the kernel of wide ones (csrc/gemm_cols.hip): host-side decisions for 256 CUs, no pointer is followed."""
import ctypes as C

import pytest

from chatts_amd import _lib

A, OUT = 0x10000000, 0x7000000000


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def takes(lib, form, m, n, k, epi=_lib.EPI_NONE, **kw):
    a = _lib.LinearArgs(**{**dict(w=0x7f0000000000, c=OUT, m=m, n=n, k=k, lda=k, ldw=k, ldc=n, a_hi=A, a_lo=A + m * k * 2, ld_planes=k, epilogue=epi, workspace=0x50000000,
                                  workspace_bytes=1 << 28), **kw})
    if form != "bf16":
        a.w8, a.w8_scale, a.ldw8, a.w8_format = 0x7e0000000000, 0x7d0000000000, k, _lib.W8_INT8 if form == "int8" else _lib.W8_FP8
    return int(lib.chatts_linear_cols(C.byref(a)))


# up to 1024 columns a workgroup; with 8-bit weights, scales and biases of more than 896 do not fit beside the rings and the sums of 16 rows.  Whatever the number of rows: their bits must not
# depend on it
@pytest.mark.parametrize("form,n,k,bias,want", [("fp8", 229376, 4224, True, 1), ("fp8", 229392, 4224, True, 0), ("int8", 262144, 4224, True, 0), ("fp8", 262144, 4224, False, 1),
                                                ("int8", 262144, 4224, False, 1), ("fp8", 262160, 4224, False, 0), ("bf16", 262144, 2112, True, 1), ("bf16", 262160, 2112, True, 0)])
@pytest.mark.parametrize("m", [2, 8, 9, 16])
def test_what_a_workgroup_holds(lib, form, n, k, bias, want, m):
    assert takes(lib, form, m, n, k, bias=0x30000000 if bias else None) == want
