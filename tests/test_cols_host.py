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


# both sides of the line, which the matrix draws alone: us of the other two / of this one beside the shape
@pytest.mark.parametrize("form,n,k,epi,want", [
    ("bf16", 24576, 4096, _lib.EPI_SWIGLU, 1),            # 5 rows 39 / 32.5, 16 rows 40.7 / 33.0
    ("bf16", 18432, 4096, _lib.EPI_NONE, 1),              # 44 / 26
    ("bf16", 12288, 4096, _lib.EPI_NONE, 1),
    ("bf16", 12288, 2048, _lib.EPI_NONE, 0),              # 2 rows 10.9 / 11.5
    ("bf16", 12304, 2048, _lib.EPI_NONE, 1),
    ("bf16", 32000, 2048, _lib.EPI_NONE, 1),              # 31 / 23.7
    ("bf16", 12272, 8192, _lib.EPI_NONE, 0),              # 10240 columns 0.83 .. 1.2 times as fast, 8192 0.6 .. 1.0
    ("fp8", 24576, 4096, _lib.EPI_SWIGLU, 1),             # 25.8 / 20.9
    ("fp8", 16384, 4096, _lib.EPI_NONE, 0),               # short K at the lower end: the widest instances of the other two
    ("fp8", 16400, 4096, _lib.EPI_NONE, 1),
    ("fp8", 16384, 8192, _lib.EPI_NONE, 1),               # 37 / 28
    ("fp8", 12288, 4224, _lib.EPI_NONE, 1),
    ("int8", 12288, 4096, _lib.EPI_NONE, 0),
    ("int8", 152064, 5120, _lib.EPI_NONE, 1),
])
def test_the_faster_side(lib, form, n, k, epi, want):
    for m in (2, 5, 8, 9, 16):
        assert takes(lib, form, m, n, k, epi) == want, m


@pytest.mark.parametrize("why,kw", [("17 rows", dict(m=17)), ("a result that does not start on 16 bytes", dict(c=OUT + 4)), ("a result at an odd stride", dict(ldc=24577)), ("a result over A", dict(c=A + 64)),
                                    ("planes of a result over A", dict(c=None, c_hi=A, c_lo=OUT, ld_cplanes=24576)), ("planes at an odd stride", dict(c=None, c_hi=OUT, c_lo=OUT + (1 << 24), ld_cplanes=24578)),
                                    ("a K that ends inside a line", dict(k=4096 + 32, ld_planes=4096 + 32, ldw=4096 + 32)), ("no planes", dict(a_hi=None, a_lo=None, a=A)), ("tiles", dict(planes_tiled=1)),
                                    ("several products", dict(batch=2))])
def test_calls_that_stay_out(lib, why, kw):
    assert takes(lib, "bf16", 5, 24576, 4096) == 1
    kw = dict(kw)
    assert takes(lib, "bf16", kw.pop("m", 5), 24576, kw.pop("k", 4096), **kw) == 0
