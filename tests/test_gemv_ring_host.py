"""Which batch-1 projections take the kernel whose waves stream through a ring of loads (csrc/gemv_ring.hip): host-side decisions for 256 CUs, no pointer is followed."""
import pytest

from chatts_amd import _lib


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def takes(lib, form, n, k, epi=_lib.EPI_NONE, norm=False, **kw):
    a = _lib.LinearArgs(**{**dict(a=0x10000000, w=0x7f0000000000, c=0x20000000, m=1, n=n, k=k, lda=k, ldw=k, ldc=n, epilogue=epi, norm_w=0x30000000 if norm else None), **kw})
    if form != "bf16":
        a.w8, a.w8_scale, a.ldw8, a.w8_format = 0x7e0000000000, 0x7d0000000000, k, _lib.W8_INT8 if form == "int8" else _lib.W8_FP8
    return int(lib.chatts_gemv_ring(a))


# both sides of every line: us of gemv_ldsx_kernel / of the ring beside the shape
@pytest.mark.parametrize("form,n,k,want", [
    ("bf16", 4096, 4096, 1),               # 8.2 / 7.9
    ("bf16", 8192, 2048, 0),               # 7.6 / 8.1
    ("bf16", 12288, 2560, 1),
    ("bf16", 2560, 8192, 0),               # five tasks a CU: the K split
    ("bf16", 3072, 8192, 1),               # six: 12.1 / 11.0
    ("bf16", 65504, 4096, 1),
    ("bf16", 65536, 4096, 0),              # vocabularies keep two workgroups a CU: 151936 x 4096 192 / 192, 152064 x 5120 232 / 235
    ("bf16", 4096, 16384, 0),              # x of more than 64 KB
    ("fp8", 152064, 5120, 1),              # 127 / 122
    ("fp8", 7168, 5120, 1),                # 9.7 / 9.0
    ("fp8", 8192, 4096, 0),                # 32 MB
    ("int8", 6144, 4096, 0),               # 7.5 / 7.9
    ("fp8", 5120, 8192, 0),                # ten tasks a CU: 10.1 / 10.4
    ("fp8", 5120, 10240, 1),               # 11.6 / 11.4
    ("fp8", 6144, 7168, 0),                # twelve: 10.8 / 11.2
    ("int8", 6144, 8192, 1),
    ("fp8", 4096, 12288, 1),               # eight: 12.2 / 11.0
])
def test_the_faster_side(lib, form, n, k, want):
    assert takes(lib, form, n, k) == want


def test_gated_and_normed(lib):
    for form in ("bf16", "fp8", "int8"):
        assert takes(lib, form, 24576, 4096, _lib.EPI_SWIGLU, norm=True) == 1
    assert takes(lib, "bf16", 5120, 2560, norm=True) == 0 and takes(lib, "bf16", 5120, 2560) == 1      # (the K split of short matrices behind a norm)


@pytest.mark.parametrize("why,kw", [("4-bit codes", dict(w4=0x40000000, w4_sz=0x50000000, ldw4=2048, w4_group=128)), ("an exchange over ranks", dict(tp_reduce=0x60000000)), ("two rows", dict(m=2)),
                                    ("another activation", dict(epilogue=_lib.EPI_GELU))])
def test_calls_that_stay_out(lib, why, kw):
    assert takes(lib, "bf16", 4096, 4096) == 1
    epi = kw.get("epilogue", _lib.EPI_RESID)
    assert takes(lib, "bf16", 4096, 4096, epi, **{k: v for k, v in kw.items() if k != "epilogue"}) == 0


def test_switches(lib):
    with _lib.options(GEMV_RING=0):
        assert takes(lib, "bf16", 4096, 4096) == 0
    with _lib.options(GEMV_RING=2):
        assert takes(lib, "bf16", 32, 32) == 1 and takes(lib, "fp8", 6144, 4096) == 1
    for opts in (dict(GEMV_ROWS=4), dict(GEMV_UNR=4), dict(GEMV_KS=4)):
        with _lib.options(**opts):
            assert takes(lib, "bf16", 4096, 4096) == 0 and takes(lib, "fp8", 4096, 12288) == 1
