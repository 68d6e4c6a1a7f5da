"""Which projections of few rows write their result while other workgroups still read A: never one whose outputs share memory with A (host-side decisions for 256 CUs, no
pointer is followed)."""
import ctypes as C

import pytest

from chatts_amd import _lib

M, N, K = 6, 4096, 4096
PLANE = M * K * 2                                      # bytes of a plane of A
A_HI, A_LO, OUT = 0x10000000, 0x10000000 + PLANE, 0x40000000


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def args(**kw):
    base = dict(w=0x7f0000000000, c=OUT, m=M, n=N, k=K, lda=K, ldw=K, ldc=N, a_hi=A_HI, a_lo=A_LO, ld_planes=K, epilogue=_lib.EPI_NONE, workspace=0x50000000, workspace_bytes=1 << 28)
    return _lib.LinearArgs(**{**base, **kw})


def few_rows(lib, a, chain=None):
    return int(lib.chatts_linear_few_rows(C.byref(a), C.byref(chain) if chain else None))


@pytest.mark.parametrize("at,takes", [(OUT, True), (A_HI, False), (A_LO, False), (A_LO + PLANE, True), (A_LO + PLANE - 16, False), (A_HI - M * N * 4, True), (A_HI - M * N * 4 + 16, False)])
def test_float_result(lib, at, takes):
    assert (few_rows(lib, args(c=at)) > 1) == takes


@pytest.mark.parametrize("hi,lo,takes", [(OUT, OUT + PLANE, True), (A_HI, A_LO, False), (A_LO, A_HI, False), (OUT, A_LO, False), (A_LO + PLANE - 16, OUT, False), (A_HI - M * N * 2, OUT, True),
                                         (OUT, A_HI - M * N * 2 + 16, False)])
def test_planes_as_the_result(lib, hi, lo, takes):
    assert (few_rows(lib, args(c=None, c_hi=hi, c_lo=lo, ld_cplanes=N)) > 1) == takes


def test_strides_count(lib):
    assert few_rows(lib, args(ldc=2 * N, c=A_HI - (M * 2 - 1) * N * 4)) > 1               # (nothing lies behind the last row)
    assert few_rows(lib, args(ldc=2 * N, c=A_HI - (M * 2 - 1) * N * 4 + 16)) == 0
    assert few_rows(lib, args(ld_planes=2 * K, a_lo=A_HI + K * 2, c=A_HI + (2 * M * K) * 2)) > 1      # planes row by row in turn
    assert few_rows(lib, args(ld_planes=2 * K, a_lo=A_HI + K * 2, c=A_HI + (2 * M * K) * 2 - 16)) == 0


@pytest.mark.parametrize("m", [6, 12])                 # the few-rows kernel; the split's epilogue, which keeps to the same rule
@pytest.mark.parametrize("hi,lo,takes", [(OUT + (1 << 24), OUT + (2 << 24), True), (A_HI, A_LO, False), (A_LO, A_HI, False), (OUT + (1 << 24), A_LO, False), (A_HI + 16, OUT + (1 << 24), False),
                                         (OUT + (1 << 24), A_HI + 32, False)])
def test_planes_for_the_norm(lib, m, hi, lo, takes):
    a = args(m=m, a_lo=A_HI + m * K * 2, post_norm_w=0x60000000, post_hi=hi, post_lo=lo, ld_post=N)
    assert (int(lib.chatts_linear_post_ss_parts(C.byref(a))) > 0) == takes


@pytest.mark.parametrize("over", ["a_hi", "a_lo", "c", "post_hi", "row_ss"])
def test_sums_of_squares_have_their_own_memory(lib, over):
    """refused before anything is launched"""
    a = args(post_norm_w=0x60000000, post_hi=OUT + (1 << 24), post_lo=OUT + (2 << 24), ld_post=N)
    chain = _lib.NormChain(row_ss=0x70000000, row_ss_parts=256, row_eps=1e-6)
    chain.post_ss = {"a_hi": A_HI, "a_lo": A_LO + 64, "c": OUT + 32, "post_hi": OUT + (1 << 24) + 16, "row_ss": 0x70000000 + 16}[over]
    assert int(lib.chatts_linear_chain(C.byref(a), C.byref(chain), None)) == _lib.E_SHAPE
    assert b"overlap" in lib.chatts_last_error()


@pytest.mark.parametrize("over", ["c", "c_hi", "c_lo"])
def test_results_leave_the_sums_that_are_read_alone(lib, over):
    a = args() if over == "c" else args(c=None, c_hi=OUT, c_lo=OUT + (1 << 24), ld_cplanes=N)
    chain = _lib.NormChain(row_ss={"c": OUT + 64, "c_hi": OUT - 16 * 256 * 4 + 16, "c_lo": OUT + (1 << 24)}[over], row_ss_parts=256, row_eps=1e-6)
    assert int(lib.chatts_linear_chain(C.byref(a), C.byref(chain), None)) == _lib.E_SHAPE
    assert b"overlap" in lib.chatts_last_error()


# both sides of every line: us of the split with its epilogue / of the few-rows kernel beside the shape
@pytest.mark.parametrize("form,m,n,k,takes", [
    ("bf16", 8, 4096, 4096, True),         # 10.7 / 9.6
    ("bf16", 3, 4096, 12288, True),        # 147 KB of X: 19.9 / 19.2
    ("bf16", 8, 4096, 12288, False),       # 393 KB: 20.1 / 23.5
    ("bf16", 6, 5120, 5120, True),         # 13.0 / 12.5
    ("bf16", 6, 5120, 13824, False),       # 25.2 / 26.3
    ("bf16", 8, 8192, 8192, True),         # four ranges, 256 KB: 32.9 / 31.2
    ("bf16", 7, 8192, 10240, False),       # 28.8 / 31.9
    ("bf16", 2, 4096, 16384, False),       # rows 32 KB apart: 33.3 / 37.6
    ("bf16", 8, 7168, 5120, True),         # the split has more workgroups than CUs: 20.6 / 15.7
    ("bf16", 8, 2048, 6144, False),        # sixteen ranges (the epilogue asks for all their slabs at once): 9.1 / 10.7
    ("bf16", 4, 2048, 6144, True),         # 8.9 / 8.5
    ("bf16", 8, 2048, 4096, False),        # 7.9 / 8.7
    ("bf16", 4, 2048, 4096, True),         # 7.7 / 7.7
    ("bf16", 2, 1024, 4096, False),        # under 8 million weights: 6.3 / 6.8
    ("bf16", 5, 2048, 3584, True),         # fourteen ranges: 7.3 / 7.1
    ("bf16", 6, 2048, 3584, False),        # 7.4 / 7.4
    ("bf16", 2, 1024, 3584, True),         # 6.3 / 6.3
    ("bf16", 4, 1024, 3584, False),        # 6.5 / 6.8
    ("bf16", 6, 1024, 3072, True),         # twelve: 6.4 / 6.4
    ("bf16", 8, 1024, 3072, False),        # 6.4 / 7.1
    ("bf16", 8, 1024, 2304, True),         # nine: 6.3 / 6.0
    ("fp8", 8, 4096, 4096, True),          # 8.3 / 7.6
    ("fp8", 3, 4096, 12288, False),
    ("fp8", 4, 4096, 12288, False),        # 13.1 / 13.8
    ("fp8", 8, 4096, 12288, False),        # 13.2 / 17.7
    ("fp8", 4, 6144, 4096, True),          # 9.4 / 8.4
    ("fp8", 4, 6144, 10240, False),        # five ranges, 164 KB
    ("fp8", 2, 5120, 13824, False),        # six ranges, a third of the fragments empty: 15.6 / 17.2
    ("fp8", 2, 5120, 2048, True),          # four ranges: 31 % less here
    ("int8", 4, 7168, 11264, True),
    ("int8", 8, 4096, 4096, True),         # 8.7 / 7.7
    ("int8", 8, 4096, 12288, False),       # 14.0 / 17.9
])
def test_the_faster_of_the_two(lib, form, m, n, k, takes):
    a = args(m=m, n=n, k=k, lda=k, ldw=k, ldc=n, ld_planes=k, a_lo=A_HI + m * k * 2)
    if form != "bf16":
        a.w8, a.w8_scale, a.ldw8, a.w8_format = 0x7e0000000000, 0x7d0000000000, k, _lib.W8_INT8 if form == "int8" else _lib.W8_FP8
    assert (few_rows(lib, a) > 1) == takes
    a.post_norm_w, a.post_hi, a.post_lo, a.ld_post = 0x60000000, OUT + (1 << 24), OUT + (2 << 24), n
    assert int(lib.chatts_linear_post_ss_parts(C.byref(a))) == 256      # (either of the two hands a norm on; with more than eight ranges the few-rows kernel alone)


@pytest.mark.parametrize("m,k,takes", [(8, 6144, True), (7, 8192, False)])
def test_a_norm_handed_on_from_more_than_eight_ranges(lib, m, k, takes):
    """up to 192 KB of X, and from this kernel only: what the host promises is what the launch does"""
    a = args(m=m, n=2048, k=k, lda=k, ldw=k, ldc=2048, ld_planes=k, a_lo=A_HI + m * k * 2, post_norm_w=0x60000000, post_hi=OUT + (1 << 24), post_lo=OUT + (2 << 24), ld_post=2048)
    assert (int(lib.chatts_linear_post_ss_parts(C.byref(a))) == 256) == takes
    assert (few_rows(lib, a, _lib.NormChain(post_ss=0x70000000)) > 1) == takes and few_rows(lib, a) == 0
