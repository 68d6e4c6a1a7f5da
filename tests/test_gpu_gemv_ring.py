"""Batch-1 projections of long rows (csrc/gemv_ring.hip): the same bits as gemv_ldsx_kernel for every format, epilogue and norm - rows that end inside a chunk, NaN behind them, one task and
more tasks a wave than it has lanes, x longer than the part of it that a workgroup holds in registers, waves without a task, several products in a launch."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"
GATED = (_lib.EPI_SWIGLU, _lib.EPI_CLAMPGLU, _lib.EPI_GEGLU)


def operands(n, k, ldw, fmt, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(k, generator=g, device=DEV)
    norm = torch.rand(k, generator=g, device=DEV) + 0.5
    if fmt == "bf16":
        w = torch.full((n, ldw), float("nan"), dtype=torch.bfloat16, device=DEV)
        w[:, :k] = (torch.randn((n, k), generator=g, device=DEV) * k ** -0.5).bfloat16()
        return x, norm, dict(w=w)
    q = torch.full((n, ldw), 0x7f, dtype=torch.uint8, device=DEV)      # (NaN in e4m3fn)
    q[:, :k] = torch.randint(0, 120, (n, k), generator=g, device=DEV, dtype=torch.uint8) | (torch.randint(0, 2, (n, k), generator=g, device=DEV, dtype=torch.uint8) << 7)
    return x, norm, dict(w=torch.zeros(8, device=DEV), w8=q, w8_scale=torch.exp2(torch.randint(-8, -4, (n,), generator=g, device=DEV).float()))


def call(lib, x, norm, ops, n, k, epi, fmt, bias, resid):
    cols = n // 2 if epi in GATED else n
    out = torch.full((cols,), float("nan"), device=DEV)
    ldw = ops["w8" if fmt != "bf16" else "w"].shape[1]
    a = _lib.LinearArgs(a=x.data_ptr(), w=ops["w"].data_ptr(), c=out.data_ptr(), m=1, n=n, k=k, lda=k, ldw=ldw, ldc=cols, epilogue=epi, glu_limit=7.0, glu_alpha=1.702,
                        norm_w=norm.data_ptr() if norm is not None else None, norm_eps=1e-6, bias=bias.data_ptr() if bias is not None else None,
                        resid=resid.data_ptr() if epi == _lib.EPI_RESID else None)
    if fmt != "bf16":
        a.w8, a.w8_scale, a.ldw8, a.w8_format = ops["w8"].data_ptr(), ops["w8_scale"].data_ptr(), ldw, _lib.W8_FP8 if fmt == "fp8" else _lib.W8_INT8
    _lib.check(lib.chatts_linear(C.byref(a), _lib.stream_ptr()))
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("fmt", ["bf16", "fp8", "int8"])
@pytest.mark.parametrize("n,k,ldw,nw", [(32, 32, 64, 8), (4128, 2080, 2080, 8), (6176, 4096, 4096, 0), (5120, 5120, 5120, 0), (4096, 3104, 4096, 12), (35968, 544, 1024, 1), (40992, 1024, 1024, 1)])
def test_the_same_bits_as_the_kernel_of_short_rows(fmt, n, k, ldw, nw):
    lib = _lib.load()
    x, norm, ops = operands(n, k, ldw, fmt, n + k)
    bias, resid = torch.randn(n, device=DEV), torch.randn(n, device=DEV)
    epis = [_lib.EPI_NONE, _lib.EPI_RESID, _lib.EPI_SWIGLU] + ([_lib.EPI_RELU2, _lib.EPI_CLAMPGLU, _lib.EPI_GEGLU] if fmt == "bf16" else [])
    for epi in epis:
        for nm in (None, norm):
            # (the norm's sum of squares runs over the workgroup's threads: the same number of waves on both sides)
            with _lib.options(GEMV_KS=1, GEMV8_ROWS=2, GEMV_NW=nw or 8, GEMV_OCC=1, GEMV_RING=0):
                want = call(lib, x, nm, ops, n, k, epi, fmt, bias, resid)
            with _lib.options(GEMV_KS=1, GEMV_NW=nw or 8, GEMV_RING=2):
                got = call(lib, x, nm, ops, n, k, epi, fmt, bias, resid)
            assert torch.isfinite(got).all() and torch.equal(got, want), (epi, nm is not None)


def test_against_float64_where_the_rule_takes_it():
    lib = _lib.load()
    for n, k in ((6144, 4096), (4096, 12288), (7168, 5120)):
        x, norm, ops = operands(n, k, k, "bf16", n)
        z = ops["w"].double() @ (x.double() * torch.rsqrt((x.double() ** 2).mean() + 1e-6) * norm.double())
        out = call(lib, x, norm, ops, n, k, _lib.EPI_NONE, "bf16", None, None)
        assert float((out.double() - z).norm() / z.norm()) < 1e-6      # (products exact, sums of at most 12288 terms and the norm in 32 bits)


def test_several_products_in_a_launch():
    lib = _lib.load()
    n, k, b = 3104, 2560, 3
    x = torch.randn((b, k), device=DEV)
    w = (torch.randn((b, n, k), device=DEV) * k ** -0.5).bfloat16()
    outs = []
    for ring in (0, 2):
        out = torch.full((b, n), float("nan"), device=DEV)
        a = _lib.LinearArgs(a=x.data_ptr(), w=w.data_ptr(), c=out.data_ptr(), m=1, n=n, k=k, lda=k, ldw=k, ldc=n, epilogue=_lib.EPI_NONE, batch=b, a_stride=k, w_stride=n * k, c_stride=n)
        with _lib.options(GEMV_KS=1, GEMV_RING=ring):
            _lib.check(lib.chatts_linear(C.byref(a), _lib.stream_ptr()))
        torch.cuda.synchronize()
        outs.append(out)
    assert torch.isfinite(outs[0]).all() and torch.equal(outs[0], outs[1])


# waves that the rule picks: 5, 9, 12 (two tasks some, one the others), 6, 12, 10, 8 with a ragged last walk
@pytest.mark.parametrize("fmt,n,k", [("bf16", 5120, 4096), ("bf16", 4608, 5120), ("bf16", 4608, 8192), ("fp8", 5120, 10240), ("bf16", 6000, 4096), ("int8", 6144, 8192), ("bf16", 9216, 2560), ("fp8", 10240, 8192),
                                     ("int8", 11264, 4096)])
def test_the_shipped_geometry(fmt, n, k):
    """the waves of the launch as it is chosen, a norm among them, against float64"""
    lib = _lib.load()
    x, norm, ops = operands(n, k, k, fmt, n + k)
    x *= 3.0
    w = ops["w"].double() if fmt == "bf16" else (ops["w8"].view(torch.float8_e4m3fn if fmt == "fp8" else torch.int8).double() * ops["w8_scale"].double()[:, None])
    bias = torch.randn(n, device=DEV)
    for nm in (None, norm):
        z = w @ (x.double() if nm is None else x.double() * torch.rsqrt((x.double() ** 2).mean() + 1e-6) * norm.double()) + bias.double()
        out = call(lib, x, nm, ops, n, k, _lib.EPI_NONE, fmt, bias, None)
        assert float((out.double() - z).norm() / z.norm()) < 1e-6      # (products exact, sums of at most 10240 terms and the norm in 32 bits)
