"""Projections of 2 .. 8 rows (csrc/gemm_rows.hip, or the split where that is faster) against float64 on the stored weights, and bit for bit against the weight-streaming
kernel that runs 16 rows: columns that deal unevenly over the CUs, K ranges of unequal length, every weight format and epilogue, and an RMSNorm between two
projections."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def planes(lib, x):
    hi, lo = torch.empty((2, *x.shape), dtype=torch.bfloat16, device=DEV)      # (neighbours: the few-rows kernel reads both through one descriptor)
    _lib.check(lib.chatts_split_bf16x2(x.data_ptr(), *x.shape, x.shape[1], hi.data_ptr(), lo.data_ptr(), x.shape[1], _lib.stream_ptr()))
    return hi, lo


def problem(m, n, k, form, seed):
    from chatts_amd.modeling import quantize_fp8_rows, quantize_int8_rows
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, w, bias, resid = 2 * r(m, k), (r(n, k) * k ** -0.5).bfloat16(), r(n), r(m, n)
    q = scale = None
    if form != "bf16":
        w[3] *= 40.0
        q, scale, w = (quantize_fp8_rows if form == "fp8" else quantize_int8_rows)(w)
    return x, w, bias, resid, q, scale


def args(m, n, k, hi, lo, w, q, scale, form, out, **kw):
    a = _lib.LinearArgs(w=w.data_ptr(), c=_lib.ptr(out), m=m, n=n, k=k, lda=k, ldw=k, a_hi=hi.data_ptr(), a_lo=lo.data_ptr(), ld_planes=k, **kw)
    if q is not None:
        a.w8, a.w8_scale, a.ldw8, a.w8_format = q.data_ptr(), scale.data_ptr(), k, _lib.W8_INT8 if form == "int8" else _lib.W8_FP8
    return a


def run(lib, a, m, n, k, chain=None):
    size = max(16, int(lib.chatts_linear_workspace(m, n, k)))
    ws = torch.empty(size, dtype=torch.uint8, device=DEV)
    a.workspace, a.workspace_bytes = ws.data_ptr(), size
    _lib.check(lib.chatts_linear(C.byref(a), _lib.stream_ptr()) if chain is None else lib.chatts_linear_chain(C.byref(a), C.byref(chain), _lib.stream_ptr()))
    torch.cuda.synchronize()


def rel(a, b):
    return float((a.double() - b).norm() / b.norm())


GLU = {_lib.EPI_SWIGLU, _lib.EPI_GEGLU, _lib.EPI_CLAMPGLU}


def reference(epi, z, resid):
    if epi in GLU:
        z = z.view(z.shape[0], -1, 2, 16)
        g, u = (z[:, :, i].reshape(z.shape[0], -1) for i in (0, 1))
        if epi == _lib.EPI_SWIGLU:
            return torch.nn.functional.silu(g) * u
        if epi == _lib.EPI_GEGLU:
            return torch.nn.functional.gelu(g, approximate="tanh") * u
        g, u = g.clamp(max=1.5), u.clamp(-1.5, 1.5)
        return g * torch.sigmoid(1.7 * g) * (u + 1)
    return {_lib.EPI_NONE: z, _lib.EPI_GELU: torch.nn.functional.gelu(z), _lib.EPI_RELU2: z.clamp(min=0) ** 2, _lib.EPI_RESID: resid.double() + z}[epi]


# columns that leave some workgroups a group more, fewer groups than CUs, 2 .. 16 waves; shapes on either side of the line to the split (test_every_size_of_a_workgroup
# has those that the few-rows kernel takes, and says so)
@pytest.mark.parametrize("form", ["bf16", "fp8", "int8"])
@pytest.mark.parametrize("m,n,k", [(2, 64, 1024), (8, 5120, 5120), (5, 4096, 1024), (7, 7168, 2048), (8, 5120, 13824), (7, 6160, 1152), (3, 10256, 640), (8, 16384, 512),
                                   (5, 14352, 512), (6, 2048, 4096), (4, 8192, 2176)])
@pytest.mark.parametrize("epi", [_lib.EPI_NONE, _lib.EPI_GELU, _lib.EPI_RESID, _lib.EPI_RELU2])
def test_columns(lib, form, m, n, k, epi):
    x, w, bias, resid, q, scale = problem(16, n, k, form, n + k)
    hi, lo = planes(lib, x)
    want = reference(epi, x.double() @ w.double().T + bias.double(), resid)
    more = dict(bias=bias.data_ptr(), ldc=n, epilogue=epi)
    out, all16 = (torch.full((r, n), float("nan"), device=DEV) for r in (m, 16))
    run(lib, args(m, n, k, hi, lo, w, q, scale, form, out, resid=resid.data_ptr(), **more), m, n, k)
    assert rel(out, want[:m]) < 1e-5                      # (x to 2^-17, sums in 32 bits: 3e-6 measured)
    run(lib, args(16, n, k, hi, lo, w, q, scale, form, all16, resid=resid.data_ptr(), **more), 16, n, k)
    assert torch.equal(out, all16[:m])
    if epi != _lib.EPI_RESID:                             # the same values as planes
        ph, pl = (torch.full((m, n + 8), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
        run(lib, args(m, n, k, hi, lo, w, q, scale, form, None, c_hi=ph.data_ptr(), c_lo=pl.data_ptr(), ld_cplanes=n + 8, **more), m, n, k)
        assert torch.equal(ph[:, :n], out.bfloat16()) and torch.equal(pl[:, :n], (out - out.bfloat16().float()).bfloat16()) and bool(ph[:, n:].isnan().all())


@pytest.mark.parametrize("form", ["bf16", "fp8"])
@pytest.mark.parametrize("m,n,k", [(8, 6144, 2048), (4, 96, 512), (7, 12288, 1024), (2, 5152, 1024)])
@pytest.mark.parametrize("epi", sorted(GLU))
def test_gated(lib, form, m, n, k, epi):
    x, w, bias, _, q, scale = problem(m, n, k, form, n + k)
    hi, lo = planes(lib, x)
    out = torch.full((m, n // 2), float("nan"), device=DEV)
    run(lib, args(m, n, k, hi, lo, w, q, scale, form, out, bias=bias.data_ptr(), ldc=n // 2, epilogue=epi, glu_limit=1.5, glu_alpha=1.7), m, n, k)
    assert rel(out, reference(epi, x.double() @ w.double().T + bias.double(), None)) < 1e-5


@pytest.mark.parametrize("form", ["bf16", "fp8"])
@pytest.mark.parametrize("m,h,k,n2", [(4, 5120, 5120, 7168), (8, 4096, 4096, 6144), (3, 1024, 2048, 512), (5, 4096, 4096, 24576), (2, 384, 1536, 4096), (8, 5184, 1024, 64)])
def test_norm_between_two_projections(lib, form, m, h, k, n2):
    """x += A W1 with sums of squares, then RMSNorm(x) W2 by the planes without the factor: against float64, in place, rows of very different size"""
    if form == "fp8" and h % 128:
        pytest.skip("8-bit weights take K in steps of 128")
    x, w1, _, resid, q1, s1 = problem(m, h, k, form, h)
    _, w2, _, _, q2, s2 = problem(m, n2, h, form, n2)
    resid *= 10.0 ** torch.linspace(-3, 3, m, device=DEV)[:, None]
    nw = 1 + 0.1 * torch.randn(h, device=DEV)
    hi, lo = planes(lib, x)
    new = resid.double() + x.double() @ w1.double().T
    want = (new * torch.rsqrt((new * new).mean(1, keepdim=True) + 1e-6) * nw.double()) @ w2.double().T
    ph, pl = (torch.empty((m, h), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ss = torch.full((16, 256), float("nan"), device=DEV)
    c = resid.clone()
    a = args(m, h, k, hi, lo, w1, q1, s1, form, c, resid=c.data_ptr(), ldc=h, epilogue=_lib.EPI_RESID, post_norm_w=nw.data_ptr(), post_hi=ph.data_ptr(),
             post_lo=pl.data_ptr(), ld_post=h)
    parts = int(lib.chatts_linear_post_ss_parts(C.byref(a)))
    assert 1 <= parts <= 256
    run(lib, a, m, h, k, _lib.NormChain(post_ss=ss.data_ptr()))
    assert rel(c, new) < 1e-5
    out = torch.full((m, n2), float("nan"), device=DEV)
    run(lib, args(m, n2, h, ph, pl, w2, q2, s2, form, out, ldc=n2, epilogue=_lib.EPI_NONE), m, n2, h,
        _lib.NormChain(row_ss=ss.data_ptr(), row_ss_parts=parts, row_eps=1e-6))
    for i in range(m):
        assert rel(out[i], want[i]) < 2e-5
    a.post_hi = hi.data_ptr()                             # planes that the same launch still reads
    assert int(lib.chatts_linear_post_ss_parts(C.byref(a))) == 0


@pytest.mark.parametrize("form", ["bf16", "fp8"])
@pytest.mark.parametrize("m", [2, 4, 8])
@pytest.mark.parametrize("as_planes", [True, False])
def test_a_result_in_the_place_of_its_own_input(lib, form, m, as_planes):
    n = k = 2048
    x, w, bias, _, q, scale = problem(m, n, k, form, m)
    hi, lo = planes(lib, x)
    want = x.double() @ w.double().T + bias.double()
    more = dict(c_hi=hi.data_ptr(), c_lo=lo.data_ptr(), ld_cplanes=n) if as_planes else {}
    a = args(m, n, k, hi, lo, w, q, scale, form, None if as_planes else hi, bias=bias.data_ptr(), ldc=n, epilogue=_lib.EPI_NONE, **more)      # (both planes lie in a row: m x n floats)
    run(lib, a, m, n, k)
    assert lo.data_ptr() == hi.data_ptr() + m * k * 2
    out = hi.double() + lo.double() if as_planes else torch.as_strided(hi, (m, 2 * n), (2 * n, 1)).view(torch.float32)
    assert rel(out, want) < 1e-5


# 8-row pieces of W a workgroup (1 .. 8; bf16 up to 6), K ranges of it; 8-bit with fewer ranges than fragments, so that a wave only helps to finish
@pytest.mark.parametrize("form,m,n,k,pieces,ranges", [
    ("bf16", 4, 1968, 4096, 1, 16), ("bf16", 8, 1040, 2304, 1, 9), ("bf16", 2, 2048, 2048, 1, 8), ("bf16", 6, 4112, 4096, 3, 8), ("bf16", 8, 4096, 4096, 2, 8), ("bf16", 8, 5120, 4096, 3, 6), ("bf16", 5, 7184, 2048, 4, 4),
    ("bf16", 3, 9232, 1536, 5, 4), ("bf16", 8, 10240, 2048, 5, 3), ("bf16", 7, 11280, 1024, 6, 3), ("bf16", 4, 12288, 2048, 6, 3),
    *((form, m, n, k, p, r) for form in ("fp8", "int8") for m, n, k, p, r in [(3, 1040, 2048, 1, 4), (8, 4096, 4096, 2, 8), (4, 4112, 2048, 3, 4), (2, 8192, 2048, 4, 4), (4, 10240, 4096, 5, 3), (3, 9232, 1536, 5, 3),
                                                                         (4, 11280, 1024, 6, 2), (2, 13328, 2048, 7, 2), (4, 14336, 1280, 7, 2), (4, 16384, 1152, 8, 2), (3, 15376, 4096, 8, 2)])])
@pytest.mark.parametrize("epi", [_lib.EPI_NONE, _lib.EPI_RESID])
def test_every_size_of_a_workgroup(lib, form, m, n, k, pieces, ranges, epi):
    x, w, bias, resid, q, scale = problem(16, n, k, form, n + k)
    hi, lo = planes(lib, x)
    want = x.double() @ w.double().T + bias.double() + (resid.double() if epi == _lib.EPI_RESID else 0)
    out, all16 = (torch.full((r, n), float("nan"), device=DEV) for r in (m, 16))
    more = dict(bias=bias.data_ptr(), ldc=n, epilogue=epi, resid=resid.data_ptr())
    a = args(m, n, k, hi, lo, w, q, scale, form, out, **more)
    assert (-(-(n // 4) // 256) * 4 + 7) // 8 == pieces and int(lib.chatts_linear_few_rows(C.byref(a), None)) == ranges
    run(lib, a, m, n, k)
    assert rel(out, want[:m]) < 1e-5                      # (x to 2^-17, sums in 32 bits: 3e-6 measured)
    run(lib, args(16, n, k, hi, lo, w, q, scale, form, all16, **more), 16, n, k)
    assert torch.equal(out, all16[:m])


# one fragment of gates and two, the last workgroups with a group less
@pytest.mark.parametrize("form,m,n,k,ranges", [("bf16", 8, 6144, 2048, 5), ("bf16", 4, 96, 512, 2), ("bf16", 5, 8192, 1024, 4), ("bf16", 3, 5152, 1024, 4),
                                               *((form, m, n, k, r) for form in ("fp8", "int8") for m, n, k, r in [(4, 96, 1024, 2), (2, 8192, 2048, 4), (4, 12288, 1024, 2), (3, 8224, 2048, 3), (4, 16384, 1024, 2)])])
@pytest.mark.parametrize("epi", sorted(GLU))
def test_gated_as_with_sixteen_rows(lib, form, m, n, k, ranges, epi):
    x, w, bias, _, q, scale = problem(16, n, k, form, n + k)
    hi, lo = planes(lib, x)
    got = []
    for rows in (m, 16):
        ph, pl = torch.full((2, rows, n // 2), float("nan"), dtype=torch.bfloat16, device=DEV)
        a = args(rows, n, k, hi, lo, w, q, scale, form, None, bias=bias.data_ptr(), ldc=n // 2, c_hi=ph.data_ptr(), c_lo=pl.data_ptr(), ld_cplanes=n // 2, epilogue=epi, glu_limit=1.5, glu_alpha=1.7)
        assert int(lib.chatts_linear_few_rows(C.byref(a), None)) == (ranges if rows == m else 0)
        run(lib, a, rows, n, k)
        got.append((ph[:m], pl[:m]))
    want = reference(epi, x.double() @ w.double().T + bias.double(), None)
    assert rel(got[0][0].double() + got[0][1].double(), want[:m]) < 1e-5
    assert all(torch.equal(a, b) for a, b in zip(*got))
