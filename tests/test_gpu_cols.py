"""Wide projections of 2 .. 16 rows (csrc/gemm_cols.hip) against float64 on the stored weights, and a row's bits for any number of rows: shares of the columns that differ by a group,
one panel and several, fewer K-steps than waves, every weight format and epilogue, a norm's factors on the rows; and which calls come here."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib
from .test_gpu_rows import DEV, GLU, args, planes, problem, reference, rel, run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


@pytest.fixture()
def everywhere():
    with _lib.options(GEMM_COLS=2):                       # (small shapes, too)
        yield


# groups of 4 columns of a workgroup: 1, 3 / 2, 8, 17 / 16, 24, 25 / 24, 33 / 32 (two panels), 65 / 64 (three, unequal)
@pytest.mark.parametrize("form", ["bf16", "fp8", "int8"])
@pytest.mark.parametrize("n,k", [(64, 128), (2064, 256), (8192, 384), (16400, 640), (24576, 1152), (24592, 256), (32784, 640), (65552, 256)])
@pytest.mark.parametrize("epi", [_lib.EPI_NONE, _lib.EPI_GELU, _lib.EPI_RESID, _lib.EPI_RELU2])
def test_columns(lib, everywhere, form, n, k, epi):
    x, w, bias, resid, q, scale = problem(16, n, k, form, n + k)
    hi, lo = planes(lib, x)
    want = reference(epi, x.double() @ w.double().T + bias.double(), resid)
    out = {}
    for m in (2, 8, 9, 16):
        out[m] = torch.full((m, n), float("nan"), device=DEV)
        run(lib, args(m, n, k, hi, lo, w, q, scale, form, out[m], resid=resid.data_ptr(), bias=bias.data_ptr(), ldc=n, epilogue=epi), m, n, k)
        assert torch.equal(out[m], out[2][:m] if m == 2 else torch.cat([out[2], out[m][2:]])), m
    assert rel(out[16], want) < 1e-5                      # (x to 2^-17, sums in 32 bits: 3e-6 measured)
    assert all(torch.equal(out[m], out[16][:m]) for m in (8, 9))
    if epi == _lib.EPI_RESID:                             # in place
        c = resid.clone()
        run(lib, args(16, n, k, hi, lo, w, q, scale, form, c, resid=c.data_ptr(), bias=bias.data_ptr(), ldc=n, epilogue=epi), 16, n, k)
        assert torch.equal(c, out[16])


# groups of 4 gates: 1, 5 / 4, 8, 12, 13 / 12, 17 / 16 (two panels), 33 / 32 (three)
@pytest.mark.parametrize("form", ["bf16", "fp8", "int8"])
@pytest.mark.parametrize("n,k", [(64, 128), (8224, 384), (16384, 256), (24576, 640), (24608, 256), (32800, 1152), (65568, 256)])
@pytest.mark.parametrize("epi", sorted(GLU))
def test_gated(lib, everywhere, form, n, k, epi):
    x, w, bias, _, q, scale = problem(16, n, k, form, n + k)
    hi, lo = planes(lib, x)
    want = reference(epi, x.double() @ w.double().T + bias.double(), None)
    got = {}
    for m in (3, 8, 11, 16):
        ph, pl = torch.full((2, m, n // 2 + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
        run(lib, args(m, n, k, hi, lo, w, q, scale, form, None, bias=bias.data_ptr(), ldc=n // 2, c_hi=ph.data_ptr(), c_lo=pl.data_ptr(), ld_cplanes=n // 2 + 8, epilogue=epi, glu_limit=1.5,
                      glu_alpha=1.7), m, n, k)
        assert bool(ph[:, n // 2:].isnan().all())
        got[m] = (ph[:, :n // 2], pl[:, :n // 2])
    assert rel(got[16][0].double() + got[16][1].double(), want) < 1e-5
    assert all(torch.equal(a, b[:m]) for m in got for a, b in zip(got[m], got[16]))
    out = torch.full((16, n // 2), float("nan"), device=DEV)
    run(lib, args(16, n, k, hi, lo, w, q, scale, form, out, bias=bias.data_ptr(), ldc=n // 2, epilogue=epi, glu_limit=1.5, glu_alpha=1.7), 16, n, k)
    assert torch.equal(got[16][0], out.bfloat16()) and torch.equal(got[16][1], (out - out.bfloat16().float()).bfloat16())


@pytest.mark.parametrize("form", ["bf16", "fp8"])
@pytest.mark.parametrize("m", [2, 8, 16])
@pytest.mark.parametrize("n", [24576, 65552])
def test_the_factor_of_a_norm(lib, everywhere, form, m, n):
    k = 512
    x, w, _, _, q, scale = problem(m, n, k, form, m)
    x *= 10.0 ** torch.linspace(-2, 2, m, device=DEV)[:, None]
    hi, lo = planes(lib, x)
    ss = torch.full((16, 256), float("nan"), device=DEV)
    ss[:m, :4] = (x * x).view(m, 4, -1).sum(2)
    out = torch.full((m, n), float("nan"), device=DEV)
    run(lib, args(m, n, k, hi, lo, w, q, scale, form, out, ldc=n, epilogue=_lib.EPI_NONE), m, n, k, _lib.NormChain(row_ss=ss.data_ptr(), row_ss_parts=4, row_eps=1e-6))
    d = x.double()
    want = (d * torch.rsqrt((d * d).mean(1, keepdim=True) + 1e-6)) @ w.double().T
    assert all(rel(out[i], want[i]) < 2e-5 for i in range(m))


def test_strides_and_calls_that_stay_out(lib):
    """rows of W and A further apart than K; results at a stride; results that do not start on 16 bytes, or in A's place, take another kernel and agree"""
    m, n, k = 5, 24576, 512
    x, w, bias, _, _, _ = problem(m, n, k, "bf16", 7)
    want = x.double() @ w.double().T + bias.double()
    wide = torch.full((n, k + 64), float("nan"), dtype=torch.bfloat16, device=DEV)
    wide[:, :k] = w
    hi, lo = planes(lib, x)
    far = torch.full((2, m, k + 32), float("nan"), dtype=torch.bfloat16, device=DEV)
    far[0, :, :k], far[1, :, :k] = hi, lo
    out = torch.full((m, n + 4), float("nan"), device=DEV)
    a = args(m, n, k, hi, lo, w, None, None, "bf16", out, bias=bias.data_ptr(), ldc=n + 4, epilogue=_lib.EPI_NONE)
    a.w, a.ldw, a.a_hi, a.a_lo, a.ld_planes = wide.data_ptr(), k + 64, far[0].data_ptr(), far[1].data_ptr(), k + 32
    run(lib, a, m, n, k)
    assert rel(out[:, :n], want) < 1e-5 and bool(out[:, n:].isnan().all())
    odd = torch.full((m, n + 1), float("nan"), device=DEV)
    run(lib, args(m, n, k, hi, lo, w, None, None, "bf16", odd, bias=bias.data_ptr(), ldc=n + 1, epilogue=_lib.EPI_NONE), m, n, k)
    assert rel(odd[:, :n], want) < 1e-5


@pytest.mark.parametrize("form,n", [("fp8", 229376), ("fp8", 229392), ("int8", 262144)])
def test_the_widest(lib, form, n):
    """scales and biases of as many columns a workgroup as its LDS holds; of one group more, and of the most: the kernel that runs there without a limit"""
    m, k = 16, 256
    x, w, bias, _, q, scale = problem(m, n, k, form, n)
    hi, lo = planes(lib, x)
    out = torch.full((m, n), float("nan"), device=DEV)
    with _lib.options(GEMM_COLS=2):
        run(lib, args(m, n, k, hi, lo, w, q, scale, form, out, bias=bias.data_ptr(), ldc=n, epilogue=_lib.EPI_NONE), m, n, k)
    assert rel(out, x.double() @ w.double().T + bias.double()) < 1e-5
