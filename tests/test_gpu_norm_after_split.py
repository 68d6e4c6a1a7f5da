"""The RMSNorm between two projections of few rows where K of the first is split over workgroups (splitk_epilogue_ss_kernel): c bit for bit what the call without
the norm gives, and the second projection against float64; parts of unequal length, in place, rows of very different size; and the bits of
a row do not depend on the number of rows, whichever kernel runs."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib
from tests.test_gpu_rows import DEV, args, planes, problem, rel, run

pytestmark = pytest.mark.gpu


@pytest.fixture()
def lib():
    return _lib.load()


@pytest.mark.parametrize("form", ["bf16", "fp8", "int8"])
@pytest.mark.parametrize("m,h,k,n2", [(9, 5120, 5120, 7168), (16, 4096, 4096, 6144), (12, 1152, 2048, 512), (16, 5120, 13824, 27648), (6, 5120, 5120, 7168), (16, 384, 1536, 4096)])
def test_norm_after_a_split(lib, form, m, h, k, n2):
    x, w1, _, resid, q1, s1 = problem(m, h, k, form, h)
    _, w2, _, _, q2, s2 = problem(m, n2, h, form, n2)
    resid *= 10.0 ** torch.linspace(-3, 3, m, device=DEV)[:, None]
    nw = 1 + 0.1 * torch.randn(h, generator=torch.Generator(device=DEV).manual_seed(m + h), device=DEV)
    hi, lo = planes(lib, x)
    new = resid.double() + x.double() @ w1.double().T
    normed = new * torch.rsqrt((new * new).mean(1, keepdim=True) + 1e-6) * nw.double()
    want = normed @ w2.double().T
    plain = torch.empty_like(resid)
    run(lib, args(m, h, k, hi, lo, w1, q1, s1, form, plain, resid=resid.data_ptr(), ldc=h, epilogue=_lib.EPI_RESID), m, h, k)
    ph, pl = (torch.empty((m, h), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ss = torch.full((16, 256), float("nan"), device=DEV)
    c = resid.clone()
    a = args(m, h, k, hi, lo, w1, q1, s1, form, c, resid=c.data_ptr(), ldc=h, epilogue=_lib.EPI_RESID, post_norm_w=nw.data_ptr(), post_hi=ph.data_ptr(), post_lo=pl.data_ptr(), ld_post=h)
    parts = int(lib.chatts_linear_post_ss_parts(C.byref(a)))
    assert 1 <= parts <= 256
    run(lib, a, m, h, k, _lib.NormChain(post_ss=ss.data_ptr()))
    assert torch.equal(c, plain) and bool((rel(c, new) < 1e-5))
    prod = c * nw
    assert torch.equal(ph, prod.bfloat16()) and torch.equal(pl, (prod - prod.bfloat16().float()).bfloat16())
    # positive float32 terms: a rounding for each of the 4 columns, 2 across lanes, one a step of 16 columns
    assert bool(((ss[:m, :parts].double().sum(1) / (c.double() ** 2).sum(1) - 1).abs() < (6 + h / 16 / parts + 1) * 2.0 ** -24).all())
    out = torch.full((m, n2), float("nan"), device=DEV)
    run(lib, args(m, n2, h, ph, pl, w2, q2, s2, form, out, ldc=n2, epilogue=_lib.EPI_NONE), m, n2, h, _lib.NormChain(row_ss=ss.data_ptr(), row_ss_parts=parts, row_eps=1e-6))
    # Two splits into two parts, each to 2^-18 of a value, the first halfway hidden behind resid; sums in 32 bits.  They are measured against the size that the terms' squares give, not that of the
    # result: 8-bit weights have one column of forty times the others' size, and where its terms happen to cancel, the result is small and the errors are not.
    size = (normed ** 2 @ (w2.double() ** 2).T).sum(1).sqrt()
    assert bool(((out.double() - want).norm(dim=1) < 2e-5 * size).all())


@pytest.mark.parametrize("form,few", [("bf16", 8), ("bf16", 3), ("fp8", 4), ("int8", 2)])
@pytest.mark.parametrize("h,k", [(5120, 5120), (4096, 4096), (1152, 2048)])
def test_a_row_does_not_depend_on_the_number_of_rows(lib, form, few, h, k):
    x, w, _, resid, q, s = problem(16, h, k, form, h)
    nw = 1 + 0.1 * torch.randn(h, generator=torch.Generator(device=DEV).manual_seed(h), device=DEV)
    got = []
    for m in (16, few):
        hi, lo = planes(lib, x[:m].contiguous())
        ph, pl = (torch.empty((m, h), dtype=torch.bfloat16, device=DEV) for _ in range(2))
        ss, c = torch.zeros((16, 256), device=DEV), resid[:m].clone()
        a = args(m, h, k, hi, lo, w, q, s, form, c, resid=c.data_ptr(), ldc=h, epilogue=_lib.EPI_RESID, post_norm_w=nw.data_ptr(), post_hi=ph.data_ptr(), post_lo=pl.data_ptr(), ld_post=h)
        run(lib, a, m, h, k, _lib.NormChain(post_ss=ss.data_ptr()))
        got.append((c[:few], ph[:few], pl[:few], ss[:few]))
    assert all(torch.equal(a, b) for a, b in zip(*got))


# consumers with K in ranges (qkv, with a bias), in one piece (gate_up, the head), gated with K in ranges; the few-rows kernel beside the stream
@pytest.mark.parametrize("form,few", [("bf16", 8), ("bf16", 3), ("fp8", 4), ("int8", 2)])
@pytest.mark.parametrize("n,k,epi", [(6144, 4096, _lib.EPI_NONE), (7168, 5120, _lib.EPI_NONE), (24576, 4096, _lib.EPI_SWIGLU), (2048, 2048, _lib.EPI_SWIGLU), (1152, 2048, _lib.EPI_RESID)])
def test_a_product_behind_the_norm_does_not_depend_on_the_number_of_rows(lib, form, few, n, k, epi):
    x, w, bias, resid, q, s = problem(16, n, k, form, n + k)
    x *= 10.0 ** torch.linspace(-2, 2, 16, device=DEV)[:, None]
    ss = torch.full((16, 256), float("nan"), device=DEV)
    ss[:, :200] = (x.double() ** 2).reshape(16, 64, -1).sum(2).float().repeat_interleave(4, 1)[:, :200] / 4      # (parts of any kind; what lies behind the last one is not read)
    rstd = torch.rsqrt(ss[:, :200].double().sum(1, keepdim=True) / k + 1e-6)
    z = (x.double() @ w.double().T) * rstd + bias.double()
    gated = epi == _lib.EPI_SWIGLU
    if gated:
        z = z.view(16, -1, 2, 16)
        want = (torch.nn.functional.silu(z[:, :, 0]) * z[:, :, 1]).reshape(16, n // 2)
    else:
        want = z + resid.double() if epi == _lib.EPI_RESID else z
    got = []
    for m in (16, few):
        hi, lo = planes(lib, x[:m].contiguous())
        chain = _lib.NormChain(row_ss=ss.data_ptr(), row_ss_parts=200, row_eps=1e-6)
        cols = n // 2 if gated else n
        if gated:                                         # (what the decoder's gate_up writes)
            ph, pl = torch.full((2, m, cols), float("nan"), dtype=torch.bfloat16, device=DEV)
            run(lib, args(m, n, k, hi, lo, w, q, s, form, None, bias=bias.data_ptr(), epilogue=epi, c_hi=ph.data_ptr(), c_lo=pl.data_ptr(), ld_cplanes=cols, ldc=cols), m, n, k, chain)
            got.append((ph[:few], pl[:few]))
            out = ph.double() + pl.double()
        else:
            out = torch.full((m, n), float("nan"), device=DEV)
            run(lib, args(m, n, k, hi, lo, w, q, s, form, out, bias=bias.data_ptr(), resid=resid.data_ptr(), ldc=n, epilogue=epi), m, n, k, chain)
            got.append((out[:few],))
        for i in range(m):
            assert rel(out[i], want[i]) < 2e-5            # (x to 2^-17, sums in 32 bits)
    assert all(torch.equal(a, b) for a, b in zip(*got))
