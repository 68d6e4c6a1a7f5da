"""Five to eight slabs of a split K summed with all round trips at once == the row-walking epilogue bit for bit (rows that end inside a thread's columns, one to
five column groups, scratch of exactly the stated size), and several row blocks on the weight stream against float64 sums where the split is capped to one workgroup per CU."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


def run(m, n, k, epi, resid, nw, x, w, alias=False):
    lib = _lib.load()
    hi, lo = torch.empty(2, m, k, dtype=torch.bfloat16, device=DEV)
    _lib.check(lib.chatts_split_bf16x2(x.data_ptr(), m, k, k, hi.data_ptr(), lo.data_ptr(), k, _lib.stream_ptr()))
    out = resid.clone() if alias else torch.full((m, n), float("nan"), device=DEV)
    ph, pl = torch.full((2, m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
    size = int(lib.chatts_linear_workspace(m, n, k))
    ws = torch.empty(max(size, 16), dtype=torch.uint8, device=DEV)
    a = _lib.LinearArgs(w=w.data_ptr(), c=out.data_ptr(), resid=(out if alias else resid).data_ptr() if epi == _lib.EPI_RESID else None, m=m, n=n, k=k, lda=k, ldw=k, ldc=n, epilogue=epi,
                        workspace=ws.data_ptr(), workspace_bytes=size, a_hi=hi.data_ptr(), a_lo=lo.data_ptr(), ld_planes=k)
    if nw is not None:
        a.post_norm_w, a.post_norm_eps, a.post_hi, a.post_lo, a.ld_post = nw.data_ptr(), 1e-6, ph.data_ptr(), pl.data_ptr(), n
    _lib.check(lib.chatts_linear(C.byref(a), _lib.stream_ptr()))
    torch.cuda.synchronize()
    return out, ph, pl


def problem(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    return r(m, k), (r(n, k) * k ** -0.5).bfloat16(), r(m, n), 1 + 0.1 * r(n)


@pytest.mark.parametrize("sk", [5, 6, 7, 8])
@pytest.mark.parametrize("m,n,k,epi,alias", [(100, 4096, 4096, _lib.EPI_RESID, True), (223, 5120, 2048, _lib.EPI_RESID, False), (131, 2080, 2048, _lib.EPI_NONE, False),
                                             (17, 1008, 2048, _lib.EPI_RESID, False), (40, 3072, 2048, _lib.EPI_RESID, True)])
def test_all_round_trips_at_once(monkeypatch, sk, m, n, k, epi, alias):
    x, w, resid, nw = problem(m, n, k)
    monkeypatch.setenv("CHATTS_GEMM_SK", str(sk))
    got = []
    for reg in ("0", "1"):
        monkeypatch.setenv("CHATTS_EPI_NORM_REG", reg)
        got.append(run(m, n, k, epi, resid, nw, x, w, alias))
    assert all(torch.equal(a, b) and torch.isfinite(a.float()).all() for a, b in zip(*got))


@pytest.mark.parametrize("m", [17, 32, 33, 64, 65, 128])
def test_row_blocks_with_a_capped_split(m):
    n, k = 7168, 5120
    x, w, resid, _ = problem(m, n, k)
    out = run(m, n, k, _lib.EPI_NONE, resid, None, x, w)[0].double()
    # x = hi + lo loses 2^-18 of a term; at most K / 16 + 8 float32 additions of 2^-24 each
    xd, wd = x.double(), w.double()
    bound = xd.abs() @ wd.abs().T * (2.0 ** -18 + (k / 16 + 8) * 2.0 ** -24)
    assert bool(((out - xd @ wd.T).abs() <= bound).all())
