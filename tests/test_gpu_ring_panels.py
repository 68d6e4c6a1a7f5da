"""The prefill kernel with panels of 192 rows of W == with panels of 256 bit for bit: every epilogue, gated ones with their fragments of 8 gates and 8 up rows, N that ends
inside a panel, direct stores and slabs, tiled and row-major W, one to ten fragments of M."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"
GATED = (_lib.EPI_SWIGLU, _lib.EPI_GEGLU, _lib.EPI_CLAMPGLU)


@pytest.mark.parametrize("planes,tiled", [(False, False), (True, True), (True, False)])
@pytest.mark.parametrize("epi", [_lib.EPI_NONE, _lib.EPI_GELU, _lib.EPI_RESID, _lib.EPI_RELU2, *GATED])
@pytest.mark.parametrize("m,n,k,sk,t", [(97, 384, 256, 1, 1), (223, 1024, 512, 1, 2), (223, 800, 512, 2, 2), (130, 32, 192, 1, 3), (640, 2080, 128, 1, 4), (300, 6144, 320, 0, 0)])
def test_panels_agree(monkeypatch, m, n, k, sk, t, epi, planes, tiled):
    lib = _lib.load()
    g = torch.Generator(device=DEV).manual_seed(m + n)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, w, bias, resid = r(m, k), (r(n, k) * k ** -0.5).bfloat16(), r(n), r(m, n)
    hi, lo = torch.empty(2, m, k, dtype=torch.bfloat16, device=DEV)
    _lib.check(lib.chatts_split_bf16x2(x.data_ptr(), m, k, k, hi.data_ptr(), lo.data_ptr(), k, _lib.stream_ptr()))
    wt = torch.empty(int(lib.chatts_tile_bf16_elems(n, k)), dtype=torch.bfloat16, device=DEV)
    _lib.check(lib.chatts_tile_bf16(w.data_ptr(), n, k, k, wt.data_ptr(), _lib.stream_ptr()))
    cols = n // 2 if epi in GATED else n
    if sk:
        monkeypatch.setenv("CHATTS_GEMM_SK", str(sk))
        monkeypatch.setenv("CHATTS_GEMM_T", str(t))
    monkeypatch.setenv("CHATTS_GEMM_STREAM", "0")
    got = []
    for panel in (256, 192):
        monkeypatch.setenv("CHATTS_GEMM_PANEL", str(panel))
        size = max(16, int(lib.chatts_linear_workspace(m, n, k)))
        ws = torch.empty(size, dtype=torch.uint8, device=DEV)
        out = torch.full((m, cols), float("nan"), device=DEV)
        ph, pl = torch.full((2, m, cols), float("nan"), dtype=torch.bfloat16, device=DEV)
        a = _lib.LinearArgs(w=w.data_ptr(), bias=bias.data_ptr(), resid=resid.data_ptr() if epi == _lib.EPI_RESID else None, m=m, n=n, k=k, lda=k, ldw=k, ldc=cols, epilogue=epi,
                            workspace=ws.data_ptr(), workspace_bytes=size, a_hi=hi.data_ptr(), a_lo=lo.data_ptr(), ld_planes=k, glu_limit=7.0, glu_alpha=1.702)
        if planes:
            a.c_hi, a.c_lo, a.ld_cplanes = ph.data_ptr(), pl.data_ptr(), cols
        else:
            a.c = out.data_ptr()
        if tiled:
            a.w_tiled = wt.data_ptr()
        _lib.check(lib.chatts_linear(C.byref(a), _lib.stream_ptr()))
        torch.cuda.synchronize()
        got.append((ph, pl) if planes else (out,))
    if sk == 0:      # (each panel picks its own tiles and splits: the K order may differ)
        for p, q in zip(*got):
            assert torch.isfinite(p.float()).all()
        total = lambda v: sum(z.double() for z in v)
        # a sum of K terms in another order moves by at most 2 K float32 roundings of terms whose magnitudes add up to ~sqrt(K) * |row| / sqrt(K); planes hold 2^-17 of it
        assert float((total(got[0]) - total(got[1])).abs().max()) <= 2 * k * 2.0 ** -24 * 16 + float(total(got[0]).abs().max()) * 2.0 ** -16
        return
    for p, q in zip(*got):
        assert torch.isfinite(p.float()).all() and torch.equal(p, q)


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("m,n,k,sk,t", [(5, 64, 64, 1, 1), (17, 384, 64, 1, 1), (97, 400, 64, 1, 1), (160, 1024, 64, 1, 1), (223, 1024, 128, 2, 2), (145, 800, 64, 1, 1)])
def test_two_half_steps(m, n, k, sk, t, tiled):
    """the fewest that a workgroup walks: its loaders never come to their loop's wait (one unit a workgroup, one to ten fragments, tiles of unequal length)"""
    lib = _lib.load()
    g = torch.Generator(device=DEV).manual_seed(m + n)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, w, bias = r(m, k), (r(n, k) * k ** -0.5).bfloat16(), r(n)
    hi, lo = torch.empty(2, m, k, dtype=torch.bfloat16, device=DEV)
    _lib.check(lib.chatts_split_bf16x2(x.data_ptr(), m, k, k, hi.data_ptr(), lo.data_ptr(), k, _lib.stream_ptr()))
    wt = torch.empty(int(lib.chatts_tile_bf16_elems(n, k)), dtype=torch.bfloat16, device=DEV)
    _lib.check(lib.chatts_tile_bf16(w.data_ptr(), n, k, k, wt.data_ptr(), _lib.stream_ptr()))
    want = x.double() @ w.double().T + bias.double()
    # x = hi + lo loses 2^-18 of each term; float32 sums of K terms and the bias
    bound = x.double().abs() @ w.double().abs().T * (2.0 ** -18 + (k + 2) * 2.0 ** -24) + want.abs() * 2.0 ** -24
    for panel in (256, 192):
        with _lib.options(GEMM_SK=sk, GEMM_T=t, GEMM_STREAM=0, GEMM_PANEL=panel):
            size = max(16, int(lib.chatts_linear_workspace(m, n, k)))
            ws, out = torch.empty(size, dtype=torch.uint8, device=DEV), torch.full((m, n), float("nan"), device=DEV)
            a = _lib.LinearArgs(w=w.data_ptr(), bias=bias.data_ptr(), c=out.data_ptr(), m=m, n=n, k=k, lda=k, ldw=k, ldc=n, epilogue=_lib.EPI_NONE, workspace=ws.data_ptr(), workspace_bytes=size,
                                a_hi=hi.data_ptr(), a_lo=lo.data_ptr(), ld_planes=k)
            if tiled:
                a.w_tiled = wt.data_ptr()
            _lib.check(lib.chatts_linear(C.byref(a), _lib.stream_ptr()))
            torch.cuda.synchronize()
        assert bool(((out.double() - want).abs() <= bound).all()), panel
