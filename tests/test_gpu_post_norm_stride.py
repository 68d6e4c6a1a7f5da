"""chatts_linear with post_norm_w where the rows of c lie further apart than N: the planes are the norm of c's rows whether the norm rides on an epilogue or is a launch
of its own, and what lies between the rows is neither read nor written."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


# split K (few rows, a stream with an epilogue, several row blocks) and K in one piece; strides of whole and of broken vectors
@pytest.mark.parametrize("epi", [_lib.EPI_NONE, _lib.EPI_RESID])
@pytest.mark.parametrize("m,n,k,gap", [(2, 5120, 5120, 64), (8, 4096, 4096, 64), (16, 4096, 4096, 64), (5, 384, 1536, 4), (2, 512, 64, 64), (8, 512, 64, 7), (16, 1040, 128, 64),
                                       (40, 3072, 2048, 64), (200, 512, 128, 64)])
def test_planes_are_the_norm_of_the_rows(m, n, k, gap, epi):
    lib = _lib.load()
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    x, w, nw, resid = r(m, k), (r(n, k) * k ** -0.5).bfloat16(), 1 + 0.1 * r(n), r(m, n)
    resid *= 10.0 ** torch.linspace(-2, 2, m, device=DEV)[:, None]
    hi, lo = torch.empty(2, m, k, dtype=torch.bfloat16, device=DEV)
    _lib.check(lib.chatts_split_bf16x2(x.data_ptr(), m, k, k, hi.data_ptr(), lo.data_ptr(), k, _lib.stream_ptr()))
    size = int(lib.chatts_linear_workspace(m, n, k))
    ws = torch.empty(max(size, 16), dtype=torch.uint8, device=DEV)
    got = []
    for ldc in (n, n + gap):
        c, add = torch.full((m, ldc), 1e6, device=DEV), torch.full((m, ldc), 1e6, device=DEV)
        add[:, :n] = resid
        ph, pl = torch.full((2, m, n), float("nan"), dtype=torch.bfloat16, device=DEV)
        a = _lib.LinearArgs(w=w.data_ptr(), c=c.data_ptr(), resid=add.data_ptr() if epi == _lib.EPI_RESID else None, m=m, n=n, k=k, lda=k, ldw=k, ldc=ldc, epilogue=epi,
                            workspace=ws.data_ptr(), workspace_bytes=size, a_hi=hi.data_ptr(), a_lo=lo.data_ptr(), ld_planes=k)
        a.post_norm_w, a.post_norm_eps, a.post_hi, a.post_lo, a.ld_post = nw.data_ptr(), 1e-6, ph.data_ptr(), pl.data_ptr(), n
        _lib.check(lib.chatts_linear(C.byref(a), _lib.stream_ptr()))
        torch.cuda.synchronize()
        assert bool((c[:, n:] == 1e6).all())
        want = c[:, :n].double()
        want = want * torch.rsqrt((want * want).mean(1, keepdim=True) + 1e-6) * nw.double()
        # two planes hold a value to 2^-17; the sum of squares takes n / 256 + 16 float32 roundings, the factor and the two products one or two each
        bound = want.abs() * (2.0 ** -17 + (n / 256 + 24) * 2.0 ** -24)
        assert bool(((ph.double() + pl.double() - want).abs() <= bound).all())
        got.append((c[:, :n].clone(), ph, pl))
    assert all(torch.equal(p, q) for p, q in zip(*got))
