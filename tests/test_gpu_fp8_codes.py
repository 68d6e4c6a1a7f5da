"""Few rows on fp8 weights: every finite code arrives as the number it stands for, bit for bit, and both codes of no number as none, in each kernel that widens them (csrc/gemm_rows.hip,
gemm_cols.hip, gemm.hip)."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(autouse=True)
def own_random_numbers():
    """the tests behind these draw what they would draw without them"""
    with torch.random.fork_rng():
        yield


@pytest.mark.parametrize("m", [2, 16])
@pytest.mark.parametrize("n,k", [(256, 256), (5120, 5120), (24576, 4096)])
def test_every_code(n, k, m):
    lib = _lib.load()
    codes = ((torch.arange(n, device=DEV)[:, None] * 3 + torch.arange(k, device=DEV)[None]) % 256).to(torch.uint8)
    codes[(codes & 0x7f) == 0x7f] = 0                              # (no number)
    codes[5, 3], codes[n - 1, k - 1] = 0x7f, 0xff
    scale = 2.0 ** (torch.arange(n, device=DEV) % 7 - 3).float()
    w = codes.view(torch.float8_e4m3fn).float() * scale[:, None]
    deq = w.bfloat16()
    hi, lo, out = torch.zeros((m, k), dtype=torch.bfloat16, device=DEV), torch.zeros((m, k), dtype=torch.bfloat16, device=DEV), torch.full((m, n), float("nan"), device=DEV)
    at = [j * (k // m) + j for j in range(m)]
    for j, c in enumerate(at):
        hi[j, c] = 1.0
    size = int(lib.chatts_linear_workspace(m, n, k))
    ws = torch.empty(max(size, 16), dtype=torch.uint8, device=DEV)
    a = _lib.LinearArgs(w=deq.data_ptr(), c=out.data_ptr(), m=m, n=n, k=k, lda=k, ldw=k, ldc=n, epilogue=_lib.EPI_NONE, workspace=ws.data_ptr(), workspace_bytes=size, w8=codes.data_ptr(),
                        w8_scale=scale.data_ptr(), ldw8=k, a_hi=hi.data_ptr(), a_lo=lo.data_ptr(), ld_planes=k)
    _lib.check(lib.chatts_linear(C.byref(a), _lib.stream_ptr()))
    torch.cuda.synchronize()
    rows = [5, n - 1]                                              # (nothing times no number is none, too)
    assert bool(torch.isnan(out[:, rows]).all())
    finite = torch.ones(n, dtype=torch.bool, device=DEV)
    finite[rows] = False
    assert torch.equal(out[:, finite], w[:, at].T[:, finite])
