"""The batch-1 projection on 4-bit codes (csrc/gemv4.hip): every weight it rebuilds is the stored bf16 value bit for bit, sums against float64; rows that deal
unevenly over the CUs, K that ends inside a unit of 512, all group sizes it takes, gated rows, the fused norm."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


def problem(n, k, group, seed):
    from chatts_amd.modeling import pack_int4, quantize_int4_rows
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    w = (r(n, k) * k ** -0.5 * 10.0 ** (3 * torch.rand((n, 1), generator=g, device=DEV) - 2)).bfloat16()
    codes, scale, zero, deq = quantize_int4_rows(w, group)
    return r(1, k), pack_int4(codes, scale, zero), deq, r(n), r(1, n), 1 + 0.1 * r(k)


def run(x, w4, sz, deq, group, epi, bias=None, resid=None, norm=None):
    n, k = deq.shape
    out = torch.full((1, n // 2 if epi == _lib.EPI_SWIGLU else n), float("nan"), device=DEV)
    a = _lib.LinearArgs(a=x.data_ptr(), w=deq.data_ptr(), bias=_lib.ptr(bias), resid=_lib.ptr(resid), c=out.data_ptr(), norm_w=_lib.ptr(norm), norm_eps=1e-6, m=1, n=n, k=k,
                        lda=k, ldw=k, ldc=out.shape[1], epilogue=epi, w4=w4.data_ptr(), w4_sz=sz.data_ptr(), ldw4=k // 2, w4_group=group)
    _lib.check(_lib.load().chatts_linear(C.byref(a), _lib.stream_ptr()))
    torch.cuda.synchronize()
    return out


# the smallest of K, of N, of both; K that ends inside a unit; a row of units for some workgroups only; the largest K; both sides of the line to the old kernel
SHAPES = [(16, 2560, 128), (16, 2080, 32), (1040, 2112, 64), (5120, 5120, 128), (7168, 5120, 128), (96, 13824, 128), (13200, 640, 64), (98304, 96, 32), (4096, 12288, 64),
          (320, 16384, 128), (4096, 2048, 1024), (4112, 2048, 1024), (32, 4096, 256), (48, 96, 32), (1040, 1024, 32),
          (16, 3584, 128), (16, 3104, 32), (1040, 3136, 64), (6144, 2048, 1024), (6160, 2048, 1024), (4096, 2560, 64), (4112, 2560, 64), (2064, 3072, 32)]


@pytest.mark.parametrize("n,k,group", SHAPES)
def test_rebuilt_weights_are_the_stored_ones(n, k, group):
    _, (w4, sz), deq, *_ = problem(n, k, group, n + k)
    for at in [0, 1, 4, 7, 31, 32, k // 2 + 5, k - 1]:
        x = torch.zeros((1, k), device=DEV)
        x[0, at] = 1.0
        assert torch.equal(run(x, w4, sz, deq, group, _lib.EPI_NONE)[0], deq[:, at].float())


@pytest.mark.parametrize("epi", [_lib.EPI_NONE, _lib.EPI_RESID, _lib.EPI_SWIGLU])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("n,k,group", SHAPES + [(27648, 5120, 128)])
def test_sums(n, k, group, norm, epi):
    if epi == _lib.EPI_SWIGLU and n % 32:
        n += 16
    x, (w4, sz), deq, bias, resid, nw = problem(n, k, group, n * k)
    xd = x.double()
    if norm:
        xd = xd * torch.rsqrt((xd * xd).mean() + 1e-6) * nw.double()
    want = xd @ deq.double().T + bias.double()
    # x = hi + lo loses 2^-18 of each term; float32 sums of K / 16 terms a lane and 16 more: 2^-24 a step, at most (K / 16 + 32) of them
    bound = xd.abs() @ deq.double().abs().T * (2.0 ** -18 + (k / 16 + 32) * 2.0 ** -24) + want.abs() * 2.0 ** -20
    if epi == _lib.EPI_RESID:
        want = want + resid.double()
        bound = bound + want.abs() * 2.0 ** -24
    if epi == _lib.EPI_SWIGLU:
        z, dz = want.view(-1, 2, 16), bound.view(-1, 2, 16)
        gate = torch.nn.functional.silu(z[:, 0])
        want = (gate * z[:, 1]).reshape(1, -1)
        bound = (1.1 * dz[:, 0] * (z[:, 1].abs() + dz[:, 1]) + gate.abs() * dz[:, 1]).reshape(1, -1) + want.abs() * 2.0 ** -20      # (silu's slope is below 1.1)
    out = run(x, w4, sz, deq, group, epi, bias, resid, nw if norm else None)
    assert bool(((out.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("k", [2592, 2560, 5088, 3616, 3584])
def test_rows_do_not_read_each_other(k):
    x, (w4, sz), deq, *_ = problem(128, k, 32, k)
    clean = run(x, w4, sz, deq, 32, _lib.EPI_NONE)
    sz = sz.clone()
    sz[1::2] = float("nan")
    assert torch.equal(run(x, w4, sz, deq, 32, _lib.EPI_NONE)[:, ::2], clean[:, ::2])


@pytest.mark.parametrize("at", [0, 1])                # the first columns of a wider matrix, and the last ones: the last row ends where the memory ends
@pytest.mark.parametrize("k,group", [(2592, 32), (3104, 32), (4096 + 64, 64), (5088, 32), (5120, 128)])
def test_columns_of_a_wider_matrix(at, k, group):
    n = 96
    x, (w4, sz), deq, *_ = problem(n, k, group, k)
    want = run(x, w4, sz, deq, group, _lib.EPI_NONE)
    wide = torch.full((n, k), 0xff, dtype=torch.uint8, device=DEV)
    part = wide[:, k // 2 * at:][:, :k // 2]
    part.copy_(w4)
    out = torch.full((1, n), float("nan"), device=DEV)
    a = _lib.LinearArgs(a=x.data_ptr(), w=deq.data_ptr(), c=out.data_ptr(), m=1, n=n, k=k, lda=k, ldw=k, ldc=n, epilogue=_lib.EPI_NONE, w4=part.data_ptr(), w4_sz=sz.data_ptr(), ldw4=k,
                        w4_group=group)
    _lib.check(_lib.load().chatts_linear(C.byref(a), _lib.stream_ptr()))
    torch.cuda.synchronize()
    assert torch.equal(out, want)


@pytest.mark.parametrize("power", [-140, -100, 100, 103, 104, 110, 120])
def test_scales_of_any_size(power):
    n, k, group = 96, 4096 + 96, 32
    x, _, _, *_ = problem(n, k, group, power)
    g = torch.Generator(device=DEV).manual_seed(power)
    from chatts_amd.modeling import pack_int4
    codes = torch.randint(0, 16, (n, k), generator=g, device=DEV, dtype=torch.uint8)
    scale = (1 + torch.rand((n, k // group), generator=g, device=DEV)) * 2.0 ** -6
    scale[5::7, 3::11] = 1.5 * 2.0 ** power               # in some groups only: the others' weights must not suffer
    zero = torch.randint(0, 16, scale.shape, generator=g, device=DEV).float()
    deq = (codes.float() * scale.repeat_interleave(group, 1) - (scale * zero).repeat_interleave(group, 1)).bfloat16()
    w4, sz = pack_int4(codes, scale, zero)
    x = x * 2.0 ** min(0, 60 - power)                     # sums stay finite
    out = run(x, w4, sz, deq, group, _lib.EPI_NONE)
    want = x.double() @ deq.double().T
    bound = x.double().abs() @ deq.double().abs().T * (2.0 ** -18 + (k / 16 + 32) * 2.0 ** -24) + 2.0 ** -126
    assert bool(((out.double() - want).abs() <= bound).all())
