"""The batch-1 projection on 4-bit codes laid out once (csrc/gemv4_tiles.hip): every weight is the stored bf16 value bit for bit, sums against float64; rows that deal unevenly over the CUs,
K below a unit, ending inside one and the largest, gated rows, the fused norm; what the layout refuses."""
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


# one unit a row that K does not fill; fewer quads than CUs and the largest K; K that ends inside a unit; groups of more than a part; ChatTS shapes
SHAPES = [(65568, 128, 128), (544, 16384, 128), (2080, 4224, 128), (6176, 2048, 1024), (3296, 2560, 256), (7168, 5120, 128), (5120, 13824, 128), (27648, 5120, 128)]


def problem(n, k, group, seed):
    from chatts_amd.modeling import pack_int4, quantize_int4_rows
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)
    codes, scale, zero, deq = quantize_int4_rows((r(n, k) * k ** -0.5 * 10.0 ** (torch.rand((n, 1), generator=g, device=DEV) - 1)).bfloat16(), group)
    return r(1, k), pack_int4(codes, scale, zero), deq, r(n), r(1, n), 1 + 0.1 * r(k)


def tiled(w4, sz, n, k, group, gated=False):
    lib = _lib.load()
    need = lib.chatts_tile_w4_bytes(n, k, group)
    assert need > 0
    tiles, bad = torch.empty(need, dtype=torch.uint8, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV)
    _lib.check(lib.chatts_tile_w4(w4.data_ptr(), sz.data_ptr(), n, k, k // 2, group, int(gated), tiles.data_ptr(), bad.data_ptr(), _lib.stream_ptr()))
    return tiles, int(bad.item())


def run(x, tiles, n, epi, bias=None, resid=None, norm=None):
    k = x.shape[1]
    out = torch.full((1, n // 2 if epi == _lib.EPI_SWIGLU else n), float("nan"), device=DEV)
    a = _lib.LinearArgs(a=x.data_ptr(), bias=_lib.ptr(bias), resid=_lib.ptr(resid), c=out.data_ptr(), norm_w=_lib.ptr(norm), norm_eps=1e-6, m=1, n=n, k=k, lda=k, ldw=k, ldc=out.shape[1],
                        epilogue=epi)
    _lib.check(_lib.load().chatts_linear_w4_tiles(C.byref(a), tiles.data_ptr(), _lib.stream_ptr()))
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("n,k,group", SHAPES)
def test_weights_are_the_stored_ones(n, k, group):
    _, (w4, sz), deq, *_ = problem(n, k, group, n + k)
    tiles, bad = tiled(w4, sz, n, k, group)
    assert bad == 0
    for at in [0, 3, 15, 16, 47, 127, k // 2 + 5, k - 1]:
        x = torch.zeros((1, k), device=DEV)
        x[0, at] = 1.0
        assert torch.equal(run(x, tiles, n, _lib.EPI_NONE)[0], deq[:, at].float())


@pytest.mark.parametrize("epi,norm", [(_lib.EPI_NONE, True), (_lib.EPI_RESID, False), (_lib.EPI_SWIGLU, True)])
@pytest.mark.parametrize("n,k,group", SHAPES)
def test_sums(n, k, group, norm, epi):
    x, (w4, sz), deq, bias, resid, nw = problem(n, k, group, n * k)
    xd = x.double()
    if norm:
        xd = xd * torch.rsqrt((xd * xd).mean() + 1e-6) * nw.double()
    deqd = deq.double()
    want = (deqd @ xd[0])[None] + bias.double()
    # x = hi + lo loses 2^-18 of each term; float32 sums of K / 16 terms a lane and 16 more: 2^-24 a step, at most (K / 16 + 32) of them
    bound = (deqd.abs() @ xd[0].abs())[None] * (2.0 ** -18 + (k / 16 + 32) * 2.0 ** -24) + want.abs() * 2.0 ** -20
    if epi == _lib.EPI_RESID:
        want = want + resid.double()
        bound = bound + want.abs() * 2.0 ** -24
    if epi == _lib.EPI_SWIGLU:
        z, dz = want.view(-1, 2, 16), bound.view(-1, 2, 16)
        gate = torch.nn.functional.silu(z[:, 0])
        want = (gate * z[:, 1]).reshape(1, -1)
        bound = (1.1 * dz[:, 0] * (z[:, 1].abs() + dz[:, 1]) + gate.abs() * dz[:, 1]).reshape(1, -1) + want.abs() * 2.0 ** -20      # (silu's slope is below 1.1)
    tiles, bad = tiled(w4, sz, n, k, group, epi == _lib.EPI_SWIGLU)
    assert bad == 0
    out = run(x, tiles, n, epi, bias, resid, nw if norm else None)
    assert bool(((out.double() - want).abs() <= bound).all())


def test_scales_of_the_whole_range():
    """float16's smallest and largest scales that are taken, signs, zeros of both ends; and what is counted as not to be had: no float16, too large, a fraction, not finite"""
    from chatts_amd.modeling import pack_int4
    n, k, group = 2080, 4224, 128
    g = torch.Generator(device=DEV).manual_seed(3)
    codes = torch.randint(0, 16, (n, k), generator=g, device=DEV, dtype=torch.uint8)
    scale = (2.0 ** torch.randint(-24, 12, (n, k // group), generator=g, device=DEV)) * torch.where(torch.rand((n, k // group), generator=g, device=DEV) < 0.5, -1.0, 1.0)
    scale[::5, ::3] = 1.2666015625                    # (eleven significant bits)
    scale[3::7, 2::5] = 0.0
    zero = torch.randint(-64, 65, scale.shape, generator=g, device=DEV).float()
    deq = (codes.float() * scale.repeat_interleave(group, 1) - (scale * zero).repeat_interleave(group, 1)).bfloat16()
    w4, sz = pack_int4(codes, scale, zero)
    tiles, bad = tiled(w4, sz, n, k, group)
    assert bad == 0
    for at in [0, 129, 1000, k - 1]:
        x = torch.zeros((1, k), device=DEV)
        x[0, at] = 1.0
        assert torch.equal(run(x, tiles, n, _lib.EPI_NONE)[0], deq[:, at].float())
    for s, z in [(1.0 + 2.0 ** -11, 8.0), (4096.0, 8.0), (1.0, 7.5), (1.0, 65.0), (float("inf"), 8.0), (float("nan"), 8.0)]:
        scale2, zero2 = scale.clone(), zero.clone()
        scale2[17, 2], zero2[17, 2] = s, z
        assert tiled(*pack_int4(codes, scale2, zero2), n, k, group)[1] >= 1


def test_what_is_refused():
    lib = _lib.load()
    for n, k, group in [(8, 16384, 128), (2072, 4224, 128), (2080, 4224, 64), (2080, 4224, 96), (2080, 4224 + 64, 128), (544, 16512, 128), (1024, 4096, 128), (1 << 21, 4096, 128)]:
        assert lib.chatts_tile_w4_bytes(n, k, group) == 0
    x, (w4, sz), *_ = problem(2080, 4224, 128, 1)
    tiles, _ = tiled(w4, sz, 2080, 4224, 128)
    for kw in [dict(m=2), dict(epilogue=_lib.EPI_GELU), dict(epilogue=_lib.EPI_RESID), dict(n=2072), dict(k=16512)]:
        a = _lib.LinearArgs(**{**dict(a=x.data_ptr(), c=x.data_ptr(), m=1, n=2080, k=4224, lda=4224, ldw=4224, ldc=2080, epilogue=_lib.EPI_NONE), **kw})
        assert lib.chatts_linear_w4_tiles(C.byref(a), tiles.data_ptr(), None) != 0
