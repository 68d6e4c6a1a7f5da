"""The feed-forward beside experts in their launches (2 to 16 rows) and in launches of its own: the same products on the same operands, and whole prompts of either side of the line against
the plain references, with the tolerances of the models' own tests."""
import ctypes as C
import math

import pytest
import torch

from chatts_amd import _lib
from tests import test_gpu_mefurax as mefurax
from tests import test_gpu_muvetar as muvetar

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("module,name", [(m, n) for m in (muvetar, mefurax) for n in sorted(m.CONFIGS)], ids=lambda v: v if isinstance(v, str) else v.__name__.rsplit("_", 1)[-1])
def test_prompts_on_both_sides_of_sixteen_rows(module, name):
    m = module.load(name, "bfloat16", max_ctx=256, max_batch=2)
    for n in (1, 2, 15, 16, 17):
        toks = module.tokens(name, n, n)
        got = m.step_tokens([(n % 2, toks, list(range(n)))])
        assert module.worst(got, module.want(name, toks, "bfloat16")) < module.TOL[(name, "bfloat16")], n
        m.release_slot(n % 2)


class Beside(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("up", "up_t", "down", "down_t")] + [("ff", C.c_int)] + [(n, C.c_void_p) for n in ("f_hi", "f_lo", "y")] + [("limit", C.c_float), ("alpha", C.c_float)]


def experts_beside(args, beside, direct=False):
    f = getattr(_lib.load(), "_ZN6chatts11moe_expertsEPK13ChattsMoeArgsRKNS_9MoeBesideEbPv")
    f.argtypes = [C.c_void_p, C.c_void_p, C.c_bool, C.c_void_p]
    _lib.check(f(C.addressof(args), C.addressof(beside), direct, _lib.stream_ptr()))


def tiles(w):
    """chatts_tile_bf16's copy of every matrix of w [..., n, k]"""
    out = torch.empty_like(w)
    for a, b in zip(w.view(-1, *w.shape[-2:]), out.view(-1, *w.shape[-2:])):
        _lib.check(_lib.load().chatts_tile_bf16(a.data_ptr(), *a.shape, a.shape[1], b.data_ptr(), _lib.stream_ptr()))
    return out


def planes_of(t):
    hi = t.to(torch.bfloat16)
    return torch.stack([hi, (t - hi.float()).to(torch.bfloat16)])


# The activation is held in two bf16 parts on both sides; 32-bit sums in another order (1e-7) put one in a hundred of them into the next step of the low part: 1e-6 of the result.  The experts' own
# products are the same bits with and without.
@pytest.mark.parametrize("rows", [2, 15, 16])
@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("kind,epilogue", [(_lib.EXPERT_CLAMPGLU, _lib.EPI_CLAMPGLU), (_lib.EXPERT_RELU2, _lib.EPI_RELU2)])
@pytest.mark.parametrize("width,ff,shared,experts,top", [(192, 64, 320, 5, 2), (1088, 128, 64, 40, 3)])
def test_the_same_products(width, ff, shared, experts, top, kind, epilogue, tiled, rows):
    g, lib, DEV = torch.Generator(device="cuda").manual_seed(width + rows), _lib.load(), "cuda"
    two = 2 if kind == _lib.EXPERT_CLAMPGLU else 1
    w = lambda *s: (torch.randn(s, generator=g, device=DEV) / math.sqrt(s[-1])).bfloat16()
    up, down, sup, sdown = w(experts, two * ff, width), w(experts, width, ff), w(two * shared, width), w(width, shared)
    up_t, down_t, sup_t, sdown_t = (tiles(t) if tiled else None for t in (up, down, sup, sdown))
    h = planes_of(torch.randn((rows, width), generator=g, device=DEV))
    z = torch.randn((rows, experts), generator=g, device=DEV)
    table = torch.tensor([[i, 5, i, 0] for i in range(rows)], dtype=torch.int32, device=DEV)
    ints = lambda n: torch.zeros(n, dtype=torch.int32, device=DEV)
    ids, place, order, offsets, lists = ints(rows * top), ints(rows * top), ints(rows * top), ints(experts + 2), ints(4 * int(lib.chatts_moe_tiles(rows, top, experts)))
    weight, kept, y, act = torch.zeros((rows, top), device=DEV), torch.zeros(rows, device=DEV), torch.zeros((rows * top, width), device=DEV), torch.zeros((2, rows * top, ff), dtype=torch.bfloat16, device=DEV)
    a = _lib.MoeArgs(experts=experts, top=top, groups=1, keep=1, choose=_lib.CHOOSE_SOFTMAX, act_kind=kind, width_p=width, ff_p=ff, gate_up=up.data_ptr(), down=down.data_ptr(),
                     gate_up_t=_lib.ptr(up_t), down_t=_lib.ptr(down_t), logits=z.data_ptr(), ld_logits=experts, rows=table.data_ptr(), n_rows=rows, ids=ids.data_ptr(), place=place.data_ptr(),
                     order=order.data_ptr(), offsets=offsets.data_ptr(), tiles=lists.data_ptr(), weight=weight.data_ptr(), kept=kept.data_ptr(), y=y.data_ptr(), glu_limit=0.9, glu_alpha=1.3)
    a.h.hi, a.h.lo, a.h.ld = h[0].data_ptr(), h[1].data_ptr(), width
    a.act.hi, a.act.lo, a.act.ld = act[0].data_ptr(), act[1].data_ptr(), ff
    _lib.check(lib.chatts_moe_route(C.byref(a), _lib.stream_ptr()))
    _lib.check(lib.chatts_moe_experts(C.byref(a), _lib.stream_ptr()))
    alone = y.clone()
    y.fill_(float("nan"))
    f, own = torch.full((2, rows, shared), float("nan"), dtype=torch.bfloat16, device=DEV), torch.full((rows, width), float("nan"), device=DEV)
    experts_beside(a, Beside(up=sup.data_ptr(), up_t=_lib.ptr(sup_t), down=sdown.data_ptr(), down_t=_lib.ptr(sdown_t), ff=shared, f_hi=f[0].data_ptr(), f_lo=f[1].data_ptr(), y=own.data_ptr(),
                             limit=0.7, alpha=1.7))
    assert torch.equal(y, alone)
    f2, want, ws = torch.zeros_like(f), torch.zeros_like(own), torch.empty(1 << 26, dtype=torch.uint8, device=DEV)
    for x, m, out, n, k, epi in ((h, sup, f2, two * shared, width, epilogue), (f2, sdown, want, width, shared, _lib.EPI_NONE)):
        l = _lib.LinearArgs(w=m.data_ptr(), m=rows, n=n, k=k, ldw=k, a_hi=x[0].data_ptr(), a_lo=x[1].data_ptr(), ld_planes=k, epilogue=epi, workspace=ws.data_ptr(), workspace_bytes=ws.numel(),
                            glu_limit=0.7, glu_alpha=1.7)
        if out is f2:
            l.c_hi, l.c_lo, l.ld_cplanes = f2[0].data_ptr(), f2[1].data_ptr(), shared
        else:
            l.c, l.ldc = want.data_ptr(), width
        _lib.check(lib.chatts_linear(C.byref(l), _lib.stream_ptr()))
    value = lambda p: p[0].double() + p[1].double()
    assert float((value(f) - value(f2)).norm() / value(f2).norm()) < 3e-6
    assert float((own - want).double().norm() / want.double().norm()) < 3e-6
