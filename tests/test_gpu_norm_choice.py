"""The choice of experts in the norm's launch and experts without lists (2 to 16 rows and up to 64 pairs): the kernels against the norm, the router, the choice and the lists in launches of
their own, and whole models against the plain reference: the rows at which a step changes its kernels, routers of up to 32 and up to 64 outputs, K-steps that leave waves without work, and
pairs beyond 64."""
import ctypes as C
import math

import pytest
import torch

from chatts_amd import _lib
from chatts_amd.muvetar import MuvetarConfig, MuvetarForCausalLM
from oracle import muvetar as F
from tests.test_gpu_moe_beside import Beside, experts_beside, tiles

pytestmark = pytest.mark.gpu


def model(width, experts, top):
    moe = {"kind": "moe", "expert": {"ff": 96, "limit": 2.0}, "router": {"experts": experts, "top": top, "scale": 1.3}, "shared": {"ff": 160, "limit": 1.5}}
    cfg = {"vocab": 96, "width": width, "norm": {"eps": 1e-5}, "residual_mult": 0.6, "logit_softcap": 20.0,
           "layers": [{"type": "mingru", "mixer": {"width": 64}, "mlp": moe}, {"type": "mingru", "mixer": {"width": 80}, "mlp": dict(moe, shared=None)}]}
    for l in cfg["layers"]:
        if l["mlp"]["shared"] is None:
            l["mlp"] = {k: v for k, v in l["mlp"].items() if k != "shared"}
    return cfg, F.random_model(cfg, width + experts)


# bf16 weights and activations in two bf16 parts (2^-17 of a value, in seven products of a layer), 32-bit sums: the reference (float64 on the same weights) is 2e-6 to 8e-6 away for two such
# layers, where the same experts are chosen, and four times that is allowed; three chances in a thousand rows that a rounding turns a choice are left to the seeds, which are fixed
@pytest.mark.parametrize("width,experts,top", [(64, 5, 1), (128, 32, 4), (704, 33, 4), (2112, 64, 4), (1024, 12, 7), (4096, 20, 3), (4160, 9, 2)])
def test_rows(width, experts, top):
    cfg, sd = model(width, experts, top)
    m = MuvetarForCausalLM(MuvetarConfig.from_dict(dict(cfg, architecture="Muvetar")), dtype="bfloat16", max_ctx=64, max_batch=2)
    m.load_weights(sd.items())
    for n in (1, 2, 9, 15, 16, 17):
        toks = torch.randint(0, 96, (n,), generator=torch.Generator().manual_seed(n + experts)).tolist()
        got = m.step_tokens([(n % 2, toks, list(range(n)))]).double().cpu()
        want = F.forward(cfg, sd, toks).double()
        assert float((got - want).norm() / want.norm()) < 3e-5, n
        m.release_slot(n % 2)


class FewRouterRows(MuvetarForCausalLM):
    """a C caller's router: as many rows as its outputs fill in blocks of 16"""

    def _experts(self, L, m):
        super()._experts(L, m)
        L.router_n = -(-(len(m.experts) + m.identity) // 16) * 16


# the norm's launch reads 32 rows of a router or 64: one that is shorter goes through launches of its own (its logits say so)
@pytest.mark.parametrize("experts,own", [(9, True), (16, True), (17, False), (32, False), (33, True), (48, True), (49, False)])
def test_a_router_of_few_rows(experts, own):
    cfg, sd = model(128, experts, 2)
    m = FewRouterRows(MuvetarConfig.from_dict(dict(cfg, architecture="Muvetar")), dtype="bfloat16", max_ctx=64, max_batch=2)
    m.load_weights(sd.items())
    m.buf["moe_logits"].fill_(float("nan"))
    toks = list(range(5))
    got = m.step_tokens([(0, toks, toks)]).double().cpu()
    want = F.forward(cfg, sd, toks).double()
    assert float((got - want).norm() / want.norm()) < 3e-5
    assert bool(m.buf["moe_logits"].view(-1)[:experts].isfinite().all()) == own


def choose(norm, moe, router, router_t):
    f = getattr(_lib.load(), "_ZN6chatts17depth_norm_chooseEPK19ChattsDepthNormArgsPK13ChattsMoeArgsPKtS7_iPv")
    f.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_void_p]
    _lib.check(f(C.addressof(norm), C.addressof(moe), router.data_ptr(), _lib.ptr(router_t), router.shape[0], _lib.stream_ptr()))


# The same norm and the same planes: bit for bit.  Logits are sums of the same products in another order, 1e-6 of their size (2) at most, and so are the weights; experts that are given the same
# choice are the same bits, in lists or not.
@pytest.mark.parametrize("kind", [_lib.CHOOSE_SOFTMAX, _lib.CHOOSE_LOGITS, _lib.CHOOSE_SCORES])
@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("width,experts,identity,top,corrected", [(64, 5, 0, 1, False), (192, 29, 3, 4, True), (1088, 33, 0, 4, False), (2112, 60, 4, 6, True), (4096, 32, 0, 32, False),
                                                                  (1024, 64, 0, 4, True)])
def test_launches_of_their_own(width, experts, identity, top, corrected, tiled, kind):
    g, lib, DEV = torch.Generator(device="cuda").manual_seed(width + experts), _lib.load(), "cuda"
    outputs, ff = experts + identity, 64
    R, M = 64 if outputs > 32 else 32, 64 // top if top > 4 else 16
    lin = lambda *s: (torch.randn(s, generator=g, device=DEV) / math.sqrt(s[-1])).bfloat16()
    router = torch.zeros((R, width), dtype=torch.bfloat16, device=DEV)
    router[:outputs] = 2 * lin(outputs, width)
    up, down = lin(experts, 2 * ff, width), lin(experts, width, ff)
    router_t, up_t, down_t = (tiles(t) if tiled else None for t in (router, up, down))
    w, cor = torch.randn(width, generator=g, device=DEV), torch.randn(outputs, generator=g, device=DEV) * 0.05 if corrected else None
    for T in sorted({t for t in (2, 3, 15, 16) if t <= M} | {M}):
        x, y = (torch.randn((T, width), generator=g, device=DEV) for _ in "xy")
        rows = torch.tensor([[i, -1 if i == 2 else 5, i, 0] for i in range(T)], dtype=torch.int32, device=DEV)

        def buffers():
            ints = lambda n: torch.full((n,), -7, dtype=torch.int32, device=DEV)
            b = dict(x=x.clone(), planes=torch.full((2, T, width), float("nan"), dtype=torch.bfloat16, device=DEV), ids=ints(T * top), place=ints(T * top), order=ints(T * top),
                     offsets=ints(experts + 2), tiles=ints(4 * int(lib.chatts_moe_tiles(T, top, experts))), weight=torch.full((T, top), -7.0, device=DEV), kept=torch.full((T,), -7.0, device=DEV),
                     z=torch.full((T, R), float("nan"), device=DEV), act=torch.zeros((2, T * top, ff), dtype=torch.bfloat16, device=DEV), ey=torch.zeros((T * top, width), device=DEV))
            n = _lib.DepthNormArgs(x=b["x"].data_ptr(), t=T, width=width, ldx=width, mult=0.5, eps=1e-5, y=y.data_ptr(), w=w.data_ptr())
            n.out.hi, n.out.lo, n.out.ld = b["planes"][0].data_ptr(), b["planes"][1].data_ptr(), width
            a = _lib.MoeArgs(experts=experts, identity=identity, top=top, groups=1, keep=1, choose=kind, act_kind=_lib.EXPERT_CLAMPGLU, width_p=width, ff_p=ff, gate_up=up.data_ptr(),
                             down=down.data_ptr(), gate_up_t=_lib.ptr(up_t), down_t=_lib.ptr(down_t), correction=_lib.ptr(cor), logits=b["z"].data_ptr(), ld_logits=R, rows=rows.data_ptr(), n_rows=T,
                             weight_scale=2.5, glu_limit=0.9, glu_alpha=1.3, y=b["ey"].data_ptr(),
                             **{k: b[k].data_ptr() for k in ("ids", "place", "order", "offsets", "tiles", "weight", "kept")})
            a.h.hi, a.h.lo, a.h.ld = n.out.hi, n.out.lo, width
            a.act.hi, a.act.lo, a.act.ld = b["act"][0].data_ptr(), b["act"][1].data_ptr(), ff
            return b, n, a

        one, norm, a = buffers()
        choose(norm, a, router, router_t)
        two, norm2, a2 = buffers()
        _lib.check(lib.chatts_depth_norm(C.byref(norm2), _lib.stream_ptr()))
        ws = torch.empty(1 << 24, dtype=torch.uint8, device=DEV)
        l = _lib.LinearArgs(w=router.data_ptr(), m=T, n=R, k=width, ldw=width, a_hi=a2.h.hi, a_lo=a2.h.lo, ld_planes=width, c=two["z"].data_ptr(), ldc=R, epilogue=_lib.EPI_NONE,
                            workspace=ws.data_ptr(), workspace_bytes=ws.numel())
        _lib.check(lib.chatts_linear(C.byref(l), _lib.stream_ptr()))
        _lib.check(lib.chatts_moe_route(C.byref(a2), _lib.stream_ptr()))
        assert torch.equal(one["planes"], two["planes"]) and torch.equal(one["x"], two["x"])
        assert torch.equal(one["ids"], two["ids"]) and (T <= 2 or one["ids"].view(T, top)[2].eq(-1).all())
        live = [i for i in range(T) if i != 2]
        scale = float(two["weight"][live].abs().max())
        assert float((one["weight"] - two["weight"])[live].abs().max()) < 4e-6 * scale and float((one["kept"] - two["kept"]).abs().max()) < 4e-6 * scale * top
        own = torch.arange(T * top, dtype=torch.int32, device=DEV)
        assert torch.equal(one["place"], torch.where(one["ids"] >= 0, own, -torch.ones_like(own))) and torch.equal(one["place"] >= 0, two["place"] >= 0)
        experts_beside(a, Beside(), direct=True)
        _lib.check(lib.chatts_moe_experts(C.byref(a2), _lib.stream_ptr()))
        pairs = (one["ids"] >= 0).nonzero().view(-1)
        assert torch.equal(one["ey"][pairs], two["ey"][two["place"][pairs].long()])
