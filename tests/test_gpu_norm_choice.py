"""The choice of experts in the norm's launch and experts without lists (up to 16 rows and 64 pairs) against the norm, the router, the choice and the lists in launches of their own: the
rows at which a step changes its kernels, routers of up to 32 and up to 64 outputs, K-steps that leave waves without work, and pairs beyond 64."""
import pytest
import torch

from chatts_amd.muvetar import MuvetarConfig, MuvetarForCausalLM
from oracle import muvetar as F

pytestmark = pytest.mark.gpu


def model(width, experts, top):
    moe = {"kind": "moe", "expert": {"ff": 96, "limit": 2.0}, "router": {"experts": experts, "top": top, "scale": 1.3}, "shared": {"ff": 160, "limit": 1.5}}
    cfg = {"vocab": 96, "width": width, "norm": {"eps": 1e-5}, "residual_mult": 0.6, "logit_softcap": 20.0,
           "layers": [{"type": "mingru", "mixer": {"width": 64}, "mlp": moe}, {"type": "mingru", "mixer": {"width": 80}, "mlp": dict(moe, shared=None)}]}
    for l in cfg["layers"]:
        if l["mlp"]["shared"] is None:
            l["mlp"] = {k: v for k, v in l["mlp"].items() if k != "shared"}
    return cfg, F.random_model(cfg, width + experts)


# bf16 weights and activations in two bf16 parts, 32-bit sums: the reference (float64 on the same weights) is 1e-5 away for two such layers, where the same experts are chosen; three
# chances in a thousand rows that a rounding turns a choice are left to the seeds, which are fixed
@pytest.mark.parametrize("width,experts,top", [(64, 5, 1), (128, 32, 4), (704, 33, 4), (2112, 64, 4), (1024, 12, 7), (4096, 20, 3), (4160, 9, 2)])
def test_rows(width, experts, top):
    cfg, sd = model(width, experts, top)
    m = MuvetarForCausalLM(MuvetarConfig.from_dict(dict(cfg, architecture="Muvetar")), dtype="bfloat16", max_ctx=64, max_batch=2)
    m.load_weights(sd.items())
    for n in (1, 2, 9, 15, 16, 17):
        toks = torch.randint(0, 96, (n,), generator=torch.Generator().manual_seed(n + experts)).tolist()
        got = m.step_tokens([(n % 2, toks, list(range(n)))]).double().cpu()
        want = F.forward(cfg, sd, toks).double()
        assert float((got - want).norm() / want.norm()) < 2e-4, n
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
    assert float((got - want).norm() / want.norm()) < 2e-4
    assert bool(m.buf["moe_logits"].view(-1)[:experts].isfinite().all()) == own
