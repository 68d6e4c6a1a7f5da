"""Muvetar's steps of few rows where the input projection leaves its splits to the layer's own launches (csrc/gru.hip, csrc/window.hip) and the output projection to the norm that chooses
experts (csrc/depth.hip): heads of 48 to 200 channels, one to five taps, sizes that no quad fits (those keep the launches of their own), up to eight splits and sixteen, a place that is not
taken - against the plain reference, against projections without splits, and bit for bit against sums in launches of their own; that the sums are left at all."""
import pytest
import torch

from chatts_amd import _lib
from chatts_amd.muvetar import MuvetarConfig, MuvetarForCausalLM
from oracle import muvetar as F
from tests.muvetar_models import CONFIGS, _gru, _moe, _par, model
from tests.test_gpu_muvetar import TOL, tokens, worst

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def own_random_numbers():
    """the tests behind these draw what they would draw without them"""
    with torch.random.fork_rng():
        yield


def steps(name, n=5):
    _, public, sd = model(name, all_experts=True)
    m = MuvetarForCausalLM(MuvetarConfig.from_dict(public), dtype="bfloat16", max_ctx=128, max_batch=4)
    m.load_weights(sd.items())
    toks = {s: tokens(name, k + n, 20 + s) for s, k in ((0, 3), (1, 70), (3, 1))}
    out = {s: [] for s in toks}
    pos = torch.full((4,), -1, dtype=torch.int32)
    for s, t in toks.items():
        pos[s] = len(t) - n
        m.step_tokens([(s, t[:len(t) - n], [])])
        m.reserve_kv(s, 100)
    for i in range(n):
        m.buf["pos_all"].copy_(pos)
        m.buf["token_all"].copy_(torch.tensor([toks[s][len(toks[s]) - n + i] if s in toks else 0 for s in range(4)]))
        m.batched_step()
        for s in toks:
            out[s].append(m.buf["logits_all"][s, :CONFIGS[name]["vocab"]].clone())
        pos[pos >= 0] += 1
    return toks, {s: torch.stack(v) for s, v in out.items()}


@pytest.mark.parametrize("splits", [2, 3, 5, 8, 12])
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_sums_left_to_the_layer(name, splits):
    cfg, _, sd = model(name, all_experts=True)
    with _lib.options(GEMM_SK=splits):      # (the workspace is sized for them, too)
        toks, got = steps(name)
    with _lib.options(GEMM_SK=splits, SPLIT_SUMS=0):
        _, apart = steps(name)
    with _lib.options(GEMM_SK=1):
        _, whole = steps(name)
    for s, t in toks.items():
        assert worst(got[s], F.forward(cfg, sd, t)[-len(got[s]):]) < TOL[name, "bfloat16"]
        assert worst(got[s], whole[s].cpu()) < TOL[name, "bfloat16"]
        assert torch.equal(got[s], apart[s])


# one layer of each kind whose sums are left, nothing behind it that writes what its projections would have written; K of 1024 for both
ALONE = {"recurrence": _moe(_gru(1024), 64, 7.0, 4, 4, 1.0), "attention beside a scan": _moe(_par(8, 2, 64, 64, 0.2, 512, 16, 16, 4, (0.9, 0.5)), 64, 7.0, 4, 4, 1.0)}


@pytest.mark.parametrize("splits", [2, 8, 16])
@pytest.mark.parametrize("kind", sorted(ALONE))
def test_the_sums_are_left(kind, splits):
    public = {"vocab": 96, "width": 1024, "norm": {"eps": 1e-5}, "residual_mult": 0.5, "logit_softcap": 30.0, "layers": [ALONE[kind]], "architecture": "Muvetar"}
    sd = F.random_model({k: v for k, v in public.items() if k != "architecture"}, 1)
    got = {}
    for on in (1, 0):
        with _lib.options(GEMM_SK=splits, SPLIT_SUMS=on):
            m = MuvetarForCausalLM(MuvetarConfig.from_dict(public), dtype="bfloat16", max_ctx=128, max_batch=4)
            m.load_weights(sd.items())
            for s in range(4):
                m.step_tokens([(s, tokens("plain", 5 + s, s), [])])
                m.reserve_kv(s, 100)
            m.buf["pos_all"].copy_(torch.arange(5, 9, dtype=torch.int32))
            m.buf["token_all"].copy_(torch.tensor([3, 50, 7, 90]))
            m.buf["proj"].fill_(5.0)
            m.buf["y"].fill_(5.0)
            m.batched_step()
            got[on] = [m.buf[n].clone() for n in ("logits_all", "proj", "y")]
    assert torch.equal(got[1][0], got[0][0])
    written = {on: [int((t != 5.0).sum()) for t in got[on][1:]] for on in got}
    assert (written[1][0] < written[0][0]) == (splits <= 8) and written[1][1] == 0 < written[0][1]      # (the mixers take eight splits, the norm sixteen)
