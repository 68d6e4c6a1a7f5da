"""Muvetar's steps of few rows where the input projection leaves its splits to the layer's own launches (csrc/gru.hip, csrc/window.hip) and the output projection to the norm that chooses
experts (csrc/depth.hip): heads of 48 to 200 channels, one to five taps, sizes that no quad fits (those keep the launches of their own), up to eight splits and sixteen, a place that is not
taken - against the plain reference, and against projections without splits."""
import pytest
import torch

from chatts_amd import _lib
from chatts_amd.muvetar import MuvetarConfig, MuvetarForCausalLM
from oracle import muvetar as F
from tests.muvetar_models import CONFIGS, model
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
    with _lib.options(GEMM_SK=1):
        _, whole = steps(name)
    for s, t in toks.items():
        assert worst(got[s], F.forward(cfg, sd, t)[-len(got[s]):]) < TOL[name, "bfloat16"]
        assert worst(got[s], whole[s].cpu()) < TOL[name, "bfloat16"]
