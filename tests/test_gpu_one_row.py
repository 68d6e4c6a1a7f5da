"""A single row through layers with experts: the router and the feed-forward beside the experts take it as float32, as every projection of one row does, and not as two bf16 parts.  Columns
that differ by one part in 2^14 (2^20 for the router) are told apart: float32 keeps their difference to 2^-24 of them, two bf16 parts to 2^-17."""
import pytest
import torch

from chatts_amd.mefurax import MefuraxConfig, MefuraxForCausalLM
from chatts_amd.muvetar import MuvetarConfig, MuvetarForCausalLM
from oracle import mefurax, muvetar
from tests import mefurax_models, muvetar_models

pytestmark = pytest.mark.gpu
WIDTH, VOCAB, PAIRS = 128, 24, 32      # columns 2 r and 64 + 2 r hold the same values but for a norm's weights (even ones: position 0 adds nothing to them)
LEFT, RIGHT = 2 * torch.arange(PAIRS), 64 + 2 * torch.arange(PAIRS)


def twins(sd, norm, at, step):
    """columns RIGHT: those of LEFT, times 1 + step by the norm's weights (at: what stands for 1)"""
    sd["embed"][:, RIGHT] = sd["embed"][:, LEFT]
    sd[norm] = torch.full((WIDTH,), float(at))
    sd[norm][RIGHT] += step


def differences(sd, name):
    """a projection whose output r is RIGHT[r] - LEFT[r]"""
    w = torch.zeros(64, WIDTH)
    w[torch.arange(PAIRS), RIGHT], w[torch.arange(PAIRS), LEFT] = 1.0, -1.0
    sd[name] = w


def muvetar_model(experts, top, shared):
    cfg = {"vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6}, "residual_mult": 1.0, "logit_softcap": 20.0,
           "layers": [muvetar_models._moe(muvetar_models._gru(64), 64, 7.0, experts, top, 1.0, (64, 7.0) if shared else None)]}
    sd = {k: v.float() for k, v in muvetar.random_model(cfg, 0).items()}
    sd["l0.mix.o"].zero_()
    return cfg, sd


def errors(cfg, sd, oracle, Config, Model, name):
    m = Model(Config.from_dict(dict(cfg, architecture=name)), dtype="bfloat16", max_ctx=64, max_batch=2)
    m.load_weights(sd.items())
    for t in range(VOCAB):
        got, want = m.step_tokens([(t % 2, [t], [0])]).double().cpu(), oracle.forward(cfg, sd, [t])
        yield float((got - want).norm() / want.norm())
        m.release_slot(t % 2)


# float32: the one rounding of a column, 2^-24 of 2^-14, so 1e-3 of a difference (twice that squared); two bf16 parts: 4e-2
def test_the_feed_forward_beside_gated_experts():
    cfg, sd = muvetar_model(4, 2, True)
    twins(sd, "l0.norm2", 1.0, 2.0 ** -14)
    differences(sd, "l0.mlp.shared.gate")
    sd["l0.mlp.shared.up"].zero_()
    sd["l0.mlp.shared.down"] *= 2.0 ** 14
    for e in range(4):
        sd[f"l0.mlp.e{e}.down"].zero_()
    assert max(errors(cfg, sd, muvetar, MuvetarConfig, MuvetarForCausalLM, "Muvetar")) < 1e-3


def test_the_feed_forward_beside_squared_relu_experts():
    cfg = {"vocab": VOCAB, "width": WIDTH, "norm": {"eps": 1e-6}, "postln_alpha": 1.0, "layers": [mefurax_models._moe(mefurax_models._rot(4, 4, 32, 32, 0.25, 20.0, 1000.0, 16), 64, 4, 2, 64)]}
    sd = {k: v.float() for k, v in mefurax.random_model(cfg, 0).items()}
    sd["l0.mix.o"].zero_()
    twins(sd, "l0.norm1", 0.0, 2.0 ** -14)
    differences(sd, "l0.mlp.shared.up")
    sd["l0.mlp.shared.down"] *= 2.0 ** 28
    for e in range(4):
        sd[f"l0.mlp.e{e}.down"].zero_()
    assert max(errors(cfg, sd, mefurax, MefuraxConfig, MefuraxForCausalLM, "Mefurax")) < 2e-3


# two experts' logits are LEFT[0] and RIGHT[0]; the first of the two adds nothing.  Experts take their operands as two bf16 parts: 1e-5 of what they add
@pytest.mark.parametrize("experts", [4, 40])
def test_a_close_choice(experts):
    cfg, sd = muvetar_model(experts, 1, False)
    sd["embed"][:, 0] = (sd["embed"][:, 0].abs() + 0.5).bfloat16().float()
    twins(sd, "l0.norm2", 1.0, 2.0 ** -20)
    sd["l0.mlp.router"].zero_()
    sd["l0.mlp.router"][1, LEFT[0]] = sd["l0.mlp.router"][3, RIGHT[0]] = 1.0
    sd["l0.mlp.e1.down"].zero_()
    assert max(errors(cfg, sd, muvetar, MuvetarConfig, MuvetarForCausalLM, "Muvetar")) < 2e-5
