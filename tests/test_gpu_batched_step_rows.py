"""A whole batched decode step: a sequence's logits are the same bits however many sequences share the step, and the norm that the projections hand on between them
agrees with norms in launches of their own."""
import pytest
import torch

from chatts_amd import _lib
from chatts_amd.config import preset
from chatts_amd.modeling import ChatTSForCausalLM

pytestmark = pytest.mark.gpu
SPLITS = 8


def model_of(name, form):
    cfg = preset(name, num_hidden_layers=2, vocab_size=4096, ts_token_start_index=4000, eos_token_id=[4003, 4002], pad_token_id=4002)
    m = ChatTSForCausalLM.from_synthetic(cfg, seed=5, max_ctx=256, max_prefill_tokens=512, max_batch=16, weight_format=form)
    g = torch.Generator().manual_seed(1)
    m.step_tokens([(s, torch.randint(0, 4000, (5 + 11 * s % 60,), generator=g).tolist(), []) for s in range(16)])
    return m, torch.tensor([5 + 11 * s % 60 for s in range(16)], dtype=torch.int32, device="cuda"), torch.randint(0, 4000, (16,), generator=g).cuda()


def start(m, positions, tokens):
    b = m.buf
    b["pos_all"].copy_(positions)
    b["step_all"].zero_()
    b["token_all"].copy_(tokens)
    b["logits_all"].fill_(float("nan"))
    return b


def step(m, positions, tokens, batch):
    b = start(m, positions, tokens)
    _lib.check(m.lib.chatts_decoder_decode_step_batched(m._decoder, batch, _lib.ptr(b["pos_all"]), _lib.ptr(b["step_all"]), _lib.ptr(b["token_all"]), _lib.ptr(b["token_logit_all"]),
                                                        _lib.ptr(b["out_tokens_all"]), b["out_tokens_all"].shape[1], _lib.ptr(b["logits_all"]), SPLITS, _lib.stream_ptr()))
    torch.cuda.synchronize()
    assert torch.isfinite(b["logits_all"][:batch]).all()
    return b["logits_all"][:batch].clone()


def step_in_parts(m, positions, tokens, batch):
    """the same step through the calls for one part of a layer, which leave every norm to a launch of its own"""
    b, lib = start(m, positions, tokens), m.lib
    _lib.check(lib.chatts_embed_token_batched(_lib.ptr(b["token_all"]), batch, _lib.ptr(m._tensors["embed"]), 0, 4096, m.config.hidden_size, _lib.ptr(b["x"]), _lib.stream_ptr()))
    for layer in range(m.config.num_hidden_layers):
        for part in (0, 1):
            _lib.check(lib.chatts_decoder_layer_part_batched(m._decoder, layer, part, batch, _lib.ptr(b["pos_all"]), SPLITS, _lib.stream_ptr()))
    _lib.check(lib.chatts_decoder_logits_batched(m._decoder, batch, _lib.ptr(b["logits_all"]), _lib.stream_ptr()))
    torch.cuda.synchronize()
    return b["logits_all"][:batch].clone()


FORMS = [("chatts-8b", "bf16"), ("chatts-14b", "bf16"), ("chatts-14b", "fp8"), ("chatts-8b", "int8"), ("tiny-qwen3", "bf16")]


@pytest.mark.parametrize("name,form", FORMS)
def test_the_number_of_sequences(name, form):
    m, positions, tokens = model_of(name, form)
    all16 = step(m, positions, tokens, 16)
    for batch in (2, 3, 4, 5, 8, 9, 15):
        assert torch.equal(step(m, positions, tokens, batch), all16[:batch]), batch


@pytest.mark.parametrize("name,form", FORMS)
def test_separate_norms(monkeypatch, name, form):
    m, positions, tokens = model_of(name, form)
    for batch in (3, 8, 16):
        parts, handed_on = step_in_parts(m, positions, tokens, batch), step(m, positions, tokens, batch)
        # the factor 1 / rms is applied behind the products instead of in front of them: roundings, a few of 2^-17 a layer where planes hold the row
        assert float((parts - handed_on).norm() / parts.norm()) < 1e-4
        monkeypatch.setenv("CHATTS_POST_NORM_SMALL_M", "0")
        assert torch.equal(step(m, positions, tokens, batch), parts)
        monkeypatch.delenv("CHATTS_POST_NORM_SMALL_M")


@pytest.mark.parametrize("batch", [3, 16])
def test_one_gpu_leaves_delta_alone(batch):
    """buffers.delta belongs to tensor parallelism: a program on one GPU may keep other things there"""
    m, positions, tokens = model_of("chatts-8b", "bf16")
    want = step(m, positions, tokens, batch)
    m.buf["delta"].fill_(7.0)
    assert torch.equal(step(m, positions, tokens, batch), want) and bool((m.buf["delta"] == 7.0).all())
