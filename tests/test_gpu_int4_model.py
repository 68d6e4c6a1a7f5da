"""Models on 4-bit weights whose projections have a tiled form (csrc/gemv4_tiles.hip): prompts' last rows and captured steps against the row-major codes and the bf16 weights that both stand
for, a projection whose scales are refused among tiled ones, shards of a tensor-parallel rank; which form is kept does not depend on the memory that is free."""
import pytest
import torch

from chatts_amd import _lib, modeling
from chatts_amd.config import preset
from chatts_amd.modeling import ChatTSForCausalLM
from tests.tp_emulation import EmulatedTP

pytestmark = pytest.mark.gpu
NAMES = ("qkv", "o", "gate_up", "down")
# 8 projections and the head, whose inputs lose 2^-18 of their size when they are split into two parts (the row-major kernel for few codes and the bf16 one lose less); sums differ by less
BOUND = 9 * 2 * 2.0 ** -18
T = 37


def config(name):
    return preset(name, num_hidden_layers=2, vocab_size=4096, ts_token_start_index=4000, eos_token_id=[4003, 4002], pad_token_id=4002)


def model_of(name, **kw):
    return ChatTSForCausalLM.from_synthetic(config(name), seed=5, max_ctx=256, max_prefill_tokens=128, weight_format="int4", **kw)


def embedded(m):
    return m.get_input_embeddings(torch.randint(0, 4000, (T,), generator=torch.Generator().manual_seed(2)))


def logits(m):
    """of the prompt's last row, which runs alone in the last layer, and of three steps on tokens that no rounding chooses"""
    m.reset()
    last = m.prefill(embedded(m), 0, for_next_token=True)
    m.buf["pos"].fill_(T)
    m._first_token(last)
    out = [m.buf["logits"].clone()]
    for token in (7, 1234, 3999):
        m.buf["token"].fill_(token)
        m._load_token_embedding()
        m.decode_step()
        out.append(m.buf["logits"].clone())
    return torch.stack(out)


def rel(a, b):
    return float(((a.double() - b.double()).norm(dim=-1) / b.double().norm(dim=-1)).max())


def without_tiles(monkeypatch, make):
    with monkeypatch.context() as p:
        p.setattr(_lib.load(), "chatts_tile_w4_bytes", lambda *a: 0)
        return make()


@pytest.mark.parametrize("name", ["chatts-14b", "chatts-8b"])
def test_tiles_against_row_major_codes_and_bf16_weights(name, monkeypatch):
    m, plain = model_of(name), without_tiles(monkeypatch, lambda: model_of(name))
    for lw, lp in zip(m.layers, plain.layers):
        for n in NAMES:
            assert n + "4_tiles" in lw and n + "4" not in lw and n + "4_sz" not in lw and n + "4" in lp and n + "4_tiles" not in lp
            assert torch.equal(lw[n], lp[n])
            assert lw[n + "4_tiles"].numel() <= lp[n + "4"].numel() + lp[n + "4_sz"].numel() * 4 + lw[n].shape[0] // 4 * 1088      # (a unit per four rows that K does not fill)
    assert m.weight_bytes_local() < plain.weight_bytes_local()
    got, want = logits(m), logits(plain)
    assert torch.isfinite(got).all() and rel(got, want) < BOUND
    assert not torch.equal(got, want)                     # (another order of sums: the tiles ran)
    _lib.check(m.lib.chatts_decoder_set_w4_tiles(m._decoder, None, 0))      # no codes of any form are left: the bf16 weights
    m._graph = None
    assert rel(logits(m), got) < BOUND


def test_a_refused_scale_keeps_its_projection_row_major(monkeypatch):
    refused = {"calls": 0, "at": (1, 4 + 2)}               # o of the first layer, gate_up of the second
    quantize = modeling.quantize_int4_rows

    def odd_scales(w, group=128):
        codes, scale, zero, deq = quantize(w, group)
        if refused["calls"] % 8 in refused["at"]:
            scale[17, 2] *= 1 + 2.0 ** -13                  # (no float16 number)
            deq = (codes.float() * scale.repeat_interleave(group, 1) - (scale * zero).repeat_interleave(group, 1)).bfloat16()
        refused["calls"] += 1
        return codes, scale, zero, deq

    monkeypatch.setattr(modeling, "quantize_int4_rows", odd_scales)
    m, plain = model_of("chatts-14b"), without_tiles(monkeypatch, lambda: model_of("chatts-14b"))
    assert [[n + "4_tiles" in lw for n in NAMES] for lw in m.layers] == [[True, False, True, True], [True, True, False, True]]
    assert all((n + "4" in lw) != (n + "4_tiles" in lw) for lw in m.layers for n in NAMES)
    got, want = logits(m), logits(plain)
    assert rel(got, want) < BOUND and not torch.equal(got, want)


def test_codes_of_a_checkpoint(monkeypatch):
    """(codes that come with the weights of q, k, v, gate and up one by one)"""
    quantize, made = modeling.quantize_int4_rows, []
    with monkeypatch.context() as p:
        p.setattr(modeling, "quantize_int4_rows", lambda w, group=128: made.append(quantize(w, group)) or made[-1])
        want = model_of("chatts-8b")
    c = want.config
    d, pairs = c.head_dim, {"model.embed_tokens.weight": want._tensors["embed"], "model.norm.weight": want._tensors["final_norm"], "lm_head.weight": want._tensors["lm_head"]}
    rows = [n * d for n in (c.num_attention_heads, c.num_key_value_heads, c.num_key_value_heads)]
    for l, lw in enumerate(want.layers):
        qkv, o, gate_up, down = made[4 * l:4 * l + 4]
        halves = [t.view(-1, 2, 16, t.shape[1]) for t in gate_up]
        parts = dict(zip(("self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj"), zip(*(t.split(rows) for t in qkv))))
        parts |= {"self_attn.o_proj": o, "mlp.down_proj": down, "mlp.gate_proj": [t[:, 0].reshape(-1, t.shape[3]) for t in halves], "mlp.up_proj": [t[:, 1].reshape(-1, t.shape[3]) for t in halves]}
        for name, (codes, scale, zero, deq) in parts.items():
            pairs[f"model.layers.{l}.{name}.weight"], pairs[f"model.layers.{l}.{name}.gptq_codes"] = deq, (codes, scale, zero)
        for name, key in (("input_layernorm", "input_norm"), ("post_attention_layernorm", "post_norm"), ("self_attn.q_norm", "q_norm"), ("self_attn.k_norm", "k_norm")):
            pairs[f"model.layers.{l}.{name}.weight"] = lw[key]
    m = ChatTSForCausalLM(c, max_ctx=256, max_prefill_tokens=128)
    m.load_weights(pairs.items())
    assert all(torch.equal(a[n + "4_tiles"], b[n + "4_tiles"]) and n + "4" not in a for a, b in zip(m.layers, want.layers) for n in NAMES)
    assert torch.equal(logits(m), logits(want))


def test_free_memory_does_not_choose_the_form(monkeypatch):
    want = logits(model_of("chatts-14b", prefill_tiled_weights=False))
    before = torch.cuda.memory_allocated()
    plain = without_tiles(monkeypatch, lambda: model_of("chatts-14b", prefill_tiled_weights=False))
    row_major = torch.cuda.memory_allocated() - before
    del plain
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda *a: (1 << 30, 288 << 30))
    before = torch.cuda.memory_allocated()
    m = model_of("chatts-14b", prefill_tiled_weights=False)
    assert torch.cuda.memory_allocated() - before <= row_major
    assert torch.equal(logits(m), want)


def test_shards_of_two_ranks(monkeypatch):
    """(K of down_proj ends inside a unit)"""
    def run():
        tp = EmulatedTP(config("chatts-14b"), 2, seed=5, max_ctx=256, max_prefill_tokens=128, weight_format="int4")
        last = tp.prefill(embedded(tp.ms[0]))
        out = [tp.first_token(last, T)[1].clone()]
        for token in (7, 1234, 3999):
            for m in tp.ms:
                m.buf["token"].fill_(token)
                m._load_token_embedding()
            out.append(tp.decode_step()[1].clone())
            assert tp.residual_streams_identical(1)
        return tp, torch.stack(out)

    (tp, got), (plain, want) = run(), without_tiles(monkeypatch, run)
    assert all(n + "4_tiles" in lw for m in tp.ms for lw in m.layers for n in NAMES) and "qkv4" in plain.ms[0].layers[0]
    assert rel(got, want) < BOUND and not torch.equal(got, want)


def test_tiles_that_are_refused():
    """shapes without a tiled form, copies off 16 bytes, lists of another length"""
    import ctypes as C
    tiny, m = ChatTSForCausalLM.from_synthetic("tiny-qwen2", max_ctx=64, max_prefill_tokens=64, weight_format="int4"), model_of("chatts-8b")
    assert all(n + "4" in lw and n + "4_tiles" not in lw for lw in tiny.layers for n in NAMES)
    want = logits(m)
    at = m.layers[0]["qkv4_tiles"].data_ptr()

    def give(model, entries):
        return model.lib.chatts_decoder_set_w4_tiles(model._decoder, (C.c_void_p * len(entries))(*entries), len(entries))

    assert give(tiny, [at] + [None] * (4 * len(tiny.layers) - 1)) != 0 and give(tiny, [None] * (4 * len(tiny.layers))) == 0
    assert give(m, [at + 8] + [None] * 7) != 0 and give(m, [at] * 7) != 0 and give(m, [None] * 9) != 0
    assert m.lib.chatts_decoder_set_w4_tiles(m._decoder, None, 8) != 0 and m.lib.chatts_decoder_set_w4_tiles(None, None, 0) != 0
    m._graph = None
    assert torch.equal(logits(m), want)                   # (what was refused changed nothing)
