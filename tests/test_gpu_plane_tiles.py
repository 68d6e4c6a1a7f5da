"""Planes between the projections of a prefill chunk and of the encoder in the prefill kernel's blocks (PLANE_TILES, on from 129 rows): the same bits as row-major planes, for chunks
that end with a whole block of 16 rows, with one more row and with one row less, split and unsplit projections, packed prompts, and every kernel that writes such planes."""
import threading

import pytest
import torch

from chatts_amd import _lib
from chatts_amd.config import preset
from chatts_amd.modeling import ChatTSForCausalLM

pytestmark = pytest.mark.gpu


def both(f):
    on = f()
    with _lib.options(PLANE_TILES=0):
        off = f()
    return on, off


@pytest.fixture(scope="module", params=["chatts-8b", "chatts-14b"])
def model(request):
    cfg = preset(request.param, num_hidden_layers=3, vocab_size=4096, ts_token_start_index=4000, eos_token_id=[4003, 4002], pad_token_id=4002)
    return ChatTSForCausalLM.from_synthetic(cfg, seed=3, max_ctx=1024, max_prefill_tokens=512, max_batch=4, enable_prefix_caching=False)


@pytest.fixture(scope="module")
def narrow():
    """(a workspace that holds ten slabs of 201 rows)"""
    cfg = preset("chatts-8b", num_hidden_layers=3, intermediate_size=1024, vocab_size=4096, ts_token_start_index=4000, eos_token_id=[4003, 4002], pad_token_id=4002)
    return ChatTSForCausalLM.from_synthetic(cfg, seed=4, max_ctx=2048, max_prefill_tokens=2048, max_batch=1, enable_prefix_caching=False)


def prompt(n, seed):
    return torch.randint(0, 4000, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


# 600: a second chunk behind 512 rows
@pytest.mark.parametrize("n", [129, 143, 144, 145, 223, 400, 512, 600])
def test_a_prompt(model, n):
    ids = prompt(n, n)

    def run():
        return model.generate_one(ids, None, None, max_new_tokens=1, return_logits=True)[1].clone()

    on, off = both(run)
    assert torch.isfinite(on).all() and torch.equal(on, off)


@pytest.mark.parametrize("opts", [dict(GEMM_SK=1), dict(GEMM_SK=2), dict(GEMM_SK=6), dict(GEMM_SK=10), dict(ATTN_PLANES=0), dict(ATTN_BF16X3=0), dict(ATTN_KSPLIT=2, ATTN_BF16X3=0), dict(ROPE_FUSE=0),
                                  dict(EPI_NORM_REG=0)])
def test_every_writer(narrow, opts):
    """other splits (direct results, the epilogues behind a split), the other attention kernels and their combine"""
    ids = prompt(201, 1)
    with _lib.options(**opts):
        on, off = both(lambda: narrow.generate_one(ids, None, None, max_new_tokens=1, return_logits=True)[1].clone())
    assert torch.isfinite(on).all() and torch.equal(on, off)


def test_packed_prompts(model):
    lengths = (70, 33, 129, 5)

    def run():
        for s in range(len(lengths)):
            model.release_slot(s)
        logits = model.step_tokens([(s, prompt(n, 10 + s), [n - 1]) for s, n in enumerate(lengths)])
        return [z.clone() for z in logits]

    on, off = both(run)
    assert all(torch.isfinite(a).all() and torch.equal(a, b) for a, b in zip(on, off))


@pytest.mark.parametrize("name", ["chatts-8b", "chatts-14b"])
@pytest.mark.parametrize("patches", [64, 65, 96, 128, 129, 144, 159, 300, 1036])
@pytest.mark.parametrize("fused", [True, False])
def test_the_encoder(name, patches, fused):
    from chatts_amd.ts_encoder import TimeSeriesEmbedding
    ts = preset(name).ts
    e = TimeSeriesEmbedding(ts, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(patches)
    e.load_tensor("position_embedding.weight", torch.randn((ts["max_sequence_length"] + 1, ts["embedding_dim"]), generator=g, device="cuda"))
    k = ts["patch_size"] * (1 + ts["embedding_dim"])
    for l in range(ts["num_layers"]):
        e.load_tensor(f"mlp.{2 * l}.weight", (torch.randn((ts["hidden_size"], k), generator=g, device="cuda") * k ** -0.5).bfloat16())
        e.load_tensor(f"mlp.{2 * l}.bias", (torch.randn(ts["hidden_size"], generator=g, device="cuda") * 0.1).bfloat16())
        k = ts["hidden_size"]
    n = patches * ts["patch_size"] // 3
    lengths = [n, n, patches * ts["patch_size"] - 2 * n]
    x = torch.zeros((3, max(lengths), 2), device="cuda")
    for i, m in enumerate(lengths):
        x[i, :m, 0] = torch.randn(m, generator=g, device="cuda")
        x[i, :m, 1] = 1.0
    with _lib.options(TS_L0_FUSED=int(fused)):
        on, off = both(lambda: e(x.view(3, -1, 1), valid_lengths=lengths)[0].clone())
    assert on.shape[0] >= patches and torch.isfinite(on).all() and torch.equal(on, off)


def test_a_switch_thrown_beside_running_prompts(model):
    """PLANE_TILES changed by another thread while the layers are being enqueued: every projection reads its planes in the form in which they were written"""
    ids, stop = prompt(300, 7), threading.Event()
    lib = _lib.load()

    def run():
        return model.generate_one(ids, None, None, max_new_tokens=1, return_logits=True)[1].clone()

    want = run()

    def throw():
        while not stop.is_set():
            for v in (0, 1) * 50:
                lib.chatts_set_option(b"PLANE_TILES", v)

    t = threading.Thread(target=throw)
    t.start()
    try:
        got = [run() for _ in range(40)]
    finally:
        stop.set()
        t.join()
        lib.chatts_unset_option(b"PLANE_TILES")
    assert all(torch.equal(g, want) for g in got)


# widths that are whole K-steps of the prefill kernel and widths that are half a step more: hidden, feed-forward, both
@pytest.mark.parametrize("hidden,inter", [(288, 512), (256, 544), (288, 544), (256, 512)])
@pytest.mark.parametrize("n", [128, 129, 150])
def test_widths_that_other_kernels_take(hidden, inter, n):
    cfg = preset("chatts-8b", num_hidden_layers=3, hidden_size=hidden, intermediate_size=inter, vocab_size=4096, ts_token_start_index=4000, eos_token_id=[4003, 4002], pad_token_id=4002)
    m = ChatTSForCausalLM.from_synthetic(cfg, seed=5, max_ctx=256, max_prefill_tokens=256, max_batch=1, enable_prefix_caching=False)
    ids = prompt(n, n)
    on, off = both(lambda: m.generate_one(ids, None, None, max_new_tokens=1, return_logits=True)[1].clone())
    assert torch.isfinite(on).all() and torch.equal(on, off)


@pytest.mark.parametrize("change", ["in place", "by a view", "another tensor", "without a version"])
def test_the_encoder_follows_its_weights(change):
    """weights changed after they were loaded act on calls of any size: the copy that calls of 129 rows and more read follows"""
    from chatts_amd.ts_encoder import TimeSeriesEmbedding
    ts = dict(preset("chatts-8b").ts, hidden_size=256)
    g = torch.Generator(device="cuda").manual_seed(11)
    k = [ts["patch_size"] * (1 + ts["embedding_dim"])] + [256] * (ts["num_layers"] - 1)
    draw = lambda: [(torch.randn((256, n), generator=g, device="cuda") * n ** -0.5).bfloat16() for n in k]
    pos, bias, first, then = torch.randn((ts["max_sequence_length"] + 1, ts["embedding_dim"]), generator=g, device="cuda"), torch.randn(256, generator=g, device="cuda"), draw(), draw()

    def encoder(weights):
        e = TimeSeriesEmbedding(ts, device="cuda")
        e.load_tensor("position_embedding.weight", pos)
        for l, w in enumerate(weights):
            e.load_tensor(f"mlp.{2 * l}.weight", w)
            e.load_tensor(f"mlp.{2 * l}.bias", bias)
        return e

    def call(e, patches):
        x = torch.zeros((1, patches * ts["patch_size"], 2), device="cuda")
        x[0, :, 0], x[0, :, 1] = torch.sin(torch.arange(x.shape[1], device="cuda") * 0.1), 1.0
        return e(x.view(1, -1, 1), valid_lengths=[x.shape[1]])[0].clone()

    e, want = encoder(first), encoder([first[0]] + then[1:])
    before = call(e, 300)
    assert torch.equal(before, call(encoder(first), 300))
    for l in range(1, len(k)):
        if change == "in place":
            with torch.no_grad():
                e.weights[l].copy_(then[l])
        elif change == "by a view":
            e.weights[l].view(-1)[:] = then[l].view(-1)
        elif change == "another tensor":
            e.weights[l] = then[l].clone()
        else:
            with torch.inference_mode():
                e.weights[l] = then[l].clone()
    for patches in (300, 128, 129):
        assert torch.equal(call(e, patches), call(want, patches))
    assert not torch.equal(before, call(e, 300))
