"""Chunks of 17 .. 128 rows on planes, at the rows where the kernels change (weight stream up to 64 rows, and up to 128 where the result has 8192 columns at most; else the prefill
kernel): against the same rows in portions of 16 and fewer, which run the weight stream of batched steps."""
import pytest
import torch

from chatts_amd import _lib
from chatts_amd.config import preset
from chatts_amd.modeling import ChatTSForCausalLM
from chatts_amd.ts_encoder import TimeSeriesEmbedding

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


# the last: rows that the float32 path takes (K below 1024) beside a projection of 1088 values on planes
@pytest.fixture(scope="module", params=[("chatts-8b", {}), ("chatts-14b", {}), ("chatts-8b", dict(hidden_size=512, intermediate_size=1088))], ids=["8b", "14b", "narrow"])
def models(request):
    name, sizes = request.param
    cfg = preset(name, num_hidden_layers=2, vocab_size=4096, ts_token_start_index=4000, eos_token_id=[4003, 4002], pad_token_id=4002, **sizes)
    whole, parts = (ChatTSForCausalLM.from_synthetic(cfg, seed=6, max_ctx=512, max_prefill_tokens=n, max_batch=2, enable_prefix_caching=False) for n in (256, 16))
    return whole, parts


# Both sides hold activations as two bf16 parts (2^-17 of a value) and drop the product of the low parts in attention (2^-16 of a term), rounded at other places: 2e-5 a layer, 4e-5 for two.
@pytest.mark.parametrize("n", [17, 31, 33, 63, 64, 65, 80, 95, 96, 127, 128, 129])
def test_a_chunk_and_its_portions(models, n):
    whole, parts = models
    ids = torch.randint(0, 4000, (n,), generator=torch.Generator().manual_seed(n)).tolist()
    run = lambda m: m.generate_one(ids, None, None, max_new_tokens=1, return_logits=True)[1].clone()
    got, want = run(whole), run(parts)
    assert torch.isfinite(got).all() and rel(got, want) < 4e-5
    with _lib.options(PLANE_TILES=0):
        assert torch.equal(run(whole), got)


def test_packed_chunks(models):
    whole, parts = models
    prompts = [torch.randint(0, 4000, (n,), generator=torch.Generator().manual_seed(n)).tolist() for n in (40, 29)]
    got = [z.clone() for z in whole.step_tokens([(s, ids, [len(ids) - 1]) for s, ids in enumerate(prompts)])]
    for ids, z in zip(prompts, got):
        assert rel(z.view(-1), parts.generate_one(ids, None, None, max_new_tokens=1, return_logits=True)[1].view(-1)) < 4e-5


# 32-bit sums of 5120 products in another order: a few 1e-7 of a layer's result, five layers
@pytest.mark.parametrize("name", ["chatts-8b", "chatts-14b"])
@pytest.mark.parametrize("patches", [65, 79, 80, 96, 127, 128])
def test_the_encoder_and_its_series_alone(name, patches):
    ts = preset(name).ts
    e = TimeSeriesEmbedding(ts, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(patches)
    e.load_tensor("position_embedding.weight", torch.randn((ts["max_sequence_length"] + 1, ts["embedding_dim"]), generator=g, device="cuda"))
    k = ts["patch_size"] * (1 + ts["embedding_dim"])
    for l in range(ts["num_layers"]):
        e.load_tensor(f"mlp.{2 * l}.weight", (torch.randn((ts["hidden_size"], k), generator=g, device="cuda") * k ** -0.5).bfloat16())
        e.load_tensor(f"mlp.{2 * l}.bias", (torch.randn(ts["hidden_size"], generator=g, device="cuda") * 0.1).bfloat16())
        k = ts["hidden_size"]
    lengths = [60 * 16, (patches - 60) * 16 - 3]
    x = torch.zeros((2, max(lengths), 2), device="cuda")
    for i, n in enumerate(lengths):
        x[i, :n, 0] = torch.randn(n, generator=g, device="cuda")
        x[i, :n, 1] = 1.0
    got = e(x.view(2, -1, 1), valid_lengths=lengths)[0].clone()
    want = torch.cat([e(x[i:i + 1].view(1, -1, 1), valid_lengths=[n])[0].clone() for i, n in enumerate(lengths)])
    assert got.shape == want.shape and got.shape[0] == patches and rel(got, want) < 5e-6


# where the weight stream's workgroups fill the CUs (32 x 8, 36 x 7) or three quarters of them at most (18 x 9), it runs whether the weights lie in tiles or not; where they leave some idle (24 x 10,
# 40 x 6, 52 x 4 of 256), weights in tiles are the prefill kernel's, whose sums run in another order
@pytest.mark.parametrize("width,prefill_kernel", [(2304, False), (3072, True), (4096, False), (4608, False), (5120, True), (6656, True)])
def test_which_kernel_an_encoder_of_some_rows_takes(width, prefill_kernel):
    ts = dict(preset("chatts-8b").ts, hidden_size=width, num_layers=3)
    e = TimeSeriesEmbedding(ts, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(width)
    e.load_tensor("position_embedding.weight", torch.randn((ts["max_sequence_length"] + 1, ts["embedding_dim"]), generator=g, device="cuda"))
    k = ts["patch_size"] * (1 + ts["embedding_dim"])
    for l in range(3):
        e.load_tensor(f"mlp.{2 * l}.weight", (torch.randn((width, k), generator=g, device="cuda") * k ** -0.5).bfloat16())
        e.load_tensor(f"mlp.{2 * l}.bias", torch.randn(width, generator=g, device="cuda") * 0.1)
        k = width
    for patches in (65, 100, 128):
        x = torch.randn((1, patches * 16, 2), generator=g, device="cuda")
        x[..., 1] = 1.0
        rows = e(x.view(1, -1, 1), valid_lengths=[patches * 16])[0].clone()
        e._tsw_tiled = None
        plain = e.replay_last().clone()
        e._tsw = None
        assert rel(rows, plain) < 5e-6 and torch.equal(rows, plain) != prefill_kernel, patches
