"""Batched decode where the qkv projection leaves its splits to the attention (csrc/attn_decode.h): the bits of sums in a launch of their own, over the numbers of splits its instances end
at, groups of four heads with norms and of five with biases, scaled 8-bit weights; the keys and values it stores are those that the next step reads."""
import pytest
import torch

from chatts_amd import _lib
from tests.test_gpu_batched_step_rows import model_of, step

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def own_random_numbers():
    """the tests behind these draw what they would draw without them"""
    with torch.random.fork_rng():
        yield


@pytest.mark.parametrize("name,form", [("chatts-8b", "bf16"), ("chatts-14b", "bf16"), ("chatts-14b", "fp8"), ("chatts-8b", "int8")])
def test_splits_left_to_the_attention(name, form):
    m, positions, tokens = model_of(name, form)
    for splits in (2, 4, 5, 6, 8):
        got = []
        for exact, left in ((1, 1), (1, 0), (0, 1)):      # (heads counted at run time read whole rows)
            with _lib.options(GEMM_SK=splits, ATTN_EXACT=exact, SPLIT_SUMS=left):
                m.buf["qkv"].fill_(float("nan"))
                first = step(m, positions, tokens, 16)
                assert bool(torch.isnan(m.buf["qkv"][:16]).all()) == bool(exact and left), splits      # (the sums were left, or not)
                got.append((first, step(m, positions + 1, tokens.flip(0), 16)))
        assert all(torch.equal(a, b) for other in got[1:] for a, b in zip(got[0], other)), splits
