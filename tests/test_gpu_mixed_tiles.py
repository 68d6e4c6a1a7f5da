"""The first norm's planes in the prefill kernel's blocks (PLANE_TILES), decoders with norms before their sublayers and rows of 3072 columns and more: the same bits as row-major planes, for
rows that end with a whole block of 16, one row later and one row earlier, one prompt and several, at the smallest number of rows that travels so and above."""
import numpy as np
import pytest
import torch

from chatts_amd import _lib
from chatts_amd.muvetar import MuvetarConfig, MuvetarForCausalLM
from oracle import muvetar as F
from tests.muvetar_models import _gru, _moe, _par

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [3072, 4050, 4160])
def test_the_same_bits(width):
    cfg = {"vocab": 96, "width": width, "norm": {"eps": 1e-6}, "residual_mult": 0.5, "logit_softcap": 40.0,
           "layers": [_moe(_par(4, 2, 32, 32, 0.25, 64, 4, 8, 2, (1.0, 0.5)), 64, 7.0, 4, 2, 1.0, (64, 7.0)), dict(_gru(2100), mlp=None), _moe(_gru(64), 64, 7.0, 4, 2, 1.0)]}
    m = MuvetarForCausalLM(MuvetarConfig.from_dict(dict(cfg, architecture="Muvetar")), dtype="bfloat16", max_ctx=256, max_batch=2, max_prefill_tokens=512)
    m.load_weights(F.random_model(cfg, 0).items())
    rng = np.random.default_rng(1)
    for sizes in ([65], [96], [97], [111], [128], [129], [200], [100, 45], [131, 130]):
        prompts = [(s, rng.integers(0, 96, n).tolist(), list(range(n))) for s, n in enumerate(sizes)]

        def run():
            for s in range(len(sizes)):
                m.release_slot(s)
            return m.step_tokens(prompts).clone()

        on = run()
        with _lib.options(PLANE_TILES=0):
            off = run()
        assert torch.isfinite(on).all() and torch.equal(on, off), sizes
