"""Biases of a mixed decoder that are not 16-byte aligned, which a caller of the C interface may hand over: batches of 17 .. 95 rows keep the kernels that take them."""
import pytest
import torch

from chatts_amd import _lib
from chatts_amd.muvetar import MuvetarConfig, MuvetarForCausalLM
from oracle import muvetar as F

pytestmark = pytest.mark.gpu


class Shifted(MuvetarForCausalLM):
    by = 0

    def _blocks(self, L, blocks, split=False, bias=None):
        off = super()._blocks(L, blocks, split, bias)
        if bias:
            b = next(t for t in self._keep if t.data_ptr() == L.in_bias)
            L.in_bias = self._dev(torch.cat([torch.zeros(self.by, device=b.device), b])) + 4 * self.by
        return off


# (8256 columns: above 8192 the prefill kernel runs from 65 rows on, whose stores want an aligned bias)
# planes hold a value to 2^-17: the two forms are 1e-5 apart
@pytest.mark.parametrize("n", [17, 64, 65, 95])
def test_the_bias_is_taken(n):
    cfg = {"vocab": 96, "width": 1024, "norm": {"eps": 1e-5}, "residual_mult": 0.6, "logit_softcap": 20.0, "layers": [{"type": "mingru", "mixer": {"width": 2752}, "mlp": None}]}
    sd = F.random_model(cfg, 3)
    toks = torch.randint(0, 96, (n,), generator=torch.Generator().manual_seed(n)).tolist()

    def run(by):
        m = type("By%d" % by, (Shifted,), dict(by=by))(MuvetarConfig.from_dict(dict(cfg, architecture="Muvetar")), dtype="bfloat16", max_ctx=128, max_batch=1)
        m.load_weights(sd.items())
        return m.step_tokens([(0, toks, list(range(n)))]).double().cpu()

    want = F.forward(cfg, sd, toks).double()
    for by in (0, 1):
        assert float((run(by) - want).norm() / want.norm()) < 5e-5, by
