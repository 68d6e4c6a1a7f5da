"""The feed-forward beside experts in their launches (up to 16 rows) and in launches of its own (from 17): whole prompts of either side of the line, and of a single row, against the
plain references, with the tolerances of the models' own tests."""
import pytest

from tests import test_gpu_mefurax as mefurax
from tests import test_gpu_muvetar as muvetar

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("module,name", [(m, n) for m in (muvetar, mefurax) for n in sorted(m.CONFIGS)], ids=lambda v: v if isinstance(v, str) else v.__name__.rsplit("_", 1)[-1])
def test_prompts_on_both_sides_of_sixteen_rows(module, name):
    m = module.load(name, "bfloat16", max_ctx=256, max_batch=2)
    for n in (1, 2, 15, 16, 17):
        toks = module.tokens(name, n, n)
        got = m.step_tokens([(n % 2, toks, list(range(n)))])
        assert module.worst(got, module.want(name, toks, "bfloat16")) < module.TOL[(name, "bfloat16")], n
        m.release_slot(n % 2)
