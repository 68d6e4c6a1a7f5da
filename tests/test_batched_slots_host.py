"""Slots of the batched decode attention: by places, heads and the workspace, never by the sequences that run."""
import pytest

from chatts_amd.modeling import batched_slots


# a server's own width: enough waves where every place is taken, and enough slots for the one sequence of a server that is not
@pytest.mark.parametrize("places,nq,nkv,slots", [(1, 40, 8, 64), (2, 40, 8, 64), (3, 40, 8, 42), (4, 40, 8, 32), (5, 32, 8, 36), (6, 40, 8, 36), (7, 40, 8, 31), (8, 40, 8, 28), (10, 40, 8, 22), (14, 40, 8, 15), (16, 40, 8, 14), (32, 40, 8, 12),
                                                 (8, 64, 8, 16), (16, 64, 8, 8), (32, 56, 8, 8)])
def test_a_whole_model(places, nq, nkv, slots):
    assert batched_slots(places, nq, nkv, 64) == slots


# a shard of fewer kv heads has as many waves as the whole model
@pytest.mark.parametrize("places,nq,nkv,slots", [(5, 20, 4, 51), (8, 20, 4, 32), (8, 10, 2, 64), (8, 5, 1, 64), (16, 20, 4, 16), (16, 10, 2, 32), (16, 5, 1, 64), (32, 5, 1, 32), (16, 8, 1, 64)])
def test_a_shard(places, nq, nkv, slots):
    assert batched_slots(places, nq, nkv, 64) == slots


def test_never_more_than_the_workspace_holds():
    assert [batched_slots(b, 40, 8, 4) for b in (1, 4, 16, 64)] == [4] * 4 and batched_slots(1, 1, 1, 1) == 1
