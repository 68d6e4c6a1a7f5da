"""Lengths from the masks where a series is no whole number of the 512 steps that a wave asks for at once."""
import pytest
import torch

from chatts_amd.ts_encoder import TimeSeriesEmbedding

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lmax", [1, 63, 64, 65, 511, 512, 513, 1100])
def test_lengths(lmax):
    cfg = dict(patch_size=16, num_layers=2, hidden_size=64, num_features=2, max_sequence_length=2048, use_position_embedding=True, embedding_dim=16)
    g = torch.Generator().manual_seed(lmax)
    mask = (torch.rand((9, lmax), generator=g) < 0.7).float() * 1.5      # (truncated to 1)
    mask[0], mask[1] = 1.0, 0.0
    x = torch.stack([torch.randn((9, lmax), generator=g), mask], -1).reshape(9, -1, 1).cuda()
    vl, pc = TimeSeriesEmbedding(cfg, device="cuda").get_patch_cnt(x)
    want = mask.long().sum(1)
    assert vl.tolist() == want.tolist() and pc.tolist() == ((want + 15) // 16).tolist()
