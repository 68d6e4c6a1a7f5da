"""Patchify + first MLP layer where a workgroup walks over several column steps (csrc/ts_frontend.hip): bit-identical to the two-launch form, with column steps that
do not divide evenly, row groups with one live wave, more series than the lanes of a wave, embedding rows of one and of several eights."""
import pytest
import torch

from chatts_amd import synth
from chatts_amd.ts_encoder import TimeSeriesEmbedding

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("mode,patch,emb", [("pos_emb", 16, 16), ("pos_emb", 8, 24), ("pos_emb", 8, 8), ("pos_idx", 16, 16), ("raw", 24, 16)])
@pytest.mark.parametrize("hidden,lengths", [(5120, [1000, 64, 333, 1024, 17] * 6), (1088, [512, 100] * 40), (4096, [250] * 14), (128, [16])])
def test_walks_over_columns(monkeypatch, mode, patch, emb, hidden, lengths):
    cfg = dict(patch_size=patch, num_layers=2, hidden_size=hidden, num_features=2, max_sequence_length=2048, use_position_embedding=mode == "pos_emb",
               use_position_idx=mode == "pos_idx", embedding_dim=emb)
    enc = TimeSeriesEmbedding(cfg, device=DEV)
    enc.load_synthetic([s for s in synth.ts_encoder_specs(type("C", (), {"ts": cfg})())], 5)
    g = torch.Generator().manual_seed(hidden)
    x = torch.zeros((len(lengths), max(lengths), 2))
    for i, n in enumerate(lengths):
        x[i, :n, 0] = torch.randn(n, generator=g)
        x[i, :n, 1] = 1.0
    x = x.reshape(len(lengths), -1, 1).to(DEV)
    a = enc(x, valid_lengths=lengths)[0].clone()
    monkeypatch.setenv("CHATTS_TS_L0_FUSED", "0")
    b = enc(x, valid_lengths=lengths)[0]
    torch.cuda.synchronize()
    assert a.shape[0] == sum((n + patch - 1) // patch for n in lengths) and torch.isfinite(a).all() and torch.equal(a, b)
