"""Lengths that the host knows as arguments of the encoder's first layer (up to 64 series), against lengths that are read on the device: numbers of series around the 16 that a search takes at
once and around the 64, series of no steps at the start, in the middle and at the end of the list, masks that say other lengths than the arguments, without counts."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib, synth
from chatts_amd.ts_encoder import TimeSeriesEmbedding

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module", params=["pos_emb", "pos_idx", "raw"])
def encoder(request):
    cfg = dict(patch_size=16, num_layers=3, hidden_size=256, num_features=2, max_sequence_length=512, use_position_embedding=request.param == "pos_emb",
               use_position_idx=request.param == "pos_idx", embedding_dim=16)
    e = TimeSeriesEmbedding(cfg, device=DEV)
    e.load_synthetic([s for s in synth.ts_encoder_specs(type("C", (), {"ts": cfg})())], 5)
    return e


def encode(e, x, lengths, known, counts=True):
    lib, n, lmax = _lib.load(), len(lengths), x.shape[1]
    P, H = sum(-(-v // 16) for v in lengths), e.hidden_size
    scratch = [torch.empty((P, k), device=DEV) for k in (e.k0, H, H)]
    out, pc = torch.full((P + 1, H), 7.0, device=DEV), torch.full((n + 1,), -7, dtype=torch.int64, device=DEV)
    vl, off = torch.empty(n, dtype=torch.int32, device=DEV), torch.empty(n + 1, dtype=torch.int32, device=DEV)
    size = max(int(lib.chatts_linear_workspace(P, H, e.layer_k(l))) for l in range(e.num_layers))
    ws, st = torch.empty(max(size, 16), dtype=torch.uint8, device=DEV), _lib.stream_ptr()
    p = lambda t: t.data_ptr()
    host = (C.c_int32 * n)(*lengths)
    if known:
        _lib.check(lib.chatts_ts_encode_known(p(x), host, n, lmax, p(vl), p(off), p(pc) if counts else None, C.byref(e._tsw), e._tsw_tiled, *map(p, scratch), p(out), p(ws), size, st))
        C.memset(host, 0, C.sizeof(host))      # (the call has read them)
    else:
        _lib.check(lib.chatts_ts_lengths(host, n, 16, p(vl), p(off), p(x), lmax, p(pc), st))
        _lib.check(lib.chatts_ts_encode_tiled(p(x), p(off), p(vl), n, lmax, max(lengths), P, C.byref(e._tsw), e._tsw_tiled, *map(p, scratch), p(out), p(ws), size, st))
    torch.cuda.synchronize()
    return out, pc


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 32, 63, 64, 65, 100])
@pytest.mark.parametrize("empty", ["none", "start", "middle", "end", "all but one"])
def test_the_same_bits(encoder, n, empty):
    g, lmax = torch.Generator().manual_seed(n), 70
    lengths = torch.randint(1, lmax + 1, (n,), generator=g).tolist()
    lengths[n // 2] = lmax
    none = {"none": [], "start": range(min(2, n - 1)), "middle": range(n // 3, n // 2), "end": range(max(n - 3, n // 2 + 1), n), "all but one": [i for i in range(n) if i != n // 2]}[empty]
    for i in none:
        lengths[i] = 0
    masks = torch.randint(0, lmax + 1, (n,), generator=g)      # (other lengths than the arguments: only the counts come from them)
    x = torch.stack([torch.randn((n, lmax), generator=g), (torch.arange(lmax)[None] < masks[:, None]).float()], -1).to(DEV)
    encoder(x.view(n, -1, 1), valid_lengths=lengths)
    want, counts = encode(encoder, x, lengths, False)
    got, own = encode(encoder, x, lengths, True)
    assert torch.isfinite(want).all() and torch.equal(got, want)
    assert own.tolist() == counts.tolist() == ((masks + 15) // 16).tolist() + [-7]
    got, own = encode(encoder, x, lengths, True, counts=False)
    assert torch.equal(got, want) and own.eq(-7).all()
