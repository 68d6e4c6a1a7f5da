"""The forms of the prefill attention on K / V planes: 32 or 64 queries and two parts of the keys, 64 or 128 queries and one part, chosen by how the workgroups fill the CUs."""
import ctypes as C

import pytest
import torch

from chatts_amd import _lib
from chatts_amd.config import preset
from chatts_amd.modeling import ChatTSForCausalLM

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def _reference(q, k, v, pos0):
    """float64, one head at a time"""
    T, nq, _ = q.shape
    n, group = pos0 + T, nq // k.shape[0]
    hidden = torch.arange(n, device=DEV)[None, :] > (pos0 + torch.arange(T, device=DEV))[:, None]
    out = torch.empty((T, nq, 128), dtype=torch.float64, device=DEV)
    for h in range(nq):
        s = (q[:, h].double() @ k[h // group, :n].double().T.contiguous()) * 128 ** -0.5
        s.masked_fill_(hidden, float("-inf"))
        out[:, h] = torch.softmax(s, -1) @ v[h // group, :n].double()
    return out


# on 256 CUs: two waves of queries and two parts; four and two; four and one; four of 32 queries.  First and last tiles whole, one row, one row short; parts with one tile more than the other and without any
@pytest.mark.parametrize("nq,nkv,T,pos0", [
    (10, 2, 64, 0), (10, 2, 65, 0), (32, 8, 95, 0), (32, 8, 256, 0), (8, 8, 97, 31), (5, 1, 129, 700), (28, 4, 64, 1),
    (32, 8, 257, 0), (40, 8, 200, 33), (40, 8, 511, 0), (12, 12, 705, 2),
    (40, 8, 806, 0), (40, 8, 769, 100), (64, 8, 575, 31), (24, 3, 1409, 0),
    (40, 8, 2049, 0), (64, 8, 1407, 0), (32, 8, 1472, 2047)])
def test_every_form(lib, nq, nkv, T, pos0):
    """Against float64.  A product of split operands is off by 2^-18 of each factor and the dropped lo x lo: 4e-6 of a score's scale (rms), and P and V bring 2e-6 each, so 5e-6 of the
    output's norm; four times that is allowed."""
    ctx = pos0 + T + 5
    g = torch.Generator(device=DEV).manual_seed(T + pos0 + nq)
    qkv = torch.randn((T, (nq + 2 * nkv) * 128), generator=g, device=DEV)
    k = torch.randn((nkv, ctx, 128), generator=g, device=DEV)
    v = torch.randn((nkv, ctx, 128), generator=g, device=DEV)
    k[:, 40] *= 4.0                          # a key of the second tile that outweighs the others: the parts' maxima differ
    want = _reference(qkv.view(T, nq + 2 * nkv, 128)[:, :nq], k, v, pos0)
    k[:, pos0 + T:] = float("nan")           # rows past the context are not read
    v[:, pos0 + T:] = float("nan")
    qkv[T // 2, 128:256] = float("nan")      # a query without a score: only its own row
    cache = _lib.KvCache(k=k.data_ptr(), v=v.data_ptr(), max_ctx=ctx)
    ws = torch.empty(((pos0 + T + 31) // 32) * nkv * 32768, dtype=torch.uint8, device=DEV)
    out = torch.zeros((T, nq * 128), device=DEV)
    _lib.check(lib.chatts_attention(qkv.data_ptr(), T, nq, nkv, pos0, None, C.byref(cache), out.data_ptr(), 1, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    got = out.view(T, nq, 128).double()
    assert got[T // 2, 1].isnan().all()
    got[T // 2, 1] = want[T // 2, 1]
    assert ((got - want).norm() / want.norm()).item() < 2e-5
    assert (got - want).abs().max().item() < 2e-5 * want.abs().max().item()


# rows that are not rotated yet, planes that a projection's epilogue has written: what chose them for this path stays chosen, also when an option changes beside the call
@pytest.mark.parametrize("option,value", [("ATTN_PLANES", 0), ("ATTN_BF16X3", 0), ("ATTN_ROWS", 1)])
@pytest.mark.parametrize("written", [False, True])
def test_the_path_is_chosen_once(lib, option, value, written):
    attend, prepare = (getattr(lib, n) for n in ("_ZN6chatts14attention_implEPKfiiiiPKiPK13ChattsKvCachePfPtS8_iPvmS9_iPKNS_8RopeFuseEPKt",
                                                 "_ZN6chatts17rope_fuse_prepareEiiiPKfS1_fS1_S1_iPKiPK13ChattsKvCachePNS_8RopeFuseE"))
    P, I, F, N = C.c_void_p, C.c_int, C.c_float, C.c_size_t
    attend.argtypes, prepare.argtypes = [P, I, I, I, I, P, P, P, P, P, I, P, N, P, I, P, P], [I, I, I, P, P, F, P, P, I, P, P, P]
    nq, nkv, T, pos0 = 8, 2, 96, 33
    ctx = pos0 + T
    g = torch.Generator(device=DEV).manual_seed(1)
    raw, k0, v0 = (torch.randn(s, generator=g, device=DEV) for s in ((T, (nq + 2 * nkv) * 128), (nkv, ctx, 128), (nkv, ctx, 128)))
    turn = torch.rand((ctx, 64), generator=g, device=DEV) * 6.0
    cos, sin = turn.cos().contiguous(), turn.sin().contiguous()
    ws = torch.zeros(((ctx + 31) // 32) * nkv * 32768, dtype=torch.uint8, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream

    def run(**options):
        qkv, k, v, out = raw.clone(), k0.clone(), v0.clone(), torch.zeros((T, nq * 128), device=DEV)
        cache = _lib.KvCache(k=k.data_ptr(), v=v.data_ptr(), max_ctx=ctx)
        rope = (C.c_char * 512)()
        _lib.check(prepare(T, nq, nkv, None, None, 1e-6, cos.data_ptr(), sin.data_ptr(), pos0, None, C.byref(cache), rope))
        if written:
            _lib.check(lib.chatts_rope_kv_write(qkv.data_ptr(), T, nq, nkv, None, None, 1e-6, cos.data_ptr(), sin.data_ptr(), pos0, None, C.byref(cache), stream))
            _lib.check(lib.chatts_attention(qkv.data_ptr(), T, nq, nkv, pos0, None, C.byref(cache), out.data_ptr(), 1, ws.data_ptr(), ws.numel(), stream))
            out.zero_()
        with _lib.options(**options):
            _lib.check(attend(qkv.data_ptr(), T, nq, nkv, pos0, None, C.byref(cache), out.data_ptr(), None, None, 1, ws.data_ptr(), ws.numel(), stream, 0, None if written else rope,
                              ws.data_ptr() if written else None))
        return out, k, v

    want, got = run(), run(**{option: value})
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and not torch.equal(want[1], k0) and want[0].abs().max() > 0.01


@pytest.fixture(scope="module", params=["chatts-8b", "chatts-14b"])
def model(request):
    cfg = preset(request.param, num_hidden_layers=2, vocab_size=4096, ts_token_start_index=4000, eos_token_id=[4003, 4002], pad_token_id=4002)
    return ChatTSForCausalLM.from_synthetic(cfg, seed=3, max_ctx=1024, max_prefill_tokens=512, max_batch=2, enable_prefix_caching=False)


# portions that end inside a tile, at its end and one row behind it, the first of a prompt and later ones, two prompts at once
@pytest.mark.parametrize("portions", [[64], [65, 96], [77, 223], [300, 64, 97], [512, 31, 481]])
def test_rotation_in_the_planes_writer(model, portions):
    """ROPE_FUSE=0 rotates all heads in a launch of its own.  Keys and values are the same bits, and without a norm of the queries everything is.  That norm adds its squares in another order: a
    last bit of a query, which its split (2^-18) does not always keep."""
    ids = torch.randint(0, 4000, (sum(portions) + 70,), generator=torch.Generator().manual_seed(len(portions))).tolist()

    def run():
        at = 0
        for i, n in enumerate(portions):
            rows = [(0, ids[at:at + n], [n - 1])]
            if i == 0:
                rows.append((1, ids[:70], [69]))
            got = model.step_tokens(rows)[0].clone()
            at += n
        model.release_slot(0)
        model.release_slot(1)
        return got

    same_bits(model, run, model.config.model_type == "qwen2")


# a second chunk behind 512 rows: of 88, of 31 (too few for planes), of 481; split 1: the projection's own rows, 3: its split's epilogue, which rotates the queries, too
@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("n", [64, 65, 96, 127, 223, 512, 543, 600, 993])
def test_rotation_behind_a_chunks_projection(model, n, split):
    ids = torch.randint(0, 4000, (n,), generator=torch.Generator().manual_seed(n)).tolist()
    with _lib.options(GEMM_SK=split):
        same_bits(model, lambda: model.generate_one(ids, None, None, max_new_tokens=1, return_logits=True)[1].clone(), split > 1 or model.config.model_type == "qwen2")


def same_bits(model, run, exactly):
    fused = run()
    with _lib.options(ROPE_FUSE=0):
        apart = run()
    assert torch.isfinite(fused).all()
    assert torch.equal(fused, apart) if exactly else ((fused - apart).norm() / apart.norm()).item() < 2e-5
