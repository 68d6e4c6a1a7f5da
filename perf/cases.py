"""The cases that speed is measured on: the work that a program using this framework has it do, through the calls such a program makes.

  encode         time series of one request -> embedding rows (TimeSeriesEmbedding)
  prompt         one request of text and time series -> its first token: encoder, embeddings, prefill, logits, choice (generate_one)
  decode         one more token for every running sequence (decode_step for one, batched_step for several)
  mixed_prompt   prompts of a design of mixed layers, whole, as one ragged batch (step_tokens)
  mixed_decode   one more token for every running sequence of such a design (batched_step)

Weights are random, of the published shapes, in full depth for the ChatTS models; a design of mixed layers has eight layers.  Muvetar stands
for these designs: it shares MixedDecoder, windowed attention, experts and the projections with the others.
"""
import math
import random
import zlib

import torch

# ---- the models -----------------------------------------------------------------------------------------------------------------------
# widths, depths and heads of the two ChatTS decoders
CHATTS = {
    "chatts-14b": dict(width=5120, ff=13824, layers=48, heads=40, kv=8, dim=128, vocab=152064, bias=True, qk_norm=False),
    "chatts-8b": dict(width=4096, ff=12288, layers=36, heads=32, kv=8, dim=128, vocab=151936, bias=False, qk_norm=True),
}
EPS, THETA = 1e-6, 1e6
PATCH, EMB, MAX_SERIES, TS_LAYERS = 16, 16, 8192, 5
TS_TOKEN = 151665                     # <ts>; <ts/> is the next one
BYTES_PER_WEIGHT = {"bf16": 2.0, "fp8": 1.0, "int8": 1.0, "int4": 0.5 + 8 / 128}      # (int4: a scale and a zero point for 128 codes)
MAX_CTX, LONG_CTX = 2048, 4096
# Muvetar sizes: width, experts' and shared feed-forward of every layer, heads
MIXED = {"muvetar-s": (2048, 768, 3072, 16), "muvetar-m": (4096, 1536, 6144, 32)}
MIXED_LAYERS, MIXED_VOCAB, EXPERTS, TOP, KV_HEADS, STATES, TAPS, LIMIT, CAP, MULT, SIDE = 8, 32000, 32, 4, 8, 16, 4, 7.0, 30.0, 0.5, 0.7
SLOPE = 1.702


def listed():
    return [
        # one short series with a question: the smallest call, launches and latency
        dict(name="encode-1x256", path="encode", model="chatts-8b", series=1, length=256, known=True),
        # eight series of a metrics dashboard, the usual request
        dict(name="encode-8x256", path="encode", model="chatts-14b", series=8, length=256, known=True),
        # thirty series of 64 to 1024 steps, ragged ends; lengths read from the masks
        dict(name="encode-30-mixed", path="encode", model="chatts-14b", series=30, length=0, known=False),
        # time to the first token: a short question on one series, the usual request, the longest one
        dict(name="prompt-8b-1x256", path="prompt", model="chatts-8b", series=1, length=256, text=207),
        dict(name="prompt-14b-8x256", path="prompt", model="chatts-14b", series=8, length=256, text=670),
        dict(name="prompt-14b-30-mixed", path="prompt", model="chatts-14b", series=30, length=0, text=2500),
        # an answer that streams to one reader
        dict(name="decode-8b", path="decode", model="chatts-8b", weights="bf16", batch=1, context=223),
        # the published GPTQ-Int4 format, one reader
        dict(name="decode-14b-int4", path="decode", model="chatts-14b", weights="int4", batch=1, context=798),
        # a server with a few and with sixteen requests under way
        dict(name="decode-8b-x5", path="decode", model="chatts-8b", weights="bf16", batch=5, context=801),
        dict(name="decode-14b-fp8-x16", path="decode", model="chatts-14b", weights="fp8", batch=16, context=1204),
        # a design of mixed layers: a long prompt, and sixteen sequences under way
        dict(name="muvetar-prompt", path="mixed_prompt", model="muvetar-m", prompts=1, tokens=2048),
        dict(name="muvetar-decode-x16", path="mixed_decode", model="muvetar-s", batch=16, context=500),
    ]


def _spread(rng, low, high):
    """a whole number, its logarithm uniform"""
    return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))


def draw(rng):
    path = rng.choice(["encode", "encode", "prompt", "prompt", "decode", "decode", "mixed_prompt", "mixed_decode"])
    model = rng.choice(sorted(CHATTS))
    if path == "encode":
        return dict(path=path, model=model, series=_spread(rng, 1, 30), length=_spread(rng, 17, 1024), known=rng.random() < 0.5)
    if path == "prompt":
        return dict(path=path, model=model, series=_spread(rng, 1, 16), length=_spread(rng, 17, 512), text=_spread(rng, 40, 2000))
    if path == "decode":
        return dict(path=path, model=model, weights=rng.choice(["bf16", "bf16", "fp8", "int8", "int4"]), batch=_spread(rng, 1, 16), context=_spread(rng, 40, 1900))
    model = rng.choice(sorted(MIXED))
    if path == "mixed_prompt":
        return dict(path=path, model=model, prompts=rng.randint(1, 4), tokens=_spread(rng, 65, 2048))
    return dict(path=path, model=model, batch=_spread(rng, 1, 16), context=_spread(rng, 40, 1000))


# ---- inputs ---------------------------------------------------------------------------------------------------------------------------
def _tensor(name, shape, seed, scale, mean=0.0, dtype=torch.bfloat16):
    """a tensor that its name and the seed define: normal values"""
    gen = torch.Generator(device="cuda").manual_seed((zlib.crc32(name.encode()) << 24) + seed)
    t = torch.empty(shape, dtype=dtype, device="cuda").normal_(generator=gen)
    return t.mul_(scale).add_(mean) if mean else t.mul_(scale)


def _lengths(case):
    if case["length"]:
        return [case["length"]] * case["series"]
    r = random.Random(case["series"])                  # 64 .. 1024 steps, two with ends that fill no patch
    lengths = [r.randint(64, 1024) for _ in range(case["series"])]
    lengths[3 % len(lengths)], lengths[17 % len(lengths)] = 1000, 65
    return lengths


def _patches(case):
    return [-(-n // PATCH) for n in _lengths(case)]


def _series(case, seed):
    """[series, 2 x longest, 1] (value, mask) in turn: random walks, centred, within -3 .. 3"""
    lengths = _lengths(case)
    gen = torch.Generator(device="cuda").manual_seed(seed + 5)
    x = torch.zeros((len(lengths), max(lengths), 2), device="cuda")
    for i, n in enumerate(lengths):
        walk = torch.randn(n, generator=gen, device="cuda").cumsum(0)
        walk = walk - walk.mean()
        x[i, :n, 0] = walk * (3.0 / walk.abs().max().clamp_min(1e-6))
        x[i, :n, 1] = 1.0
    return x.view(len(lengths), -1, 1)


def _ids(n, seed, vocab):
    gen = torch.Generator().manual_seed(seed)
    return torch.randint(0, min(vocab, 151000), (n,), generator=gen).tolist()


def _request(case, seed):
    """token ids with a <ts><ts/> pair per series, spread over the text"""
    n, text = case["series"], _ids(case["text"], seed + 7, 151000)
    ids, step = [], max(1, len(text) // (n + 1))
    for i in range(n):
        ids += text[i * step:(i + 1) * step] + [TS_TOKEN, TS_TOKEN + 1]
    return ids + text[n * step:]


def _contexts(case):
    """tokens that each sequence holds: a few apart"""
    return [max(16, case["context"] - 13 * i) for i in range(case["batch"])]


def _encoder_tensors(m, seed):
    yield "position_embedding.weight", _tensor("pe", (MAX_SERIES + 1, EMB), seed, 1.0, dtype=torch.float32)
    k = PATCH * (1 + EMB)
    for l in range(TS_LAYERS):
        yield f"mlp.{2 * l}.weight", _tensor(f"ts{l}.w", (m["width"], k), seed, 1.4 * k ** -0.5)
        yield f"mlp.{2 * l}.bias", _tensor(f"ts{l}.b", (m["width"],), seed, 0.1)
        k = m["width"]


def _layer_tensors(m, l, seed):
    """HF name -> tensor of one decoder layer"""
    W, p = m["width"], f"model.layers.{l}."
    t = {}
    for n, rows in (("q", m["heads"] * m["dim"]), ("k", m["kv"] * m["dim"]), ("v", m["kv"] * m["dim"])):
        t[p + f"self_attn.{n}_proj.weight"] = _tensor(p + n, (rows, W), seed, 0.02)
        if m["bias"]:
            t[p + f"self_attn.{n}_proj.bias"] = _tensor(p + n + "b", (rows,), seed, 0.1)
        if m["qk_norm"] and n != "v":
            t[p + f"self_attn.{n}_norm.weight"] = _tensor(p + n + "n", (m["dim"],), seed, 0.1, 1.0)
    t[p + "self_attn.o_proj.weight"] = _tensor(p + "o", (W, m["heads"] * m["dim"]), seed, 0.02)
    for n, shape in (("gate", (m["ff"], W)), ("up", (m["ff"], W)), ("down", (W, m["ff"]))):
        t[p + f"mlp.{n}_proj.weight"] = _tensor(p + n, shape, seed, 0.02)
    for n in ("input", "post_attention"):
        t[p + n + "_layernorm.weight"] = _tensor(p + n, (W,), seed, 0.1, 1.0)
    return t


def _ends(m, seed):
    return {"model.embed_tokens.weight": _tensor("embed", (m["vocab"], m["width"]), seed, 0.05), "model.norm.weight": _tensor("norm", (m["width"],), seed, 0.1, 1.0),
            "lm_head.weight": _tensor("head", (m["vocab"], m["width"]), seed, 0.02)}


def _mixed_config(case):
    W, ff, shared, heads = MIXED[case["model"]]
    moe = {"kind": "moe", "expert": {"ff": ff, "limit": LIMIT}, "router": {"experts": EXPERTS, "top": TOP, "scale": 1.0}, "shared": {"ff": shared, "limit": LIMIT}}
    both = {"type": "parallel", "mlp": moe,
            "mixer": {"left": {"heads": heads, "kv_heads": KV_HEADS, "dim": 128, "vdim": 128, "scale": 128 ** -0.5},
                      "right": {"inner": 2 * W, "state": STATES, "dt_rank": W // 16, "conv": TAPS}, "left_scale": SIDE, "right_scale": SIDE}}
    gru = {"type": "mingru", "mixer": {"width": W}, "mlp": moe}
    return dict(vocab=MIXED_VOCAB, width=W, layers=[both if i % 2 == 0 else gru for i in range(MIXED_LAYERS)], norm={"eps": 1e-5}, residual_mult=MULT, logit_softcap=CAP)


def _mixed_layer(case, i, seed):
    """name -> tensor of one layer"""
    W, ff, shared, heads = MIXED[case["model"]]
    p, t = f"l{i}.", {}

    def lin(name, rows, cols, gain=1.0):
        t[p + name] = _tensor(p + name, (rows, cols), seed, gain * cols ** -0.5)

    def vec(name, shape, scale, mean=0.0):
        t[p + name] = _tensor(p + name, shape, seed, scale, mean)

    vec("norm1", (W,), 0.1, 1.0)
    vec("norm2", (W,), 0.1, 1.0)
    vec("dwa", (i + 2,), 0.1, 1.0 / (i + 2))
    if i % 2:
        for n in "zxg":
            lin("mix." + n, W, W)
        vec("mix.z.b", (W,), 1.0)
        vec("mix.x.b", (W,), 0.3)
        lin("mix.o", W, W)
    else:
        C, R = 2 * W, W // 16
        lin("mix.left.q", heads * 128, W)
        lin("mix.left.k", KV_HEADS * 128, W)
        lin("mix.left.v", KV_HEADS * 128, W)
        vec("mix.left.r1", (heads,), 0.1, 0.5)
        vec("mix.left.r2", (heads,), 0.05, 0.4)
        lin("mix.left.o", W, heads * 128)
        lin("mix.right.in", 2 * C, W)
        vec("mix.right.conv", (C, TAPS), 0.5)
        vec("mix.right.conv.b", (C,), 0.2)
        lin("mix.right.x", R + 2 * STATES, C, 2.0)
        lin("mix.right.dt", C, R)
        vec("mix.right.dt.b", (C,), 0.5, -3.0)
        vec("mix.right.A_log", (C, STATES), 1.0)
        vec("mix.right.D", (C,), 0.2, 0.8)
        lin("mix.right.o", W, C)
    lin("mlp.router", EXPERTS, W, 2.0)
    for n, f in [(f"e{e}", ff) for e in range(EXPERTS)] + [("shared", shared)]:
        lin(f"mlp.{n}.gate", f, W)
        lin(f"mlp.{n}.up", f, W)
        lin(f"mlp.{n}.down", W, f)
    return t


def _mixed_ends(case, seed):
    W = MIXED[case["model"]][0]
    return {"embed": _tensor("embed", (MIXED_VOCAB, W), seed, 1.0), "final.norm": _tensor("final", (W,), seed, 0.1, 1.0),
            "head": _tensor("head", (MIXED_VOCAB, W), seed, W ** -0.5)}


def _prompts(case, seed):
    """unequal prompts that share `tokens`"""
    n, T = case["prompts"], case["tokens"]
    sizes = [max(1, T * (2 * i + 1) // (n * n)) for i in range(n)]
    return [_ids(s, seed + 100 * i, MIXED_VOCAB) for i, s in enumerate(sizes)]


def _load_chatts(case, seed, **options):
    from chatts_amd.config import preset
    from chatts_amd.modeling import ChatTSForCausalLM
    m = CHATTS[case["model"]]
    model = ChatTSForCausalLM(preset(case["model"]), device="cuda", **options)

    def pairs():
        yield from _ends(m, seed).items()
        for n, t in _encoder_tensors(m, seed):
            yield "ts_encoder." + n, t
        for l in range(m["layers"]):
            yield from _layer_tensors(m, l, seed).items()

    model.load_weights(pairs())
    return model


def prepare(case, seed):
    path = case["path"]
    if path == "encode":
        from chatts_amd.config import preset
        from chatts_amd.ts_encoder import TimeSeriesEmbedding
        encoder = TimeSeriesEmbedding(preset(case["model"]).ts, device="cuda")
        for n, t in _encoder_tensors(CHATTS[case["model"]], seed):
            encoder.load_tensor(n, t)
        return dict(path=path, encoder=encoder, series=_series(case, seed), lengths=_lengths(case) if case["known"] else None)
    if path == "prompt":
        # (the same request comes again and again here: without prefix reuse, which would skip it)
        rows = case["text"] + sum(_patches(case))
        model = _load_chatts(case, seed, max_ctx=MAX_CTX if rows < MAX_CTX else LONG_CTX, enable_prefix_caching=False)
        return dict(path=path, model=model, ids=_request(case, seed), series=_series(case, seed), lengths=_lengths(case))
    if path == "decode":
        model = _load_chatts(case, seed, max_ctx=MAX_CTX, max_batch=case["batch"], weight_format=case["weights"])
        contexts, vocab = _contexts(case), CHATTS[case["model"]]["vocab"]
        model.step_tokens([(s, _ids(n, seed + 100 * s, vocab), []) for s, n in enumerate(contexts)])
        tokens = _ids(case["batch"], seed + 3, vocab)
        state = dict(path=path, model=model, tokens=torch.tensor(tokens, device="cuda"), positions=torch.tensor(contexts, dtype=torch.int32, device="cuda"))
        if case["batch"] == 1:
            state["x"] = model.get_input_embeddings(torch.tensor(tokens))
        run(state)                                      # the step is captured when it first runs
        return state
    from chatts_amd.muvetar import MuvetarConfig, MuvetarForCausalLM
    config = MuvetarConfig(**_mixed_config(case))
    sizes = dict(max_ctx=MAX_CTX + 64, max_prefill_tokens=MAX_CTX, max_batch=case["prompts"]) if path == "mixed_prompt" else \
        dict(max_ctx=4 * MAX_CTX, max_prefill_tokens=MAX_CTX, max_batch=case["batch"])
    model = MuvetarForCausalLM(config, device="cuda", **sizes)

    def pairs():
        yield from _mixed_ends(case, seed).items()
        for i in range(MIXED_LAYERS):
            yield from _mixed_layer(case, i, seed).items()

    model.load_weights(pairs())
    if path == "mixed_prompt":
        return dict(path=path, model=model, prompts=_prompts(case, seed))
    contexts = _contexts(case)
    for s, n in enumerate(contexts):
        model.step_tokens([(s, _ids(n, seed + 100 * s, MIXED_VOCAB), [])])
        model.reserve_kv(s, 4 * MAX_CTX - 8)
    model.buf["pos_all"].copy_(torch.tensor(contexts, dtype=torch.int32))
    model.buf["token_all"].copy_(torch.tensor(_ids(case["batch"], seed + 3, MIXED_VOCAB)))
    model.batched_step()                                # the step is captured when it first runs; a state goes on from here
    model.buf["token_all"].copy_(torch.tensor(_ids(case["batch"], seed + 4, MIXED_VOCAB)))
    return dict(path=path, model=model)


def run(state):
    path = state["path"]
    if path == "encode":
        rows, counts = state["encoder"](state["series"], valid_lengths=state["lengths"])
        return {"rows": rows, "counts": counts}
    model = state["model"]
    if path == "prompt":
        tokens, logits = model.generate_one(state["ids"], state["series"], state["lengths"], max_new_tokens=1, return_logits=True)
        return {"logits": [logits], "tokens": tokens}
    if path == "mixed_prompt":
        for s in range(len(state["prompts"])):
            model.release_slot(s)
        logits = model.step_tokens([(s, ids, [len(ids) - 1]) for s, ids in enumerate(state["prompts"])])
        return {"logits": list(logits), "tokens": []}
    b = model.buf
    if path == "mixed_decode":                          # (recurrent states: every pass is the next token)
        model.batched_step()
        return {"logits": list(b["logits_all"][:, :MIXED_VOCAB]), "tokens": b["token_all"]}
    b["pos_all"].copy_(state["positions"])
    b["step_all"].zero_()
    if "x" in state:
        b["x"][:1].copy_(state["x"])
        model.decode_step()
        return {"logits": [b["logits"]], "tokens": b["token"]}
    b["token_all"].copy_(state["tokens"])
    model.batched_step()
    return {"logits": list(b["logits_all"]), "tokens": b["token_all"]}


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------------------
def _encoder_work(case):
    W, P = CHATTS[case["model"]]["width"], sum(_patches(case))
    weights = PATCH * (1 + EMB) * W + (TS_LAYERS - 1) * W * W
    return dict(bytes=2.0 * weights + 4.0 * P * W + 8.0 * sum(_lengths(case)), flops=2.0 * P * weights)


def work(case):
    path = case["path"]
    if path == "encode":
        return _encoder_work(case)
    if path in ("prompt", "decode"):
        m = CHATTS[case["model"]]
        W = m["width"]
        layer = W * m["dim"] * (2 * m["heads"] + 2 * m["kv"]) + 3 * W * m["ff"]
        head = W * m["vocab"]
        kv = 8.0 * m["layers"] * m["kv"] * m["dim"]     # keys and values of a token, 32 bits
        if path == "prompt":
            T, e = case["text"] + sum(_patches(case)), _encoder_work(case)
            return dict(bytes=e["bytes"] + 2.0 * (layer * m["layers"] + head) + T * (kv + 2.0 * W),
                        flops=e["flops"] + 2.0 * (T * layer * m["layers"] + head) + 2.0 * m["layers"] * m["heads"] * m["dim"] * T * T)
        b, contexts = BYTES_PER_WEIGHT[case["weights"]], _contexts(case)
        return dict(bytes=b * layer * m["layers"] + (2.0 if case["weights"] == "int4" else b) * head + kv * (sum(contexts) + len(contexts)) + 4.0 * len(contexts) * m["vocab"],
                    flops=2.0 * len(contexts) * (layer * m["layers"] + head) + 4.0 * m["layers"] * m["heads"] * m["dim"] * sum(contexts))
    W, ff, shared, heads = MIXED[case["model"]]
    sizes = [len(p) for p in _prompts(case, 0)] if path == "mixed_prompt" else [1] * case["batch"]
    T, C, R = sum(sizes), 2 * W, W // 16
    left, right = W * 128 * (2 * heads + 2 * KV_HEADS), 3 * W * C + C * (R + 2 * STATES) + C * R
    used = EXPERTS * (1 - (1 - TOP / EXPERTS) ** T)
    half = MIXED_LAYERS // 2
    dense = half * (left + right + 4 * W * W) + MIXED_LAYERS * (3 * W * shared + EXPERTS * W)
    head, expert = W * MIXED_VOCAB, 3 * W * ff
    flops = 2.0 * T * (dense + MIXED_LAYERS * TOP * expert) + 2.0 * len(sizes) * head + half * 8.0 * T * C * STATES
    moved = 2.0 * (dense + MIXED_LAYERS * used * expert + head) + 4.0 * len(sizes) * MIXED_VOCAB + half * len(sizes) * 4.0 * (C * (STATES + TAPS) + W)
    if path == "mixed_prompt":
        flops += half * sum(2.0 * heads * 128 * n * n for n in sizes)
        moved += half * T * 4.0 * KV_HEADS * 128
    else:
        flops += half * 4.0 * heads * 128 * sum(_contexts(case))
        moved += half * (4.0 * KV_HEADS * 128 * sum(_contexts(case)) + 4.0 * len(sizes) * C * STATES)
    return dict(bytes=moved, flops=flops)


def tolerance(case):
    # Activations as two bf16 parts, sums in 32 bits: 6e-6 from 64 bits for the encoder, 1e-4 for the whole depth of a decoder.  Designs with experts are
    # as near (2e-4), but a rounding may turn one close choice of an expert, which moves that token's row by a hundredth.
    return {"rel": 2e-5} if case["path"] == "encode" else {"rel": 4e-4, "max": 4e-3} if case["path"] in ("prompt", "decode") else {"rel": 2e-2, "max": 0.3, "differ": 0.01}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------------------------
MOST_ROWS = 4500                       # of a decoder's rows that are computed in 64 bits


def _f64(t):
    return t.to(torch.float64)


def _rms(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * _f64(w)


def _encode64(case, seed):
    t = {n: _f64(v) for n, v in _encoder_tensors(CHATTS[case["model"]], seed)}
    x, rows = _series(case, seed).view(case["series"], -1, 2), []
    for i, n in enumerate(_lengths(case)):
        c = -(-n // PATCH)
        pad = c * PATCH - n
        values = torch.cat([x[i, :n, 0], x[i, n - 1:n, 0].expand(pad)])
        at = torch.cat([torch.arange(n, device="cuda"), torch.full((pad,), MAX_SERIES, device="cuda")])
        rows.append(torch.cat([_f64(values).view(c, PATCH), t["position_embedding.weight"][at].view(c, PATCH * EMB)], 1))
    h = torch.cat(rows)
    for l in range(TS_LAYERS):
        h = h @ t[f"mlp.{2 * l}.weight"].T + t[f"mlp.{2 * l}.bias"]
        if l < TS_LAYERS - 1:
            h = torch.nn.functional.gelu(h)
    return h


def _stored(w, form):
    """the matrix that the stored codes of a weight format stand for"""
    if form == "bf16":
        return _f64(w)
    f = w.float()
    if form == "int4":
        f = f.view(w.shape[0], -1, 128)
        low = f.amin(2, keepdim=True)
        scale = ((f.amax(2, keepdim=True) - low) / 15.0).clamp_min(1e-8).half().float()
        zero = torch.round(-low / scale).clamp(0, 15)
        code = (torch.round(f / scale) + zero).clamp(0, 15)
        return _f64((code * scale - scale * zero).bfloat16()).view(w.shape)
    most = 448.0 if form == "fp8" else 127.0
    top = f.abs().amax(1, keepdim=True).clamp_min(1e-30)
    scale = torch.exp2(torch.ceil(torch.log2(top / most)))
    scale = torch.where(top / scale > most, 2 * scale, scale)
    code = (f / scale).to(torch.float8_e4m3fn).float() if form == "fp8" else torch.round(f / scale).clamp(-127, 127)
    return _f64(code * scale)


def _softmax_values(q, k, v, scale, bias=None):
    """causal attention, q [T, heads, dim], k / v [T, groups, ..]; bias(head, distances) is taken off the scores"""
    T, H, out = q.shape[0], q.shape[1], []
    i = torch.arange(T, device="cuda")
    ahead, far = i[None, :] > i[:, None], (i[:, None] - i[None, :]).clamp_min(0).double()
    for h in range(H):
        g = h * k.shape[1] // H
        s = q[:, h] @ k[:, g].T.contiguous() * scale
        if bias:
            s = s - bias(h, far)
        out.append(torch.softmax(s.masked_fill(ahead, -math.inf), -1) @ v[:, g])
    return torch.stack(out, 1)


def _rotate(x):
    """rotary embedding of [T, heads, dim]: angles in 32 bits, as the models are defined"""
    T, _, d = x.shape
    inv = 1.0 / (THETA ** (torch.arange(0, d, 2, dtype=torch.float32) / d))
    a = (torch.arange(T, dtype=torch.float32)[:, None] * inv[None, :]).cuda()
    cos, sin = _f64(a.cos())[:, None], _f64(a.sin())[:, None]
    u, v = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)


def _chatts64(case, seed, sequences, form="bf16"):
    """logits behind each sequence of embedding rows"""
    m = CHATTS[case["model"]]
    for l in range(m["layers"]):
        p, t = f"model.layers.{l}.", _layer_tensors(m, l, seed)
        w = {n: _stored(v, form) if v.dim() == 2 else _f64(v) for n, v in t.items()}
        for n, x in enumerate(sequences):
            h = _rms(x, w[p + "input_layernorm.weight"], EPS)
            q, k, v = ((h @ w[p + f"self_attn.{s}_proj.weight"].T + w.get(p + f"self_attn.{s}_proj.bias", 0.0)).view(x.shape[0], -1, m["dim"]) for s in "qkv")
            if m["qk_norm"]:
                q, k = _rms(q, w[p + "self_attn.q_norm.weight"], EPS), _rms(k, w[p + "self_attn.k_norm.weight"], EPS)
            a = _softmax_values(_rotate(q), _rotate(k), v, m["dim"] ** -0.5)
            x = x + a.reshape(x.shape[0], -1) @ w[p + "self_attn.o_proj.weight"].T
            h = _rms(x, w[p + "post_attention_layernorm.weight"], EPS)
            h = torch.nn.functional.silu(h @ w[p + "mlp.gate_proj.weight"].T) * (h @ w[p + "mlp.up_proj.weight"].T)
            sequences[n] = x + h @ w[p + "mlp.down_proj.weight"].T
    e = _ends(m, seed)
    head = _stored(e["lm_head.weight"], form if form != "int4" else "bf16")
    return [head @ _rms(x[-1], e["model.norm.weight"], EPS) for x in sequences]


def _glu(h, t, p):
    g, u = (h @ _f64(t[p + "gate"]).T).clamp(max=LIMIT), (h @ _f64(t[p + "up"]).T).clamp(-LIMIT, LIMIT)
    return (g * torch.sigmoid(SLOPE * g) * (u + 1)) @ _f64(t[p + "down"]).T


def _scan64(h, t, p):
    C = t[p + "D"].shape[0]
    x, z = (h @ _f64(t[p + "in"]).T).split([C, C], -1)
    y = torch.zeros_like(x) + _f64(t[p + "conv.b"])
    for back in range(min(TAPS, x.shape[0])):
        y[back:] += _f64(t[p + "conv"])[:, TAPS - 1 - back] * x[:x.shape[0] - back]
    x = torch.nn.functional.silu(y)
    R = t[p + "dt"].shape[1]
    dt, B, Cn = (x @ _f64(t[p + "x"]).T).split([R, STATES, STATES], -1)
    dt = torch.nn.functional.softplus(dt @ _f64(t[p + "dt"]).T + _f64(t[p + "dt.b"]), threshold=100.0)
    A, out = -torch.exp(_f64(t[p + "A_log"])), torch.empty_like(x)
    S = torch.zeros_like(A)
    for i in range(x.shape[0]):
        S = torch.exp(dt[i, :, None] * A) * S + (dt[i] * x[i])[:, None] * B[i]
        out[i] = S @ Cn[i]
    return ((out + _f64(t[p + "D"]) * x) * torch.nn.functional.silu(z)) @ _f64(t[p + "o"]).T


def _mixed64(case, seed, sequences):
    """logits behind each sequence of token ids"""
    W, _, _, heads = MIXED[case["model"]]
    e = _mixed_ends(case, seed)
    streams = []
    for ids in sequences:
        a = torch.arange(len(ids), device="cuda", dtype=torch.float64)[:, None] * 10000.0 ** (-torch.arange(0, W, 2, device="cuda", dtype=torch.float64) / W)
        streams.append([_f64(e["embed"][torch.tensor(ids, device="cuda")]) + torch.stack([a.sin(), a.cos()], -1).view(len(ids), W)])
    xs = [s[0] for s in streams]
    for i in range(MIXED_LAYERS):
        p, t = f"l{i}.", _mixed_layer(case, i, seed)
        for n, x in enumerate(xs):
            h = _rms(x, t[p + "norm1"], 1e-5)
            if i % 2:
                z = torch.sigmoid(h @ _f64(t[p + "mix.z"]).T + _f64(t[p + "mix.z.b"]))
                u = h @ _f64(t[p + "mix.x"]).T + _f64(t[p + "mix.x.b"])
                c, S, y = torch.where(u >= 0, u + 0.5, torch.sigmoid(u)), torch.zeros_like(z[0]), torch.empty_like(z)
                for j in range(z.shape[0]):
                    S = (1 - z[j]) * S + z[j] * c[j]
                    y[j] = S
                y = (y * torch.nn.functional.silu(h @ _f64(t[p + "mix.g"]).T)) @ _f64(t[p + "mix.o"]).T
            else:
                q, k, v = ((h @ _f64(t[p + "mix.left." + s]).T).view(h.shape[0], -1, 128) for s in "qkv")
                r1, r2 = _f64(t[p + "mix.left.r1"]), _f64(t[p + "mix.left.r2"])
                a = _softmax_values(q, k, v, 128 ** -0.5, lambda g, d: r1[g] * torch.log(1 + r2[g] * d)).reshape(h.shape[0], -1)
                y = SIDE * (a @ _f64(t[p + "mix.left.o"]).T) + SIDE * _scan64(h, t, p + "mix.right.")
            x = x + MULT * y
            h = _rms(x, t[p + "norm2"], 1e-5)
            best = torch.softmax(h @ _f64(t[p + "mlp.router"]).T, -1).topk(TOP, -1)
            y = _glu(h, t, p + "mlp.shared.")
            for g in range(EXPERTS):
                r, j = (best.indices == g).nonzero(as_tuple=True)
                y[r] += best.values[r, j, None] * _glu(h[r], t, f"{p}mlp.e{g}.")
            streams[n].append(x + MULT * y)
            xs[n] = sum(a * s for a, s in zip(_f64(t[p + "dwa"]), streams[n]))
    final = [_rms(x[-1], e["final.norm"], 1e-5) @ _f64(e["head"]).T for x in xs]
    return [CAP * torch.tanh(z / CAP) for z in final]


def _some(sequences):
    """as many of the first sequences as are computed in 64 bits"""
    n = rows = 0
    while n < len(sequences) and (n == 0 or rows + len(sequences[n]) <= MOST_ROWS):
        rows += len(sequences[n])
        n += 1
    return n


@torch.no_grad()
def exact(case, seed):
    path = case["path"]
    if path == "encode":
        return {"rows": _encode64(case, seed), "counts": None}
    if path == "prompt":
        embed, rows = _ends(CHATTS[case["model"]], seed)["model.embed_tokens.weight"], _encode64(case, seed)
        parts, ids, at = [], _request(case, seed), 0
        counts, i, text = _patches(case), 0, []
        for t in ids + [TS_TOKEN]:
            if t not in (TS_TOKEN, TS_TOKEN + 1):
                text.append(t)
            elif t == TS_TOKEN:
                parts.append(_f64(embed[torch.tensor(text, dtype=torch.long, device="cuda")]))
                text = []
                if i < len(counts):
                    parts.append(rows[at:at + counts[i]])
                    at, i = at + counts[i], i + 1
        return {"logits": _chatts64(case, seed, [torch.cat(parts)]), "tokens": None}
    if path == "mixed_prompt":
        return {"logits": _mixed64(case, seed, _prompts(case, seed)), "tokens": None}
    vocab = MIXED_VOCAB if path == "mixed_decode" else CHATTS[case["model"]]["vocab"]
    sequences = [_ids(n, seed + 100 * s, vocab) + [_ids(case["batch"], seed + 3, vocab)[s]] for s, n in enumerate(_contexts(case))]
    n = _some(sequences)
    if path == "mixed_decode":
        found = _mixed64(case, seed, [q + [_ids(case["batch"], seed + 4, vocab)[s]] for s, q in enumerate(sequences[:n])])
    else:
        form = case["weights"]
        # (8-bit formats replace the embedding table only where it is tied to the head, which it is not here)
        embed = _ends(CHATTS[case["model"]], seed)["model.embed_tokens.weight"]
        found = _chatts64(case, seed, [_f64(embed[torch.tensor(q, device="cuda")]) for q in sequences[:n]], form)
    return {"logits": found + [None] * (len(sequences) - n), "tokens": None}
