"""What this framework is measured on: the calls a serving program makes.

Each case names a `path` and its sizes.  The paths, and what each stands for:

  step          one serving step of one attention layer: append the new K/V
                row of every sequence, then attend (strided views for one
                sequence, paged views for a batch of ragged lengths).
  prefill       one attention layer of a prompt: causal attention that writes
                the K/V pages.
  cache         a prompt's K/V into the pages and the paged gather back out.
  prompt_ops    the row-wise operators of a prompt around its matrix products
                (embedding, RMSNorm, q/k/v split with RoPE, SwiGLU).
  token_layer   one decoder layer and the LM head for one sequence, replayed
                from a HIP graph as a decode loop does.
  rows_layer    the same for a batch of 2..32 sequences on tiled weights.
  model_prefill a prompt through the decoder (host ids in, host logits out),
                whole or behind a cached prefix.
  model_step    one decode step of the decoder for a batch.

Sizes are those of the repository's configurations (32/8 heads of 64 and 128,
32/4 heads of 64 with hidden 2048 and FFN 5632, 14/2 heads of 64 with hidden
896 and FFN 4864) and a generic hidden 4096 with 32/8 heads of 128.

`exact` computes the same outputs in 64 bits with plain torch.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "serving-engine_amd"))

import kvhp  # noqa: E402

PAGE = 16
EPS = 1e-5
THETA = 10000.0

# name -> (hidden, ffn, q heads, kv heads, head dim, vocab)
DIMS = {
    "h896": (896, 4864, 14, 2, 64, 32000),
    "h1024": (1024, 2816, 16, 4, 64, 32000),
    "h2048": (2048, 5632, 32, 4, 64, 32000),
    "h4096": (4096, 11264, 32, 8, 128, 32000),
}


def listed():
    return [
        # the smallest call: one token, 512 cached keys, contiguous cache
        {"name": "step_1x512", "path": "step", "batch": 1, "ctx": 512, "hq": 32, "hkv": 8,
         "d": 64, "paged": False},
        # one long context, contiguous cache
        {"name": "step_1x16384", "path": "step", "batch": 1, "ctx": 16384, "hq": 32, "hkv": 8,
         "d": 128, "paged": False},
        # batched serving: 32 ragged sequences of up to 8K keys in shuffled pages
        {"name": "step_32x8192", "path": "step", "batch": 32, "ctx": 8192, "hq": 32, "hkv": 8,
         "d": 128, "paged": True},
        # an ordinary prompt
        {"name": "prefill_2048", "path": "prefill", "batch": 1, "seq": 2048, "hq": 32, "hkv": 8,
         "d": 128},
        # a few odd, short prompts at 7 query heads per KV head
        {"name": "prefill_3x777", "path": "prefill", "batch": 3, "seq": 777, "hq": 14, "hkv": 2,
         "d": 64},
        # four prompts' K/V moved into pages and gathered
        {"name": "cache_4x2048", "path": "cache", "batch": 4, "seq": 2048, "hkv": 8, "d": 128},
        # the row-wise work of one layer of an odd-sized prompt
        {"name": "prompt_ops_1999", "path": "prompt_ops", "dims": "h2048", "seq": 1999},
        # single-sequence decode of the default configuration's layer and head
        {"name": "token_layer_896", "path": "token_layer", "dims": "h896", "ctx": 700},
        # an odd batch of sequences through one layer and the head
        {"name": "rows_layer_17", "path": "rows_layer", "dims": "h2048", "batch": 17,
         "ctx": 1024},
        # a 2048-id prompt through the 22-layer, 1.1B decoder
        {"name": "model_prefill_2048", "path": "model_prefill", "dims": "h2048", "layers": 22,
         "seq": 2048, "cached": 0},
        # a prompt whose first 1488 positions are a cached prefix, through two layers
        {"name": "model_cached_2000", "path": "model_prefill", "dims": "h2048", "layers": 2,
         "seq": 2000, "cached": 1488},
        # greedy decoding's step of the 22-layer decoder at 2K context
        {"name": "model_step_1", "path": "model_step", "dims": "h2048", "layers": 22, "batch": 1,
         "ctx": 2048},
    ]


def _log(rng, lo, hi):
    """An integer between lo and hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(["step", "step", "prefill", "prefill", "cache", "prompt_ops",
                       "token_layer", "rows_layer", "model_prefill", "model_prefill",
                       "model_step"])
    heads = rng.choice([(32, 8, 128), (32, 8, 64), (32, 4, 64), (14, 2, 64)])
    if path == "step":
        batch = rng.choice([1, _log(rng, 2, 64)])
        ctx = _log(rng, 128, 65536 if batch == 1 else 8192)
        return {"path": path, "batch": batch, "ctx": ctx, "hq": heads[0], "hkv": heads[1],
                "d": heads[2], "paged": batch > 1}
    if path == "prefill":
        seq = _log(rng, 16, 8192)
        batch = rng.choice([1, 1, 2, 3, 4]) if seq <= 2048 else 1
        return {"path": path, "batch": batch, "seq": seq, "hq": heads[0], "hkv": heads[1],
                "d": heads[2]}
    if path == "cache":
        return {"path": path, "batch": _log(rng, 1, 8), "seq": _log(rng, 16, 4096),
                "hkv": heads[1], "d": heads[2]}
    if path == "prompt_ops":
        return {"path": path, "dims": rng.choice(["h896", "h2048", "h4096"]),
                "seq": _log(rng, 16, 4096)}
    if path == "token_layer":
        return {"path": path, "dims": rng.choice(["h896", "h1024", "h2048", "h4096"]),
                "ctx": _log(rng, 64, 4096)}
    if path == "rows_layer":
        return {"path": path, "dims": rng.choice(["h1024", "h2048"]), "batch": _log(rng, 2, 32),
                "ctx": _log(rng, 64, 2048)}
    if path == "model_prefill":
        dims, layers = rng.choice([("h2048", 22), ("h2048", 2), ("h896", 24)])
        seq = _log(rng, 32, 2048)
        cached = rng.choice([0, PAGE * rng.randint(0, (seq - 1) // PAGE)])
        return {"path": path, "dims": dims, "layers": layers, "seq": seq, "cached": cached}
    dims, layers = rng.choice([("h2048", 22), ("h896", 24)])
    return {"path": path, "dims": dims, "layers": layers, "batch": _log(rng, 1, 48),
            "ctx": _log(rng, 64, 2048)}


# ---------------------------------------------------------------- inputs ----
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape, std=1.0):
    t = torch.empty(shape, dtype=torch.float16, device="cuda")
    return t.normal_(0.0, std, generator=g)


def _lens(case, seed):
    """Lengths after the step: the full context for one sequence; for a batch
    the same ragged lengths for every seed, in another order."""
    if case["batch"] == 1:
        return np.array([case["ctx"]], np.int32)
    rng = np.random.default_rng([case["batch"], case["ctx"]])
    lens = rng.integers(max(1, case["ctx"] // 64), case["ctx"] + 1, case["batch"])
    lens[0] = case["ctx"]
    return np.random.default_rng(seed).permutation(lens).astype(np.int32)


def _tables(lens, seed, width=None):
    """Block tables over a shuffled pool: [batch][width], -1 past each sequence; pool pages."""
    need = [(int(n) + PAGE - 1) // PAGE for n in lens]
    total = sum(need)
    perm = np.random.default_rng(seed + 1).permutation(total).astype(np.int32)
    bt = np.full((len(lens), width or max(need)), -1, np.int32)
    at = 0
    for b, n in enumerate(need):
        bt[b, :n] = perm[at:at + n]
        at += n
    return bt, total


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _step_inputs(case, seed):
    B, hq, hkv, d = case["batch"], case["hq"], case["hkv"], case["d"]
    g, lens = _gen(seed), _lens(case, seed)
    s = {"lens_h": lens, "lens": _dev(lens), "pos": _dev(lens - 1)}
    s["q"] = _normal(g, B, hq, d)
    s["k_new"], s["v_new"] = _normal(g, B, hkv, d), _normal(g, B, hkv, d)
    if case["paged"]:
        bt, pages = _tables(lens, seed)
        s["bt"] = _dev(bt)
        shape = (hkv, pages, PAGE, d)
    else:
        shape = (hkv, case["ctx"], d)
    s["pool_k"], s["pool_v"] = _normal(g, *shape), _normal(g, *shape)
    return s


def _prefill_inputs(case, seed):
    B, S, hq, hkv, d = case["batch"], case["seq"], case["hq"], case["hkv"], case["d"]
    g = _gen(seed)
    bt, pages = _tables([S] * B, seed)
    return {"q": _normal(g, B, S, hq, d), "k": _normal(g, B, S, hkv, d),
            "v": _normal(g, B, S, hkv, d), "bt": _dev(bt), "pages": pages}


def _cache_inputs(case, seed):
    B, S, hkv, d = case["batch"], case["seq"], case["hkv"], case["d"]
    g = _gen(seed)
    bt, pages = _tables([S] * B, seed)
    return {"k": _normal(g, B, S, hkv, d), "v": _normal(g, B, S, hkv, d), "bt": _dev(bt),
            "pages": pages}


def _prompt_inputs(case, seed):
    H, F, hq, hkv, d, V = DIMS[case["dims"]]
    n, g = case["seq"], _gen(seed)
    ids = np.random.default_rng(seed).integers(0, V, n).astype(np.int32)
    return {"ids": _dev(ids), "table": _normal(g, V, H, std=0.02),
            "norm": _normal(g, H, std=0.1) + 1.0, "x": _normal(g, n, H),
            "qkv": _normal(g, n, (hq + 2 * hkv) * d), "gu": _normal(g, n, 2 * F)}


def _layer_inputs(case, seed, B):
    """Weights, hidden rows and K/V pages of one decoder layer and the head."""
    H, F, hq, hkv, d, V = DIMS[case["dims"]]
    g = _gen(seed)
    lens = _lens(dict(case, batch=B), seed)
    bt, pages = _tables(lens, seed)
    w = lambda n, k: _normal(g, n, k, std=0.02)  # noqa: E731
    return {"lens_h": lens, "lens": _dev(lens), "pos": _dev(lens - 1), "bt": _dev(bt),
            "pages": pages, "x": _normal(g, B, H), "n1": _normal(g, H, std=0.1) + 1.0,
            "n2": _normal(g, H, std=0.1) + 1.0, "n3": _normal(g, H, std=0.1) + 1.0,
            "w_qkv": w((hq + 2 * hkv) * d, H), "w_o": w(H, hq * d), "w_gu": w(2 * F, H),
            "w_down": w(H, F), "w_head": w(V, H),
            "pool_k": _normal(g, hkv, pages, PAGE, d), "pool_v": _normal(g, hkv, pages, PAGE, d)}


def _model_config(case):
    H, F, hq, hkv, d, V = DIMS[case["dims"]]
    return kvhp.LlamaConfig(V, H, case["layers"], hq, hkv, d, F, EPS, THETA, 0)


def _model_inputs(case, seed):
    """Pages with the cached keys and values, ids and lengths (not the weights)."""
    _, _, _, hkv, d, V = DIMS[case["dims"]]
    g, rng = _gen(seed), np.random.default_rng(seed)
    if case["path"] == "model_prefill":
        lens = np.array([case["seq"]], np.int32)
        ids = rng.integers(0, V, case["seq"]).astype(np.int32)
    else:
        lens = _lens(case, seed)
        ids = rng.integers(0, V, case["batch"]).astype(np.int32)
    bt, pages = _tables(lens, seed)
    return {"lens_h": lens, "ids": ids, "bt": _dev(bt), "width": bt.shape[1], "pages": pages,
            "pool": _normal(g, case["layers"], 2, hkv, pages, PAGE, d)}


# --------------------------------------------------------------- prepare ----
def _graph(fn):
    """fn captured in a HIP graph (after one eager call), as a decode loop keeps it."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        fn()
    return graph


def _workspace(B, hq, hkv, d, ctx):
    n = kvhp.decode_workspace_bytes(B, hq, hkv, d, ctx)
    return torch.empty(max(n, 256), dtype=torch.uint8, device="cuda")


def _half(*shape):
    return torch.empty(shape, dtype=torch.float16, device="cuda")


def _prepare_token_layer(case, s):
    H, F, hq, hkv, d, V = DIMS[case["dims"]]
    s["ws"] = _workspace(1, hq, hkv, d, case["ctx"])
    s["q"], s["attn"] = _half(1, hq * d), _half(1, hq * d)
    s["h1"], s["act"], s["h2"] = _half(1, H), _half(1, F), _half(1, H)
    s["logits"] = torch.empty((1, V), dtype=torch.float32, device="cuda")
    kv, vv = kvhp.paged_view(s["pool_k"], s["bt"]), kvhp.paged_view(s["pool_v"], s["bt"])

    def layer():
        kvhp.rmsnorm_qkv_rope_append(s["w_qkv"], s["x"], s["n1"], EPS, s["lens"], THETA, s["q"],
                                     s["pool_k"], s["pool_v"], s["bt"], hq, hkv, d, H)
        kvhp.decode_attention(s["q"], kv, vv, s["lens"], s["attn"], hq, hkv, d, case["ctx"],
                              workspace=s["ws"])
        kvhp.gemv_residual(s["w_o"], s["attn"], s["x"], s["h1"], H, hq * d)
        kvhp.rmsnorm_gemv_swiglu(s["w_gu"], s["h1"], s["n2"], EPS, s["act"], F, H)
        kvhp.gemv_residual(s["w_down"], s["act"], s["h1"], s["h2"], H, F)
        kvhp.rmsnorm_gemv(s["w_head"], s["h2"], s["n3"], EPS, V, H, y32=s["logits"])

    s["graph"] = _graph(layer)
    return s


def _tile(kind, W, N, K, hq=0, hkv=0, d=0):
    out = torch.empty(kvhp.rows_tiled_bytes(kind, N, K, hq, hkv, d), dtype=torch.uint8,
                      device="cuda")
    kvhp.rows_tile_weights(kind, W, N, K, out, hq, hkv, d)
    return out


def _prepare_rows_layer(case, s):
    H, F, hq, hkv, d, V = DIMS[case["dims"]]
    B = case["batch"]
    # everything the graph reads stays in the state, as long as the graph does
    s["w_qkv"] = _tile(kvhp.ROWS_QKV, s["w_qkv"], 0, H, hq, hkv, d)
    s["w_o"] = _tile(kvhp.ROWS_PLAIN, s["w_o"], H, hq * d)
    s["w_gu"] = _tile(kvhp.ROWS_SWIGLU, s["w_gu"], F, H)
    s["w_down"] = _tile(kvhp.ROWS_PLAIN, s["w_down"], H, F)
    s["w_head"] = _tile(kvhp.ROWS_PLAIN, s["w_head"], V, H)
    s["ws"] = _workspace(B, hq, hkv, d, case["ctx"])
    nws = kvhp.gemv_rows_workspace_bytes(H, F, B)
    s["ws2"] = torch.empty(nws, dtype=torch.uint8, device="cuda") if nws else None
    s["q"], s["attn"] = _half(B, hq * d), _half(B, hq * d)
    s["h1"], s["act"], s["h2"] = _half(B, H), _half(B, F), _half(B, H)
    s["logits"] = torch.empty((B, V), dtype=torch.float32, device="cuda")
    kv, vv = kvhp.paged_view(s["pool_k"], s["bt"]), kvhp.paged_view(s["pool_v"], s["bt"])

    def layer():
        kvhp.rmsnorm_qkv_rope_append_rows_tiled(s["w_qkv"], s["x"], s["n1"], EPS, s["pos"], THETA,
                                                s["q"], s["pool_k"], s["pool_v"], s["bt"], hq,
                                                hkv, d, H, B)
        kvhp.decode_attention(s["q"], kv, vv, s["lens"], s["attn"], hq, hkv, d, case["ctx"],
                              workspace=s["ws"])
        kvhp.gemv_residual_rows_tiled(s["w_o"], s["attn"], s["x"], s["h1"], H, hq * d, B)
        kvhp.rmsnorm_gemv_swiglu_rows_tiled(s["w_gu"], s["h1"], s["n2"], EPS, s["act"], F, H, B)
        kvhp.gemv_residual_rows_tiled(s["w_down"], s["act"], s["h1"], s["h2"], H, F, B,
                                      workspace=s["ws2"])
        kvhp.rmsnorm_gemv_rows_tiled(s["w_head"], s["h2"], s["n3"], EPS, V, H, B, y32=s["logits"])

    s["graph"] = _graph(layer)
    return s


def prepare(case, seed):
    path = case["path"]
    if path == "step":
        s = _step_inputs(case, seed)
        B, hq, hkv, d = case["batch"], case["hq"], case["hkv"], case["d"]
        s["out"] = _half(B, hq, d)
        s["ws"] = _workspace(B, hq, hkv, d, case["ctx"])
        view = ((lambda t: kvhp.paged_view(t, s["bt"])) if case["paged"] else
                (lambda t: kvhp.strided_view(t, t.numel(), case["ctx"] * d, d)))
        s["kv"], s["vv"] = view(s["pool_k"]), view(s["pool_v"])
    elif path == "prefill":
        s = _prefill_inputs(case, seed)
        s["out"] = torch.empty_like(s["q"])
        s["pool_k"] = torch.zeros((case["hkv"], s["pages"], PAGE, case["d"]), dtype=torch.float16,
                                  device="cuda")
        s["pool_v"] = torch.zeros_like(s["pool_k"])
    elif path == "cache":
        s = _cache_inputs(case, seed)
        B, S, hkv, d = case["batch"], case["seq"], case["hkv"], case["d"]
        s["pool_k"] = torch.zeros((hkv, s["pages"], PAGE, d), dtype=torch.float16, device="cuda")
        s["pool_v"] = torch.zeros_like(s["pool_k"])
        s["zero"] = torch.zeros(B, dtype=torch.int32, device="cuda")
        s["lens"] = torch.full((B,), S, dtype=torch.int32, device="cuda")
        s["out_k"], s["out_v"] = _half(B, hkv, S, d), _half(B, hkv, S, d)
    elif path == "prompt_ops":
        s = _prompt_inputs(case, seed)
        H, F, hq, hkv, d, V = DIMS[case["dims"]]
        n = case["seq"]
        s["hidden"], s["normed"], s["act"] = _half(n, H), _half(n, H), _half(n, F)
        s["q"], s["k"], s["v"] = _half(n, hq, d), _half(n, hkv, d), _half(n, hkv, d)
    elif path == "token_layer":
        s = _prepare_token_layer(case, _layer_inputs(case, seed, 1))
    elif path == "rows_layer":
        s = _prepare_rows_layer(case, _layer_inputs(case, seed, case["batch"]))
    else:
        s = _model_inputs(case, seed)
        V = DIMS[case["dims"]][5]
        if path == "model_prefill":
            s["model"] = kvhp.LlamaModel(_model_config(case), seed, case["seq"])
        else:
            B = case["batch"]
            s["model"] = kvhp.LlamaModel(_model_config(case), seed, max(case["ctx"], B))
            s["model"].reserve(B, case["ctx"])
            s["tok"], s["lens"] = _dev(s["ids"]), _dev(s["lens_h"])
            s["pos"] = _dev(s["lens_h"] - 1)
            s["logits"] = torch.empty((B, V), dtype=torch.float32, device="cuda")
            s["next"] = torch.empty(B, dtype=torch.int32, device="cuda")
    s["case"] = case
    return s


# ------------------------------------------------------------------- run ----
def run(s):
    case = s["case"]
    path = case["path"]
    if path == "step":
        f = kvhp.paged_append_decode if case["paged"] else kvhp.append_decode
        f(s["q"], s["k_new"], s["v_new"], s["kv"], s["vv"], s["pos"], s["lens"], s["out"],
          case["hq"], case["hkv"], case["d"], case["ctx"], workspace=s["ws"])
        return {"out": s["out"], "pool_k": s["pool_k"], "pool_v": s["pool_v"]}
    if path == "prefill":
        kvhp.flash_prefill_paged(s["q"], s["k"], s["v"], s["out"], case["seq"], case["hq"],
                                 case["hkv"], case["d"], case["batch"], s["pool_k"], s["pool_v"],
                                 s["bt"])
        return {"out": s["out"], "pool_k": s["pool_k"], "pool_v": s["pool_v"]}
    if path == "cache":
        kvhp.paged_append_kv(s["k"], s["v"], s["pool_k"], s["pool_v"], s["bt"], s["zero"],
                             case["batch"], case["seq"], case["hkv"], case["d"])
        kvhp.paged_gather_kv(s["pool_k"], s["pool_v"], s["bt"], s["lens"], case["seq"],
                             s["out_k"], s["out_v"])
        return {"pool_k": s["pool_k"], "pool_v": s["pool_v"], "k": s["out_k"], "v": s["out_v"]}
    if path == "prompt_ops":
        H, F, hq, hkv, d, V = DIMS[case["dims"]]
        n = case["seq"]
        kvhp.embedding(s["ids"], s["table"], s["hidden"], n, H, V)
        kvhp.rmsnorm(s["x"], s["norm"], s["normed"], n, H, EPS)
        kvhp.split_qkv_rope(s["qkv"], n, hq, hkv, d, 0, THETA, s["q"], s["k"], s["v"])
        kvhp.swiglu_rows(s["gu"], s["act"], n, F)
        return {k: s[k] for k in ("hidden", "normed", "q", "k", "v", "act")}
    if path in ("token_layer", "rows_layer"):
        s["graph"].replay()
        return {k: s[k] for k in ("q", "attn", "h1", "act", "h2", "logits", "pool_k", "pool_v")}
    # The greedy token follows from the logits, and two correct roundings may
    # pick either of two near-equal ones: the logits and the pages are compared.
    if path == "model_prefill":
        m, width = s["model"], s["width"]
        if case["cached"]:
            _, logits = m.prefill_cached(s["ids"], case["cached"], s["pool"], s["pages"], s["bt"],
                                         width)
        else:
            _, logits = m.prefill_paged(s["ids"], s["pool"], s["pages"], s["bt"], width)
        return {"logits": logits, "pool": s["pool"]}
    s["model"].decode_paged(s["tok"], s["pool"], s["pages"], s["bt"], s["width"], s["pos"],
                            s["lens"], case["ctx"], s["logits"], s["next"])
    return {"logits": s["logits"], "pool": s["pool"]}


# ------------------------------------------------------------------ work ----
def _layer_weights(dims):
    H, F, hq, hkv, d, _ = DIMS[dims]
    return (hq + 2 * hkv) * d * H + H * hq * d + 3 * F * H


def work(case):
    """Bytes: every input read once, every output written once.  Flops: the
    products and contractions (two per multiply-add)."""
    path = case["path"]
    if path == "step":
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        keys = int(_lens(case, 0).sum())
        return {"bytes": 4 * keys * hkv * d + 4 * case["batch"] * (hq + 2 * hkv) * d,
                "flops": 4 * keys * hq * d}
    if path == "prefill":
        B, S, hq, hkv, d = case["batch"], case["seq"], case["hq"], case["hkv"], case["d"]
        return {"bytes": 2 * B * S * d * (2 * hq + 4 * hkv), "flops": 2 * B * hq * d * S * (S + 1)}
    if path == "cache":
        return {"bytes": 16 * case["batch"] * case["seq"] * case["hkv"] * case["d"], "flops": 0}
    H, F, hq, hkv, d, V = DIMS[case["dims"]]
    if path == "prompt_ops":
        return {"bytes": 2 * case["seq"] * (4 * H + 2 * (hq + 2 * hkv) * d + 3 * F), "flops": 0}
    if path in ("token_layer", "rows_layer", "model_step"):
        B = case.get("batch", 1)
        layers = case.get("layers", 1)
        keys = int(_lens(dict(case, batch=B), 0).sum())
        w = layers * _layer_weights(case["dims"]) + V * H
        return {"bytes": 2 * w + layers * 4 * keys * hkv * d + 4 * B * V,
                "flops": 2 * B * w + layers * 4 * keys * hq * d}
    n, c, layers = case["seq"], case["cached"], case["layers"]
    w = layers * _layer_weights(case["dims"])
    attn = layers * 2 * hq * d * (n * (n + 1) - c * (c + 1))
    return {"bytes": 2 * (w + V * H) + layers * 4 * n * hkv * d,
            "flops": 2 * (n - c) * w + 2 * V * H + attn}


def tolerance(case):
    """About four times the relative error that each path shows against
    `exact`: results and intermediates rounded to fp16 (2.7e-4 for one
    attention call or row-wise operator, 6e-4 through one layer, 1.1e-3
    through two layers and the head, 4e-3 through 22)."""
    path = case["path"]
    if path == "cache":
        return "exact"
    if path in ("step", "prefill", "prompt_ops"):
        return {"rel": 1.1e-3}
    if path in ("token_layer", "rows_layer"):
        return {"rel": 2.5e-3}
    return {"rel": 1.6e-2 if case["layers"] > 2 else 4.5e-3}


# ----------------------------------------------------------------- exact ----
def _attend(q, k, v, first=0):
    """q [S][hq][d] at positions first.., k/v [T][hkv][d], causal, in 64 bits."""
    S, hq, d = q.shape
    T, hkv, _ = k.shape
    G, out = hq // hkv, torch.empty(S, hq, d, dtype=torch.float64, device=q.device)
    pos = torch.arange(first, first + S, device=q.device)
    mask = torch.arange(T, device=q.device)[None, :] > pos[:, None]
    for h in range(hkv):
        kt, vh = k[:, h].double().t().contiguous(), v[:, h].double().contiguous()
        for i in range(h * G, (h + 1) * G):
            sc = (q[:, i].double() @ kt) / math.sqrt(d)
            out[:, i] = torch.softmax(sc.masked_fill_(mask, -math.inf), dim=1) @ vh
    return out


def _norm(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos):
    """x [n][h][d] rotated in halves at positions pos [n]."""
    d = x.shape[-1]
    inv = THETA ** (-torch.arange(0, d, 2, dtype=torch.float64, device=x.device) / d)
    ang = pos.double()[:, None, None] * inv
    a, b = x[..., :d // 2].double(), x[..., d // 2:].double()
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


def _swiglu(gu):
    g, u = gu.double().chunk(2, -1)
    return g * torch.sigmoid(g) * u


def _rows(bt_row, n):
    """Pool row of each of n positions."""
    t = torch.arange(n, device="cuda")
    return bt_row.long()[t // PAGE] * PAGE + t % PAGE


def _layer_exact(x, w, pool_k, pool_v, bt, lens, first, hq, hkv, d, prompt):
    """One decoder layer in 64 bits.  prompt: x holds positions first.. of one
    sequence; else row b is sequence b's token at lens[b] - 1.  pool_* [hkv][rows][d]
    in 64 bits, updated in place.  Returns q, attention, h1, act, h2."""
    n = x.shape[0]
    pos = (torch.arange(first, first + n, device=x.device) if prompt
           else torch.as_tensor(lens, device=x.device).long() - 1)
    qkv = (_norm(x, w["n1"]) @ w["w_qkv"].double().t()).view(n, hq + 2 * hkv, d)
    q, k = _rope(qkv[:, :hq], pos), _rope(qkv[:, hq:hq + hkv], pos)
    v = qkv[:, hq + hkv:]
    attn = torch.empty(n, hq, d, dtype=torch.float64, device=x.device)
    if prompt:
        rows = _rows(bt[0], first + n)
        pool_k[:, rows[first:]], pool_v[:, rows[first:]] = k.transpose(0, 1), v.transpose(0, 1)
        attn = _attend(q, pool_k[:, rows].transpose(0, 1), pool_v[:, rows].transpose(0, 1), first)
    else:
        for b in range(n):
            rows = _rows(bt[b], int(lens[b]))
            pool_k[:, rows[-1]], pool_v[:, rows[-1]] = k[b], v[b]
            attn[b] = _attend(q[b:b + 1], pool_k[:, rows].transpose(0, 1),
                              pool_v[:, rows].transpose(0, 1), int(lens[b]) - 1)[0]
    h1 = x.double() + attn.reshape(n, hq * d) @ w["w_o"].double().t()
    act = _swiglu(_norm(h1, w["n2"]) @ w["w_gu"].double().t())
    return q, attn, h1, act, h1 + act @ w["w_down"].double().t()


def _wrap(x):
    x &= (1 << 64) - 1
    return x - (1 << 64) if x >> 63 else x


def _mix(z):
    """splitmix64 of a 64-bit integer tensor (wrapping arithmetic)."""
    shr = lambda v, n: (v >> n) & ((1 << (64 - n)) - 1)  # noqa: E731
    z = z + _wrap(0x9E3779B97F4A7C15)
    z = (z ^ shr(z, 30)) * _wrap(0xBF58476D1CE4E5B9)
    z = (z ^ shr(z, 27)) * _wrap(0x94D049BB133111EB)
    return z ^ shr(z, 31)


def _weights(n, seed, stream, shape):
    """The decoder's seeded N(0, 0.02) fp16 weights, as the library documents
    them: a Box-Muller normal of two splitmix64 hashes per element."""
    one = lambda v: torch.tensor([_wrap(v)], dtype=torch.int64, device="cuda")  # noqa: E731
    base = _mix(one(seed) ^ _mix(one(stream)))
    out = torch.empty(n, dtype=torch.float16, device="cuda")
    for a in range(0, n, 1 << 24):
        i = 2 * torch.arange(a, min(n, a + (1 << 24)), device="cuda") + base
        top = lambda z: ((_mix(z) >> 40) & 0xFFFFFF).float()  # noqa: E731
        u1, u2 = (top(i) + 0.5) * 2.0 ** -24, top(i + 1) * 2.0 ** -24
        r = torch.sqrt(-2.0 * torch.log(u1.double()))
        z = 0.02 * r * torch.cos(2.0 * math.pi * u2.double())
        out[a:a + z.numel()] = z.float().half()
    return out.view(shape)


def _model_exact(case, seed):
    H, F, hq, hkv, d, V = DIMS[case["dims"]]
    s = _model_inputs(case, seed)
    prompt = case["path"] == "model_prefill"
    first = case["cached"] if prompt else 0
    embed, head = _weights(V * H, seed, 1, (V, H)), _weights(V * H, seed, 2, (V, H))
    ids = _dev(s["ids"]).long()
    x = embed[ids[first:]].double()
    one = torch.ones(H, dtype=torch.float64, device="cuda")
    pool = s["pool"].double().view(case["layers"], 2, hkv, s["pages"] * PAGE, d)
    stream = 3
    for l in range(case["layers"]):
        nq = (hq + 2 * hkv) * d
        w = {"n1": one, "n2": one, "w_qkv": _weights(nq * H, seed, stream, (nq, H)),
             "w_o": _weights(H * hq * d, seed, stream + 1, (H, hq * d)),
             "w_gu": _weights(2 * F * H, seed, stream + 2, (2 * F, H)),
             "w_down": _weights(H * F, seed, stream + 3, (H, F))}
        stream += 4
        x = _layer_exact(x, w, pool[l, 0], pool[l, 1], s["bt"], s["lens_h"], first, hq, hkv, d,
                         prompt)[4]
    logits = _norm(x[-1:] if prompt else x, one) @ head.double().t()
    return {"logits": logits[0] if prompt else logits,
            "pool": pool.view(case["layers"], 2, hkv, s["pages"], PAGE, d)}


def exact(case, seed):
    path = case["path"]
    if path == "step":
        s = _step_inputs(case, seed)
        hq, hkv, d = case["hq"], case["hkv"], case["d"]
        out = torch.empty(case["batch"], hq, d, dtype=torch.float64, device="cuda")
        for b, n in enumerate(s["lens_h"]):
            rows = (_rows(s["bt"][b], int(n)) if case["paged"]
                    else torch.arange(int(n), device="cuda"))
            pk, pv = s["pool_k"].view(hkv, -1, d), s["pool_v"].view(hkv, -1, d)
            pk[:, rows[-1]], pv[:, rows[-1]] = s["k_new"][b], s["v_new"][b]
            out[b] = _attend(s["q"][b:b + 1], pk[:, rows].transpose(0, 1),
                             pv[:, rows].transpose(0, 1), int(n) - 1)[0]
        return {"out": out, "pool_k": s["pool_k"], "pool_v": s["pool_v"]}
    if path in ("prefill", "cache"):
        s = _prefill_inputs(case, seed) if path == "prefill" else _cache_inputs(case, seed)
        B, S, hkv, d = case["batch"], case["seq"], case["hkv"], case["d"]
        pools = [torch.zeros((hkv, s["pages"] * PAGE, d), dtype=torch.float16, device="cuda")
                 for _ in range(2)]
        for b in range(B):
            rows = _rows(s["bt"][b], S)
            for p, src in zip(pools, (s["k"], s["v"])):
                p[:, rows] = src[b].transpose(0, 1)
        pk, pv = (p.view(hkv, s["pages"], PAGE, d) for p in pools)
        if path == "cache":
            return {"pool_k": pk, "pool_v": pv, "k": s["k"].transpose(1, 2).contiguous(),
                    "v": s["v"].transpose(1, 2).contiguous()}
        out = torch.stack([_attend(s["q"][b], s["k"][b], s["v"][b]) for b in range(B)])
        return {"out": out, "pool_k": pk, "pool_v": pv}
    if path == "prompt_ops":
        s = _prompt_inputs(case, seed)
        H, F, hq, hkv, d, V = DIMS[case["dims"]]
        n = case["seq"]
        pos = torch.arange(n, device="cuda")
        qkv = s["qkv"].view(n, hq + 2 * hkv, d)
        return {"hidden": s["table"][s["ids"].long()], "normed": _norm(s["x"], s["norm"]),
                "q": _rope(qkv[:, :hq], pos), "k": _rope(qkv[:, hq:hq + hkv], pos),
                "v": qkv[:, hq + hkv:].contiguous(), "act": _swiglu(s["gu"])}
    if path in ("token_layer", "rows_layer"):
        H, F, hq, hkv, d, V = DIMS[case["dims"]]
        B = case.get("batch", 1)
        s = _layer_inputs(case, seed, B)
        pk, pv = (s[k].double().view(hkv, -1, d) for k in ("pool_k", "pool_v"))
        q, attn, h1, act, h2 = _layer_exact(s["x"], s, pk, pv, s["bt"], s["lens_h"], 0, hq, hkv,
                                            d, False)
        return {"q": q.reshape(B, hq * d), "attn": attn.reshape(B, hq * d), "h1": h1, "act": act,
                "h2": h2, "logits": _norm(h2, s["n3"]) @ s["w_head"].double().t(),
                "pool_k": pk.view(hkv, -1, PAGE, d), "pool_v": pv.view(hkv, -1, PAGE, d)}
    return _model_exact(case, seed)
