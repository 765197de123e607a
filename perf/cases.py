"""What the performance of this framework is judged on.

Each case is one call (or the short fixed sequence of calls) that a program
makes through the public entry points of ``wgkv``, on inputs of the shapes the
repository's configurations, benchmark and tests use: Llama-8B-like attention
(32 query heads, 8 KV heads, head_dim 128, window 1024, pages of 16), with
other group sizes, head dims, windows and odd lengths drawn beside them.

Kinds:
  decode   one token's attention over paged per-head caches, batch 1 to 32
  quest    the same with QUEST page selection before it
  step     a whole model's decode step (captured graph), logits out
  oneshot  a prompt's admission, metadata and sparse attention in one piece
  chunked  a prompt's admission, attention and ring rewrite in chunks
  gate     the write gate over a prompt chunk or a window
  rows     the decoder's row-wise work over a prompt chunk: norms with the
           residual add, rotary embedding, SwiGLU product
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "wg-kv_amd"))

from wgkv import e2e, model_ops, ops  # noqa: E402
from wgkv.attention import LlamaAttention  # noqa: E402
from wgkv.cache import DualCache  # noqa: E402
from wgkv.gate import GatingPredictor  # noqa: E402
from wgkv.layers import WGKVConfig  # noqa: E402

BF16 = torch.bfloat16
BLK = 64  # rows of a query block of the sparse prefill


def listed():
    heads = {"Hq": 32, "Hkv": 8, "D": 128}
    return [
        # a chat turn's token: one sequence, little more than the local window cached
        {"name": "decode_b1_2k", "kind": "decode", "B": 1, "ctx": 2048, "W": 1024, "page": 16, **heads},
        # one long-context sequence (the benchmark's batch-1 row)
        {"name": "decode_b1_128k", "kind": "decode", "B": 1, "ctx": 131072, "W": 1024, "page": 16, **heads},
        # a serving batch of ordinary contexts
        {"name": "decode_b32_8k", "kind": "decode", "B": 32, "ctx": 8192, "W": 1024, "page": 16, **heads},
        # the headline: batch 8 at 128K, 2-60 % admitted per head
        {"name": "decode_b8_128k", "kind": "decode", "B": 8, "ctx": 131072, "W": 1024, "page": 16, **heads},
        # a decode step of the QUEST baseline: select pages, attend over them
        {"name": "quest_b1_128k", "kind": "quest", "ctx": 131072, "W": 1024, "frac": 0.2, "budget": 4096, **heads},
        # a whole decode step as a server replays it: 2 layers of the 8B model and its LM head
        {"name": "step_2layers_8k", "kind": "step", "layers": 2, "ctx": 8192, "vocab": 128256, "hidden": 4096,
         "ffn": 14336, "W": 1024, "frac": 0.2, "qk_norm": False, **heads},
        # a short question, odd length
        {"name": "oneshot_777", "kind": "oneshot", "S": 777, "W": 256, "frac": 0.2, **heads},
        # an ordinary document in one piece, odd length
        {"name": "oneshot_9k", "kind": "oneshot", "S": 9001, "W": 1024, "frac": 0.2, **heads},
        # a long prompt in 4096-token chunks (the benchmark's prefill row)
        {"name": "chunked_32k", "kind": "chunked", "S": 32768, "chunk": 4096, "W": 1024, "frac": 0.2, **heads},
        # the gate over one prompt chunk, bf16 parameters (inference)
        {"name": "gate_bf16_4k", "kind": "gate", "S": 4096, "Hkv": 8, "D": 128, "expand": 4.0, "param": "bf16",
         "fast": False},
        # the gate with fp32 parameters over a window's worth of tokens, odd length
        {"name": "gate_fp32_1001", "kind": "gate", "S": 1001, "Hkv": 8, "D": 128, "expand": 4.0, "param": "fp32",
         "fast": True},
        # the decoder's row-wise work of one 4096-token prompt chunk
        {"name": "rows_4k", "kind": "rows", "rows": 4096, "hidden": 4096, "ffn": 14336, "qk_norm": False, **heads},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    Hkv = rng.choice([2, 4, 8, 8, 8])
    G = rng.choice([1, 2, 4, 4, 4, 8])
    heads = {"Hq": Hkv * G, "Hkv": Hkv, "D": rng.choice([64, 128, 128])}
    W = rng.choice([128, 256, 1024])
    kind = rng.choice(["decode", "decode", "decode", "quest", "oneshot", "oneshot", "chunked", "gate", "gate", "rows",
                       "step"])
    if kind == "decode":
        B = _log_int(rng, 1, 32)
        return {"kind": kind, "B": B, "ctx": _log_int(rng, W + 64, max(2048, min(131072, 1048576 // B))), "W": W,
                "page": rng.choice([16, 16, 32, 64]), **heads}
    if kind == "quest":
        return {"kind": kind, "ctx": _log_int(rng, 8192, 131072), "W": W, "frac": round(rng.uniform(0.05, 0.4), 3),
                "budget": W + 16 * _log_int(rng, 16, 256), **heads}
    if kind == "oneshot":
        return {"kind": kind, "S": _log_int(rng, 130, 16000), "W": W, "frac": round(rng.uniform(0.02, 0.6), 3), **heads}
    if kind == "chunked":
        chunk = rng.choice([1024, 2048, 4096])
        n = rng.randint(2, 6)
        return {"kind": kind, "S": chunk * (n - 1) + rng.randint(1024, chunk), "chunk": chunk, "W": W,
                "frac": round(rng.uniform(0.02, 0.4), 3), **heads}
    if kind == "gate":
        return {"kind": kind, "S": _log_int(rng, 5, 8192), "Hkv": Hkv, "D": heads["D"],
                "expand": rng.choice([1.5, 4.0, 4.0]), "param": rng.choice(["bf16", "bf16", "fp32"]),
                "fast": rng.random() < 0.5}
    if kind == "step":
        hidden = rng.choice([1024, 2048, 4096])
        return {"kind": kind, "layers": rng.choice([1, 2]), "ctx": 64 * rng.randint(20, 128), "vocab": 32000,
                "hidden": hidden, "ffn": hidden * 3, "W": rng.choice([256, 1024]),
                "frac": round(rng.uniform(0.1, 0.4), 3), "qk_norm": rng.random() < 0.5,
                "Hq": hidden // 128, "Hkv": hidden // 512, "D": 128}
    hidden = rng.choice([1024, 2048, 4096])
    return {"kind": "rows", "rows": _log_int(rng, 2, 4096), "hidden": hidden, "ffn": 64 * rng.randint(32, 200),
            "qk_norm": rng.random() < 0.5, **heads}


# ---- inputs -----------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(BF16)


def _decode_lengths(c, seed):
    """Cached tokens per (sequence, head): the window plus a fraction spread
    evenly over 2-60 % of the rest, dealt to the heads in a random order (the
    total does not depend on the seed)."""
    n = c["B"] * c["Hkv"]
    lens = [c["W"] + round((0.02 + 0.58 * (i + 0.5) / n) * (c["ctx"] - c["W"])) for i in range(n)]
    random.Random(seed).shuffle(lens)
    return torch.tensor(lens, dtype=torch.int64).view(c["B"], c["Hkv"])


def _prep_decode(c, seed):
    g = _gen(seed)
    lens, P, D = _decode_lengths(c, seed), c["page"], c["D"]
    pages = (lens + P - 1) // P
    total, width = int(pages.sum()), int(pages.max())
    perm = torch.randperm(total, generator=g, device="cuda").to(torch.int32)
    n = pages.flatten().cuda()
    idx = torch.arange(width, device="cuda")[None]
    src = ((torch.cumsum(n, 0) - n)[:, None] + idx).clamp(max=total - 1)
    table = torch.where(idx < n[:, None], perm[src], torch.full_like(src, -1, dtype=torch.int32))
    return {"q": _randn(g, c["B"], 1, c["Hq"], D), "k": _randn(g, total, P, D), "v": _randn(g, total, P, D),
            "lens": lens.to(torch.int32).cuda(), "table": table.view(c["B"], c["Hkv"], width).contiguous(),
            "scale": D ** -0.5}


def _config(c, per_head, layers=1, **kw):
    return WGKVConfig(num_hidden_layers=layers, num_attention_heads=c["Hq"], num_key_value_heads=c["Hkv"],
                      head_dim=c["D"], hidden_size=c["Hq"] * c["D"], local_window_size=c["W"],
                      max_tokens_per_head=per_head, max_total_tokens=layers * c["Hkv"] * (per_head + c["W"]),
                      check_capacity=False, **kw)


def _cache(cfg, c):
    cache = DualCache()
    cache.initialize(cfg, c["D"], BF16, torch.device("cuda"))
    cache.block_pool_k.zero_()
    cache.block_pool_v.zero_()
    if cache.local_pre_key is not None:
        cache.local_pre_key.zero_()
    return cache


def _mask(c, g, S):
    """Admission flags: each head has its own rate around ``frac``."""
    rate = c["frac"] * torch.linspace(0.6, 1.4, c["Hkv"], device="cuda")
    return torch.rand(c["Hkv"], S, generator=g, device="cuda") < rate[:, None]


def _prep_quest(c, seed):
    g = _gen(seed)
    H, S, D = c["Hkv"], c["ctx"], c["D"]
    cache = _cache(_config(c, S + c["W"], use_quest=True, quest_token_budget=c["budget"]), c)
    cache.quest_block_key_min.zero_()
    cache.quest_block_key_max.zero_()
    k, v = _randn(g, H, S, D), _randn(g, H, S, D)
    ops.prefill_admit(cache, 0, k, v, _mask(c, g, S))
    ops.quest_update_bounds(cache, 0)
    cache.local_length = c["W"]
    return {"cache": cache, "q": _randn(g, 1, 1, c["Hq"], D), "scale": D ** -0.5}


def _qkv_views(c, g, S):
    """q, k, v as the projection and rotary launch leave them: (1, H, S, D)
    views of one (1, S, Hq + 2 Hkv, D) buffer."""
    Hq, Hkv = c["Hq"], c["Hkv"]
    buf = _randn(g, 1, S, Hq + 2 * Hkv, c["D"])
    return (buf[:, :, :Hq].transpose(1, 2), buf[:, :, Hq:Hq + Hkv].transpose(1, 2), buf[:, :, Hq + Hkv:].transpose(1, 2))


def _prep_prefill(c, seed):
    g = _gen(seed)
    S = c["S"]
    oneshot = c["kind"] == "oneshot"
    # one-shot: a middle layer, so that the wrapper neither makes the cache nor ends the prompt
    cfg = _config(c, S + c["W"], layers=3 if oneshot else 1, g_defer=True)
    cache = _cache(cfg, c)
    q, k, v = _qkv_views(c, g, S)
    s = {"cache": cache, "q": q, "k": k, "v": v, "pre": _randn(g, 1, S, c["Hkv"], c["D"]).transpose(1, 2),
         "mask": _mask(c, g, S)[None], "free": cache.next_free_block_dev.clone()}
    if oneshot:
        with torch.device("cuda"):
            s["attn"] = LlamaAttention(cfg, 1).to(BF16)
    else:
        s["out"] = torch.zeros(S, c["Hq"], c["D"], dtype=BF16, device="cuda")
        s["spans"] = e2e.prompt_chunks(S, c["chunk"], c["W"])
    return s


def _gate_module(c, seed):
    torch.manual_seed(seed)
    with torch.device("cuda"):
        gate = GatingPredictor(c["D"], c["Hkv"], ["pre_k", "post_k"], "gelu", c["expand"], 1e-3, True, c["fast"])
    return gate.to(BF16 if c["param"] == "bf16" else torch.float32)


def _prep_gate(c, seed):
    g = _gen(seed)
    S, H, D = c["S"], c["Hkv"], c["D"]
    gate = _gate_module(c, seed)
    with torch.no_grad():  # a trained gate's norms are near one, its bias admits some of the tokens
        for m in (gate.pre_key_norm, gate.post_key_norm):
            m.weight += 0.1 * torch.randn(D, generator=g, device="cuda").to(m.weight.dtype)
        gate.conv2.bias -= 2.0
    pre, post = _randn(g, 1, S, H, D).transpose(1, 2), _randn(g, 1, S, H, D).transpose(1, 2)
    return {"gate": gate, "pre": pre, "post": post}


def _prep_rows(c, seed):
    g = _gen(seed)
    n, D = c["rows"], c["D"]
    with torch.device("cuda"):
        norm = e2e.RMSNorm(c["hidden"]).to(BF16)
        hq, hk = _randn(g, D) * 0.1 + 1.0, _randn(g, D) * 0.1 + 1.0
    norm.weight.data += 0.1 * _randn(g, c["hidden"])
    q, k, v = _qkv_views(c, g, n)
    ang = torch.arange(n, device="cuda", dtype=torch.float64)[:, None] * \
        10000.0 ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    ang = torch.cat((ang, ang), -1)[None]
    gu = _randn(g, 1, n, 2 * c["ffn"])
    return {"norm": norm, "x": _randn(g, 1, n, c["hidden"]), "res": _randn(g, 1, n, c["hidden"]),
            "q": q, "k": k, "v": v, "cos": ang.cos().to(BF16), "sin": ang.sin().to(BF16),
            "nw": (hq.contiguous(), hk.contiguous()) if c["qk_norm"] else None,
            "g": gu[..., :c["ffn"]], "u": gu[..., c["ffn"]:]}


def _prep_step(c, seed):
    # room for the tokens of some ten thousand further steps
    per_head = c["ctx"] + 2 * c["W"] + 32768
    ec = e2e.E2EConfig(hidden_size=c["hidden"], intermediate_size=c["ffn"], num_hidden_layers=c["layers"],
                       num_attention_heads=c["Hq"], num_key_value_heads=c["Hkv"], vocab_size=c["vocab"],
                       local_window_size=c["W"], qk_norm=c["qk_norm"])
    torch.manual_seed(seed)
    prev = torch.get_default_dtype()
    torch.set_default_dtype(BF16)
    try:
        with torch.device("cuda"):
            model = e2e.LlamaLite(ec, gated=True, max_tokens_per_head=per_head,
                                  max_total_tokens=c["layers"] * c["Hkv"] * per_head)
    finally:
        torch.set_default_dtype(prev)
    model.init_weights(seed=seed)
    g = _gen(seed)
    ids = torch.randint(0, c["vocab"], (1, c["ctx"]), generator=g, device="cuda")
    e2e.calibrate_gates(model, ids, c["frac"], chunk=min(4096, c["ctx"]))
    cache = DualCache()
    for c0, c1 in e2e.prompt_chunks(c["ctx"], 4096, c["W"]):
        model.forward_tokens(ids[:, c0:c1], c0, cache)
    token = torch.randint(0, c["vocab"], (1, 1), generator=g, device="cuda")
    return {"decoder": e2e.GraphDecoder(model, cache, token, c["ctx"]), "token": token}


_PREPARE = {"decode": _prep_decode, "quest": _prep_quest, "step": _prep_step, "oneshot": _prep_prefill,
            "chunked": _prep_prefill, "gate": _prep_gate, "rows": _prep_rows}


@torch.no_grad()
def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    state["case"] = case
    return state


# ---- one pass ---------------------------------------------------------------
def _run_decode(c, s):
    return ops.paged_decode_attn(s["q"], s["k"], s["v"], s["lens"], s["table"], s["scale"])


def _run_quest(c, s):
    cache = s["cache"]
    lens, table = ops.quest_select(cache, 0, s["q"][0, 0], c["W"], c["budget"])
    out = ops.paged_decode_attn(s["q"], cache.k_cache(), cache.v_cache(), lens, table, s["scale"])
    return {"out": out, "lens": lens, "table": table}


def _run_step(c, s):
    # the caller's own sampler chose the token; the cache and the position move on
    d = s["decoder"]
    d.tok.copy_(s["token"])
    d.step()
    return {"logits": d.logits}


def _run_oneshot(c, s):
    cache, attn, S = s["cache"], s["attn"], c["S"]
    cache.next_free_block_dev.copy_(s["free"])  # the pool's pages go to the next prompt
    out = attn.prefill_wrapper(attn, cache, s["q"], s["pre"], s["k"], s["v"], 1, S, s["q"].device, s["mask"],
                               c["W"] // cache.block_size)
    return {"out": out, "lengths": cache.global_lengths, "flags": cache.local_is_global, "table": cache.block_table,
            "free": cache.next_free_block_dev, "pool_k": cache.block_pool_k, "pool_v": cache.block_pool_v,
            "pre": cache.local_pre_key}


def _run_chunked(c, s):
    cache = s["cache"]
    cache.next_free_block_dev.copy_(s["free"])  # the pool's pages go to the next prompt
    cache.global_lengths.zero_()
    q, k, v = s["q"][0].transpose(0, 1), s["k"][0].transpose(0, 1), s["v"][0].transpose(0, 1)
    pre = s["pre"][0].transpose(0, 1)
    for c0, c1 in s["spans"]:
        ops.chunk_prefill(cache, 0, q[c0:c1], k[c0:c1], v[c0:c1], s["mask"][0, :, c0:c1], c0, pre_key=pre[c0:c1],
                          out=s["out"][c0:c1])
    return {"out": s["out"], "lengths": cache.global_lengths, "flags": cache.local_is_global,
            "table": cache.block_table, "free": cache.next_free_block_dev, "pool_k": cache.block_pool_k,
            "pool_v": cache.block_pool_v, "pre": cache.local_pre_key}


def _run_gate(c, s):
    scores, mask = s["gate"].scores_and_mask(s["pre"], s["post"], None, 0.1)
    return {"scores": scores, "mask": mask}


def _run_rows(c, s):
    h, x = s["norm"](s["x"], residual=s["res"])
    nw = s["nw"]
    if nw is None:
        rot = model_ops.rope_qkv(s["q"], s["k"], s["v"], s["cos"], s["sin"])
    else:
        rot = model_ops.rope_qkv(s["q"], s["k"], s["v"], s["cos"], s["sin"], nw[0], nw[1], 1e-6)
    return {"normed": h, "stream": x, "rotated": rot, "act": model_ops.silu_mul(s["g"], s["u"])}


_RUN = {"decode": _run_decode, "quest": _run_quest, "step": _run_step, "oneshot": _run_oneshot,
        "chunked": _run_chunked, "gate": _run_gate, "rows": _run_rows}


@torch.no_grad()
def run(state):
    c = state["case"]
    return _RUN[c["kind"]](c, state)


# ---- what a pass cannot do without -------------------------------------------
def _visible(S, W, frac):
    """Expected number of visible (query, key) pairs of one query head."""
    pairs = 0.0
    for r in range((S + BLK - 1) // BLK):
        rows = min(BLK, S - r * BLK)
        start = max(0, r * BLK - W + 1)
        pairs += rows * (r * BLK - start) + rows * (rows + 1) / 2 + rows * frac * start
    return pairs


def work(case):
    c = case
    kind = c["kind"]
    if kind == "decode":
        T = int(_decode_lengths(c, 0).sum())
        return {"bytes": T * c["D"] * 4 + T // c["page"] * 4 + 2 * c["B"] * c["Hq"] * c["D"] * 2,
                "flops": 4.0 * T * c["D"] * (c["Hq"] // c["Hkv"])}
    if kind == "quest":
        pages = c["Hkv"] * c["frac"] * (c["ctx"] - c["W"]) / 16
        T = c["Hkv"] * min(c["budget"], c["W"] + c["frac"] * (c["ctx"] - c["W"]))
        return {"bytes": pages * c["D"] * 4 + T * c["D"] * 4 + 2 * c["Hq"] * c["D"] * 2,
                "flops": (2.0 * pages + 4.0 * T / 1) * c["D"] * (c["Hq"] // c["Hkv"])}
    if kind == "step":
        h, Hq, Hkv, D = c["hidden"], c["Hq"], c["Hkv"], c["D"]
        weights = c["layers"] * (h * (Hq + 2 * Hkv) * D + Hq * D * h + 3 * h * c["ffn"]) + h * c["vocab"]
        kv = c["layers"] * Hkv * (c["W"] + c["frac"] * (c["ctx"] - c["W"])) * D * 2
        return {"bytes": 2.0 * (weights + kv), "flops": 2.0 * weights + 2.0 * kv * (Hq // Hkv)}
    if kind in ("oneshot", "chunked"):
        S, D, Hq, Hkv = c["S"], c["D"], c["Hq"], c["Hkv"]
        kept = Hkv * (min(S, c["W"]) + c["frac"] * max(0, S - c["W"]))
        return {"bytes": 2.0 * S * D * (2 * Hq + 2 * Hkv) + kept * D * 4 + Hkv * min(S, c["W"]) * D * 4 + Hkv * S,
                "flops": 4.0 * D * Hq * _visible(S, c["W"], c["frac"])}
    if kind == "gate":
        H, S, D = c["Hkv"], c["S"], c["D"]
        inner = int(D * c["expand"])
        weight = H * inner * (2 * D + 2) * (2 if c["param"] == "bf16" else 4)
        return {"bytes": 2.0 * 2 * S * H * D + weight + 5.0 * S * H, "flops": 2.0 * S * H * inner * (2 * D + 1)}
    n, h = c["rows"], c["hidden"]
    head_rows = n * (c["Hq"] + 2 * c["Hkv"]) * c["D"]
    kn = n * c["Hkv"] * c["D"] if c["qk_norm"] else 0
    return {"bytes": 2.0 * (4 * n * h + 2 * head_rows + kn + 2 * n * c["D"] + 3 * n * c["ffn"]),
            "flops": 6.0 * n * h + 4.0 * head_rows + 6.0 * n * c["ffn"]}


def tolerance(case):
    return {
        # bf16 inputs, outputs and probabilities
        "decode": {"rel": 1e-2, "max": 0.2},
        "quest": {"rel": 1e-2, "max": 0.2, "differ": 0.0},
        "step": {"rel": 2e-2, "max": 0.3},
        "oneshot": {"rel": 1e-2, "max": 0.3, "differ": 0.0},
        "chunked": {"rel": 1e-2, "max": 0.3, "differ": 0.0},
        # scores: bf16 values with bf16 parameters, fp32 sums with fp32 ones; the
        # flags of scores within that of the threshold may differ
        "gate": {"rel": 5e-3, "max": 0.2, "differ": 5e-3} if case.get("param") == "bf16"
        else {"rel": 1e-5, "max": 1e-2, "differ": 1e-3},
        "rows": {"rel": 5e-3, "max": 0.05},
    }[case["kind"]]


# ---- the same in 64 bits -----------------------------------------------------
def _attend64(q, k, v, scale, visible=None):
    """q (G, n, D), k / v (m, D), visible (n, m) or None -> (G, n, D), in 64 bits."""
    s = torch.matmul(q.double(), k.double().t()) * scale
    if visible is not None:
        s = s.masked_fill(~visible, -math.inf)
    return torch.matmul(torch.softmax(s, -1), v.double())


def _paged64(q, k, v, lens, table, scale):
    B, _, Hq, D = q.shape
    Hkv, P = lens.shape[1], k.shape[1]
    G = Hq // Hkv
    out = torch.empty(B, 1, Hq, D, dtype=torch.float64, device=q.device)
    for b in range(B):
        for h in range(Hkv):
            n = int(lens[b, h])
            pages = table[b, h, :(n + P - 1) // P].long()
            kk, vv = k[pages].reshape(-1, D)[:n], v[pages].reshape(-1, D)[:n]
            out[b, 0, h * G:(h + 1) * G] = _attend64(q[b, 0, h * G:(h + 1) * G, None], kk, vv, scale)[:, 0]
    return out


def _prefill64(c, s):
    S, G, W = c["S"], c["Hq"] // c["Hkv"], c["W"]
    out = torch.empty(S, c["Hq"], c["D"], dtype=torch.float64, device="cuda")
    rows = 1024
    j = torch.arange(S, device="cuda")
    for r0 in range(0, S, rows):
        i = torch.arange(r0, min(S, r0 + rows), device="cuda")
        n = int(i[-1]) + 1
        band = j[None, :n] >= (i // BLK * BLK - W + 1)[:, None]
        causal = j[None, :n] <= i[:, None]
        for h in range(c["Hkv"]):
            vis = causal & (band | s["mask"][0, h, None, :n])
            out[i[0]:n, h * G:(h + 1) * G] = _attend64(s["q"][0, h * G:(h + 1) * G, i], s["k"][0, h, :n],
                                                       s["v"][0, h, :n], c["D"] ** -0.5, vis).transpose(0, 1)
    return out


def _quest64(c, s):
    """QUEST's selection with its page scores rounded to bf16 where the
    reference's bf16 ops round them, and the attention over it."""
    cache, H, P, W = s["cache"], c["Hkv"], 16, c["W"]
    G, lb = c["Hq"] // c["Hkv"], c["W"] // 16
    width = lb + (max(c["budget"] - W, 0) + P - 1) // P + 1
    lens = torch.zeros(1, H, dtype=torch.int32, device="cuda")
    table = torch.zeros(1, H, width, dtype=torch.int32, device="cuda")
    for h in range(H):
        n = int(cache.global_lengths[0, h])
        full, rem = n // P, n % P
        cap = min((max(c["budget"] - W, 0) + P - 1) // P, (n + P - 1) // P)
        keep = max(0, min(full, cap - (1 if rem else 0)))
        glob = cache.block_table[0, h, lb:]
        pages = glob[:full].long()
        lo, hi = cache.quest_block_key_min[pages], cache.quest_block_key_max[pages]
        q = s["q"][0, 0, h * G:(h + 1) * G, None]
        prod = q * torch.where(q >= 0, hi[None], lo[None])  # bf16 products
        score = prod.double().sum(-1).to(BF16).double().max(0).values
        order = torch.sort(score, descending=True, stable=True).indices[:keep].sort().values
        ids = torch.cat((cache.block_table[0, h, :lb], glob[order], glob[full:full + 1][:1 if cap > 0 and rem else 0]))
        table[0, h, :ids.numel()] = ids
        lens[0, h] = W + keep * P + (rem if cap > 0 and rem else 0)
    return {"out": _paged64(s["q"], cache.k_cache(), cache.v_cache(), lens, table, s["scale"]), "lens": None,
            "table": None}


def _gate64(c, s):
    gate, H, D = s["gate"], c["Hkv"], c["D"]
    inner = int(D * c["expand"])
    x = []
    for t, m in ((s["pre"], gate.pre_key_norm), (s["post"], gate.post_key_norm)):
        t = t[0].double()
        t = (t * torch.rsqrt(t.pow(2).mean(-1, keepdim=True) + 1e-6)).to(BF16).double()  # cast to the input's type
        x.append(t * m.weight.double())
    x = torch.cat(x, -1)
    w1 = gate.conv1.weight.double().view(H, inner, 2 * D)
    z = torch.matmul(x, w1.transpose(1, 2).contiguous()) + gate.conv1.bias.double().view(H, 1, inner)
    z = torch.nn.functional.gelu(z)
    z = (z * gate.conv2.weight.double().view(H, 1, inner)).sum(-1) + gate.conv2.bias.double().view(H, 1)
    g = torch.sigmoid(z)
    return {"scores": (g if c["fast"] else g.clamp(min=1e-3))[None], "mask": None}


def _rows64(c, s):
    def norm(x, w, eps):
        return w * (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps))

    def rotate(x):
        half = x.shape[-1] // 2
        turned = torch.cat((-x[..., half:], x[..., :half]), -1)
        return x * s["cos"].double()[:, None] + turned * s["sin"].double()[:, None]

    x = s["x"].double() + s["res"].double()
    q, k, v = s["q"].double(), s["k"].double(), s["v"].double()
    if s["nw"] is not None:
        q, k = norm(q, s["nw"][0].double(), 1e-6), norm(k, s["nw"][1].double(), 1e-6)
    rot = (rotate(q), rotate(k), v) + ((k,) if s["nw"] is not None else ())
    return {"normed": norm(x, s["norm"].weight.double(), s["norm"].eps), "stream": x, "rotated": rot,
            "act": torch.nn.functional.silu(s["g"].double()) * s["u"].double()}


@torch.no_grad()
def exact(case, seed):
    c = case
    if c["kind"] == "step":
        return None  # a whole model: its gates' flags follow bf16 roundings that 64 bits do not make
    s = prepare(c, seed)
    if c["kind"] == "decode":
        return _paged64(s["q"], s["k"], s["v"], s["lens"], s["table"], s["scale"])
    if c["kind"] in ("oneshot", "chunked"):
        out = _prefill64(c, s)
        none = {k: None for k in ("lengths", "flags", "table", "free", "pool_k", "pool_v", "pre")}
        return {"out": out[None] if c["kind"] == "oneshot" else out, **none}
    return {"quest": _quest64, "gate": _gate64, "rows": _rows64}[c["kind"]](c, s)
