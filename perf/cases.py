"""Timed cases of the framework's public entry points: what a tensor-parallel, expert-parallel or sequence-parallel
inference program asks of one GPU, from a single decode step to a long prefill.

``listed()`` holds the named cases, ``draw(rng)`` gives further ones of the same ranges, ``prepare`` makes the inputs and
the context that a program keeps, ``run`` is one pass, ``work`` what the pass cannot do without and ``tolerance`` how far
another correct implementation may be off."""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "triton-distributed_amd"))

from triton_dist.kernels.amd import (  # noqa: E402
    ag_gemm_intra_node, ag_group_gemm_intra_node, create_ag_gemm_intra_node_context,
    create_ag_group_gemm_intra_node_context, create_all_to_all_context, create_gemm_rs_intra_node_context,
    create_moe_rs_context, fast_all_to_all, gemm_rs_intra_node, gqa_fwd_batch_decode, moe_dispatch_preprocess,
    moe_reduce_rs, moe_weighted_combine, select_experts, sort_topk_ids_align_block_size)
from triton_dist.layers.amd.sp_flash_decode_layer import SpGQAFlashDecodeAttention  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "e4m3": torch.float8_e4m3fn}
BYTES = {"bf16": 2, "f16": 2, "e4m3": 1}
MOST_FLOPS = 1.9e12   # drawn cases stay within the largest listed ones
MOST_KV_BYTES = 4.3e9


def listed():
    return [
        # A decode step's batch through a tensor-parallel projection: few rows per rank, no multiple of a tile.
        {"name": "ag_gemm_decode_bf16", "op": "ag_gemm", "dtype": "bf16", "world": 4, "m_per_rank": 50, "chunk": 50,
         "N": 1536, "K": 4096},
        # The gate + up projection of a 70B model split over 8 GPUs, a long prefill in e4m3 with row and column scales.
        {"name": "ag_gemm_prefill_e4m3", "op": "ag_gemm", "dtype": "e4m3", "world": 8, "m_per_rank": 2048, "chunk": 2048,
         "N": 7168, "K": 8192},
        # The output projection behind a short prompt, f16: the GEMM no longer fills the chip.
        {"name": "gemm_rs_short_f16", "op": "gemm_rs", "dtype": "f16", "world": 8, "m_per_rank": 128, "N": 4096, "K": 1536},
        # The down projection of the same 70B model, 8192 tokens in bf16.
        {"name": "gemm_rs_prefill_bf16", "op": "gemm_rs", "dtype": "bf16", "world": 8, "m_per_rank": 1024, "N": 8192,
         "K": 3584},
        # Expert-parallel dispatch and combine of one decode step: 128 tokens, ids as torch.topk gives them.
        {"name": "moe_a2a_decode", "op": "moe_a2a", "dtype": "e4m3", "ids": "int64", "tokens": 128, "topk": 8,
         "experts": 256, "world": 32, "hidden": 7168, "max_m": 128},
        # The same for a prefill's 4096 tokens.
        {"name": "moe_a2a_prefill", "op": "moe_a2a", "dtype": "e4m3", "ids": "int32", "tokens": 4096, "topk": 8,
         "experts": 256, "world": 32, "hidden": 7168, "max_m": 4096},
        # bf16 activations quantised in groups of 128 columns on their way out, the routing sorted for the grouped GEMM
        # that follows, an ordinary number of tokens that is no power of two.
        {"name": "moe_a2a_quant", "op": "moe_quant", "tokens": 1000, "segments": 8, "topk": 8, "experts": 256, "world": 32,
         "hidden": 7168, "block": 128},
        # A Mixtral-8x7B feed-forward layer split over 8 GPUs: gathered tokens through the experts' up projection, then the
        # down projection, the weighted sum over the experts and the reduce-scatter (the activation between is the model's).
        {"name": "moe_tp_layer", "op": "moe_layer", "world": 8, "m_per_rank": 1024, "topk": 2, "experts": 8, "hidden": 4096,
         "inter": 1792},
        # One user, a short context.
        {"name": "decode_single", "op": "decode", "dtype": "bf16", "batch": 1, "q_heads": 32, "kv_heads": 8, "dim": 128,
         "dim_v": 128, "page": 16, "longest": 1320, "even": True, "soft_cap": 0.0},
        # A serving batch: many users, contexts of every length.
        {"name": "decode_serving_f16", "op": "decode", "dtype": "f16", "batch": 48, "q_heads": 64, "kv_heads": 8, "dim": 128,
         "dim_v": 128, "page": 16, "longest": 8192, "even": False, "soft_cap": 0.0},
        # Latent attention: every query head on one 576-wide key whose first 512 columns are the value.
        {"name": "decode_latent_bf16", "op": "decode", "dtype": "bf16", "batch": 16, "q_heads": 128, "kv_heads": 1, "dim": 576,
         "dim_v": 512, "page": 16, "longest": 4096, "even": False, "soft_cap": 0.0},
        # A sequence-parallel layer over long contexts: this GPU's shard of 32 x 262144 keys, merged with 7 peers' partials.
        {"name": "sp_decode_long", "op": "sp_decode", "dtype": "bf16", "world": 8, "batch": 32, "q_heads": 64, "kv_heads": 8,
         "dim": 128, "page": 16, "longest": 32768, "even": True},
    ]


# ---- drawn cases -------------------------------------------------------------------------------------------------
def _log(rng, lo, hi, step=1):
    """A whole multiple of ``step`` from lo to hi, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(-(-lo // step) * step, min(hi // step * step, int(round(v / step)) * step))


def _draw_ag_gemm(rng):
    while True:
        m = _log(rng, 16, 2048)
        chunk = m
        if m >= 128 and rng.random() < 0.5:   # whole tiles; the others are chunks of any number of rows
            m = m // 128 * 128
            chunk = m // 2 if m % 256 == 0 and rng.random() < 0.5 else m
        c = {"op": "ag_gemm", "dtype": rng.choice(["bf16", "f16", "e4m3"]), "world": rng.choice([2, 4, 8]), "m_per_rank": m,
             "chunk": chunk, "N": _log(rng, 512, 8192, 8), "K": _log(rng, 1024, 8192, 16)}
        if work(c)["flops"] * BYTES[c["dtype"]] <= MOST_FLOPS:
            return c


def _draw_gemm_rs(rng):
    while True:
        c = {"op": "gemm_rs", "dtype": rng.choice(["bf16", "f16", "e4m3"]), "world": rng.choice([2, 4, 8]),
             "m_per_rank": _log(rng, 128, 2048, 128), "N": _log(rng, 1024, 8192, 256), "K": _log(rng, 512, 8192, 256)}
        if work(c)["flops"] * BYTES[c["dtype"]] <= MOST_FLOPS:
            return c


def _capacity(tokens, topk, world, per):
    """Rows of a slot: twice an even share and some, at most what could ever be sent to one rank."""
    return min(tokens * min(topk, per), 2 * tokens * topk // world + 64)


def _draw_moe_a2a(rng):
    T, topk = _log(rng, 1, 4096), rng.choice([2, 4, 6, 8])
    world, per = rng.choice([(8, 8), (8, 32), (16, 8), (16, 16), (32, 8)])
    return {"op": "moe_a2a", "dtype": rng.choice(["e4m3", "e4m3", "bf16"]), "ids": rng.choice(["int32", "int64"]), "tokens": T,
            "topk": topk, "experts": world * per, "world": world, "hidden": rng.choice([2048, 4096, 5120, 7168]),
            "max_m": _capacity(T, topk, world, per)}


def _draw_moe_quant(rng):
    segments = 8
    return {"op": "moe_quant", "tokens": segments * _log(rng, 1, 512), "segments": segments, "topk": rng.choice([2, 4, 6, 8]),
            "experts": rng.choice([64, 128, 256]), "world": rng.choice([8, 16, 32]),
            "hidden": rng.choice([2048, 4096, 5120, 7168]), "block": rng.choice([64, 128])}


def _draw_moe_layer(rng):
    while True:
        c = {"op": "moe_layer", "world": rng.choice([2, 4, 8]), "m_per_rank": _log(rng, 8, 1024), "topk": rng.choice([2, 4, 6]),
             "experts": rng.choice([8, 16, 32, 64]), "hidden": _log(rng, 1024, 7168, 128), "inter": _log(rng, 256, 2048, 128)}
        if work(c)["flops"] <= 0.5 * MOST_FLOPS and work(c)["bytes"] <= 2e9:
            return c


def _draw_decode(rng):
    while True:
        hq, hkv, dim, dim_v = rng.choice([(32, 8, 128, 128), (64, 8, 128, 128), (16, 16, 128, 128), (32, 8, 64, 64), (6, 1, 128, 128),
                                          (32, 8, 256, 256), (32, 8, 96, 96), (128, 1, 576, 512)])
        c = {"op": "decode", "dtype": rng.choice(["bf16", "f16"]), "batch": _log(rng, 1, 64), "q_heads": hq, "kv_heads": hkv,
             "dim": dim, "dim_v": dim_v, "page": rng.choice([1, 16]), "longest": _log(rng, 64, 16384),
             "even": rng.random() < 0.3, "soft_cap": rng.choice([0.0, 0.0, 30.0])}
        if work(c)["bytes"] <= MOST_KV_BYTES:
            return c


def _draw_sp_decode(rng):
    while True:
        hq, hkv = rng.choice([(32, 8), (64, 8), (16, 16)])
        c = {"op": "sp_decode", "dtype": rng.choice(["bf16", "f16"]), "world": rng.choice([2, 4, 8]), "batch": _log(rng, 1, 32),
             "q_heads": hq, "kv_heads": hkv, "dim": 128, "page": rng.choice([1, 16]), "longest": _log(rng, 1024, 32768),
             "even": rng.random() < 0.5}
        if work(c)["bytes"] <= MOST_KV_BYTES:
            return c


def draw(rng):
    return rng.choice([_draw_ag_gemm, _draw_gemm_rs, _draw_moe_a2a, _draw_moe_quant, _draw_moe_layer, _draw_decode,
                       _draw_decode, _draw_sp_decode])(rng)


# ---- inputs ------------------------------------------------------------------------------------------------------
def _randn(g, shape, dtype, scale=1.0):
    """Normal values times ``scale`` in ``dtype`` (e4m3 by way of bf16)."""
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float16 if dtype == torch.float16 else torch.bfloat16)
    if scale != 1.0:
        x = x.mul_(scale)
    return x if x.dtype == dtype else x.to(dtype)


def _uniform(g, n, lo, hi):
    return torch.rand(n, generator=g, device="cuda") * (hi - lo) + lo


def _prepare_ag_gemm(c, g):
    W, mpr, K, N, dtype = c["world"], c["m_per_rank"], c["K"], c["N"], DTYPES[c["dtype"]]
    rank = W // 2
    out = torch.bfloat16 if c["dtype"] == "e4m3" else dtype
    ctx = create_ag_gemm_intra_node_context(W * mpr, N, K, dtype, out, rank, W, None, M_PER_CHUNK=c["chunk"],
                                            ragged_chunks=c["chunk"] % 128 != 0)
    shards = [_randn(g, (mpr, K), dtype) for _ in range(W)]
    ctx.set_peer_shards({r: s for r, s in enumerate(shards) if r != rank})
    scales = {}
    if c["dtype"] == "e4m3":
        scales = {"row_scale": _uniform(g, W * mpr, 0.01, 0.1), "col_scale": _uniform(g, N, 0.001, 0.01)}
    weight = _randn(g, (N, K), dtype, 1.0 if scales else 0.02)
    return {"ctx": ctx, "a": shards[rank], "b": weight, "scales": scales}


def _prepare_gemm_rs(c, g):
    W, mpr, K, N, dtype = c["world"], c["m_per_rank"], c["K"], c["N"], DTYPES[c["dtype"]]
    rank = W // 2
    out = torch.bfloat16 if c["dtype"] == "e4m3" else dtype
    ctx = create_gemm_rs_intra_node_context(W * mpr, N, out, rank, W, None)
    ctx.set_peer_partials({r: _randn(g, (mpr, N), out) for r in range(W) if r != rank})
    scales = {}
    if c["dtype"] == "e4m3":
        scales = {"row_scale": _uniform(g, W * mpr, 0.01, 0.1), "col_scale": _uniform(g, N, 0.001, 0.01)}
    weight = _randn(g, (N, K), dtype, 1.0 if scales else 0.02)
    return {"ctx": ctx, "a": _randn(g, (W * mpr, K), dtype), "b": weight, "scales": scales, "rank": rank, "mpr": mpr}


def _experts(g, tokens, experts, topk):
    """Distinct experts per token, chosen evenly at random, as int64."""
    return torch.rand((tokens, experts), generator=g, device="cuda").topk(topk, dim=1).indices


def _weights(g, tokens, topk):
    return torch.softmax(torch.randn((tokens, topk), generator=g, device="cuda"), dim=-1)


def _prepare_moe_a2a(c, g):
    T, H, W, G, dtype = c["tokens"], c["hidden"], c["world"], c["experts"], DTYPES[c["dtype"]]
    ctx = create_all_to_all_context(c["max_m"], H, 0, G, W, G // W, dtype=dtype)
    ctx.recv_buf.view(torch.uint8).zero_()   # the whole slots are returned, also the rows nobody sends to
    ctx.scale_recv_buf.zero_()
    ids = _experts(g, T, G, c["topk"])
    x = torch.randn((T, H), generator=g, device="cuda")
    scale = None
    if c["dtype"] == "e4m3":
        scale = x.abs().amax(dim=1) / 448.0
        x = x / scale[:, None]
    return {"ctx": ctx, "x": x.to(dtype), "scale": scale, "ids": ids.to(getattr(torch, c["ids"])), "w": _weights(g, T, c["topk"])}


def _prepare_moe_quant(c, g):
    T, H, W, G = c["tokens"], c["hidden"], c["world"], c["experts"]
    ctx = create_all_to_all_context(_capacity(T, c["topk"], W, G // W), H, 0, G, W, G // W, dtype=torch.float8_e4m3fn, fp8_group_size=128)
    ctx.recv_buf.view(torch.uint8).zero_()
    ctx.scale_recv_buf.zero_()
    return {"ctx": ctx, "x": _randn(g, (T, H), torch.bfloat16), "ids": _experts(g, T, G, c["topk"]), "w": _weights(g, T, c["topk"]),
            "experts": G, "segments": c["segments"], "per": T // c["segments"], "block": c["block"]}


def _prepare_moe_layer(c, g):
    W, mpr, E, H, I = c["world"], c["m_per_rank"], c["experts"], c["hidden"], c["inter"]
    rank, dev, bf16 = W // 2, torch.device("cuda", torch.cuda.current_device()), torch.bfloat16
    shards = [_randn(g, (mpr, H), bf16) for _ in range(W)]
    logits = [torch.randn((mpr, E), generator=g, device="cuda") for _ in range(W)]
    peers = {r: t for r, t in enumerate(logits) if r != rank}
    # weights as the entry points take them, [E, K, N], over rows that are contiguous along K
    up, down = _randn(g, (E, I, H), bf16, 0.02).transpose(1, 2), _randn(g, (E, H, I), bf16, 0.02).transpose(1, 2)
    ids, _ = select_experts(None, W, c["topk"], bf16, dev, logits[rank], peers, rank)
    ag = create_ag_group_gemm_intra_node_context(None, shards[rank], up, ids, E, max_M=W * mpr, rank=rank, num_ranks=W)
    ag.set_peer_shards({r: s for r, s in enumerate(shards) if r != rank})
    rs = create_moe_rs_context(None, rank, W, W, W * mpr, H, E, c["topk"], bf16, bf16, dev, 128, logits[rank], peers)
    rs.set_peer_partials({r: _randn(g, (mpr, H), bf16) for r in range(W) if r != rank})
    return {"ag": ag, "rs": rs, "a": shards[rank], "up": up, "down": down, "rank": rank, "world": W}


def _lengths(c, seed):
    """Context lengths of the batch, on the host: all of them the longest, or spread over a factor of 64 below it."""
    if c["even"]:
        return [c["longest"]] * c["batch"]
    r = torch.rand(c["batch"], generator=torch.Generator().manual_seed(seed + 77))
    lens = [max(1, int(c["longest"] * 64.0 ** -float(v))) for v in r]
    lens[0] = c["longest"]
    return lens


def _paged_cache(c, g, seed, dim_v):
    """A paged cache in which every sequence's pages lie at random places: keys, values, page table and lengths. Where
    the value is a part of the key (latent attention) there is one cache, and the values are a view of it."""
    lens, page, dtype = _lengths(c, seed), c["page"], DTYPES[c["dtype"]]
    need = [-(-n // page) for n in lens]
    total = sum(need)
    k = _randn(g, (total, page, c["kv_heads"], c["dim"]), dtype)
    v = k[..., :dim_v] if dim_v < c["dim"] else _randn(g, (total, page, c["kv_heads"], dim_v), dtype)
    place = torch.randperm(total, generator=g, device="cuda", dtype=torch.int32)
    table = torch.zeros((c["batch"], max(need)), dtype=torch.int32, device="cuda")
    at = 0
    for b, n in enumerate(need):
        table[b, :n] = place[at:at + n]
        at += n
    return k, v, table, torch.tensor(lens, dtype=torch.int32, device="cuda")


def _prepare_decode(c, g, seed):
    k, v, table, lens = _paged_cache(c, g, seed, c["dim_v"])
    q = _randn(g, (c["batch"], c["q_heads"], c["dim"]), DTYPES[c["dtype"]])
    return {"q": q, "k": k, "v": v, "table": table, "lens": lens, "ones": [1] * c["batch"], "scale": c["dim"] ** -0.5,
            "soft_cap": c["soft_cap"]}


def _prepare_sp_decode(c, g, seed):
    B, W, Hq, D, dtype = c["batch"], c["world"], c["q_heads"], c["dim"], DTYPES[c["dtype"]]
    rank = W // 2
    k, v, table, lens = _paged_cache(c, g, seed, D)
    layer = SpGQAFlashDecodeAttention(rank, 0, W, 1, Hq, c["kv_heads"], D, D, page_size=c["page"], scale=D ** -0.5,
                                      max_allowed_batch=B)
    peers = (_randn(g, (W, B, Hq, D), dtype, 0.01), torch.randn((W, B, Hq), generator=g, device="cuda") * 0.2 + math.log(c["longest"]))
    return {"layer": layer, "q": _randn(g, (B, Hq, D), dtype), "k": k, "v": v, "table": table,
            "lens": lens.repeat(W, 1).contiguous(), "peers": peers}


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    op = case["op"]
    if op in ("decode", "sp_decode"):
        state = (_prepare_decode if op == "decode" else _prepare_sp_decode)(case, g, seed)
    else:
        state = {"ag_gemm": _prepare_ag_gemm, "gemm_rs": _prepare_gemm_rs, "moe_a2a": _prepare_moe_a2a,
                 "moe_quant": _prepare_moe_quant, "moe_layer": _prepare_moe_layer}[op](case, g)
    state["run"] = _RUN[op]
    return state


# ---- one pass ----------------------------------------------------------------------------------------------------
def _run_ag_gemm(s):
    return ag_gemm_intra_node(s["a"], s["b"], False, s["ctx"], **s["scales"])


def _run_gemm_rs(s):
    out = gemm_rs_intra_node(s["a"], s["b"], s["ctx"], **s["scales"])
    at, n = s["rank"] * s["mpr"], s["mpr"]
    return {"out": out, "sent": [b[at:at + n] for r, b in enumerate(s["ctx"].scatter_bufs) if r != s["rank"]]}


def _run_moe_a2a(s):
    ctx = s["ctx"]
    splits, recv, scales = fast_all_to_all(ctx, s["x"], None, s["scale"], expert_ids=s["ids"])
    _, cumsum, scatter, gather = ctx.last_index
    y = moe_weighted_combine(ctx, recv, scales, scatter, s["w"], cumsum)
    return {"splits": splits, "recv": recv.view(torch.uint8), "scales": scales, "cumsum": cumsum, "scatter": scatter,
            "gather": gather, "y": y}


def _run_moe_quant(s):
    ctx = s["ctx"]
    _, cumsum, scatter, gather = moe_dispatch_preprocess(s["ids"], s["experts"], ctx=ctx)
    splits, recv, scales = fast_all_to_all(ctx, s["x"], cumsum, None, scatter_index=scatter, online_quant_fp8=True)
    # (what the sort leaves behind the blocks in use is not written, so only the arrays that are written whole go back)
    rows, _, _, blocks, padded = sort_topk_ids_align_block_size(s["ids"], s["experts"], s["segments"], s["per"], s["block"])
    y = moe_weighted_combine(ctx, recv, scales, scatter, s["w"], cumsum)
    return {"splits": splits, "recv": recv.view(torch.uint8), "scales": scales, "cumsum": cumsum, "scatter": scatter,
            "gather": gather, "rows": rows, "blocks": blocks, "padded": padded, "y": y}


def _run_moe_layer(s):
    h = ag_group_gemm_intra_node(s["a"], s["up"], s["ag"])
    return {"h": h, "y": moe_reduce_rs(s["rank"], s["world"], s["world"], h, s["down"], s["rs"])}


def _run_decode(s):
    return gqa_fwd_batch_decode(s["q"], s["k"], s["v"], None, s["ones"], s["lens"], s["table"], s["scale"], s["soft_cap"])


def _run_sp_decode(s):
    out = s["layer"](s["q"], s["k"], s["v"], s["lens"], s["table"], s["peers"])
    return {"out": out, "gathered": s["peers"][0], "lse": s["peers"][1]}


_RUN = {"ag_gemm": _run_ag_gemm, "gemm_rs": _run_gemm_rs, "moe_a2a": _run_moe_a2a, "moe_quant": _run_moe_quant,
        "moe_layer": _run_moe_layer, "decode": _run_decode, "sp_decode": _run_sp_decode}


def run(state):
    return state["run"](state)


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def _work_gemm(c):
    e, M, N, K = BYTES[c["dtype"]], c["world"] * c["m_per_rank"], c["N"], c["K"]
    b = (M * K + N * K) * e + M * N * 2 + (4 * (M + N) if c["dtype"] == "e4m3" else 0)
    if c["op"] == "gemm_rs":   # the other owners' rows go out, the peers' partial rows come in, the sum goes out
        b += (c["world"] - 1) * c["m_per_rank"] * N * 2
    return {"bytes": b, "flops": 2 * M * N * K}


def _work_moe_a2a(c):
    T, H, n, e = c["tokens"], c["hidden"], c["tokens"] * c["topk"], BYTES[c["dtype"]]
    scales = 4 * (T + 2 * n) if c["dtype"] == "e4m3" else 0
    ids = n * (8 if c["ids"] == "int64" else 4)
    # dispatch: tokens in, slot rows out, index tensors out; combine: slot rows, index and weights in, tokens out
    return {"bytes": T * H * e + 2 * n * H * e + scales + ids + 3 * 4 * n + 4 * n + T * H * 2, "flops": 2 * n * H}


def _work_moe_quant(c):
    T, H, n = c["tokens"], c["hidden"], c["tokens"] * c["topk"]
    slots = n * (H + H // 128 * 4)
    return {"bytes": T * H * 2 + 2 * slots + n * 8 + 3 * 4 * n + 4 * n + 4 * n + T * H * 2, "flops": 2 * n * H + 3 * T * H}


def _work_moe_layer(c):
    M, H, I, E = c["world"] * c["m_per_rank"], c["hidden"], c["inter"], c["experts"]
    n = M * c["topk"]
    used = min(E, n)
    b = 2 * (M * H + 2 * used * H * I + 2 * n * I + c["world"] * c["m_per_rank"] * H)
    return {"bytes": b, "flops": 4 * n * H * I + 2 * n * H}


def _mean_keys(c):
    return c["longest"] if c["even"] else c["longest"] * (1 - 1 / 64) / math.log(64)


def _work_decode(c):
    e, keys, dv = BYTES[c["dtype"]], c["batch"] * _mean_keys(c), c.get("dim_v", c["dim"])
    cache = c["dim"] if dv < c["dim"] else c["dim"] + dv
    b = keys * c["kv_heads"] * cache * e + keys / c["page"] * 4 + c["batch"] * c["q_heads"] * (c["dim"] + dv) * e
    if c["op"] == "sp_decode":
        b += c["world"] * c["batch"] * c["q_heads"] * (dv * e + 4)
    return {"bytes": b, "flops": 2 * keys * c["q_heads"] * (c["dim"] + dv)}


def work(case):
    return {"ag_gemm": _work_gemm, "gemm_rs": _work_gemm, "moe_a2a": _work_moe_a2a, "moe_quant": _work_moe_quant,
            "moe_layer": _work_moe_layer, "decode": _work_decode, "sp_decode": _work_decode}[case["op"]](case)


def tolerance(case):
    # 16-bit results: the rounding of the output, and of the 16-bit values between two steps; indices, moved bytes and
    # counts are whole numbers and have to be the same
    return {"rel": 2e-3, "max": 0.02} if case.get("dtype") == "f16" else {"rel": 1e-2, "max": 0.05}
