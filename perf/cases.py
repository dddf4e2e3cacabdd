"""Timed cases of the KV-cache path on one GPU: one attention or GDN layer's
share of a serving step, through the package's public entry points.

* ``decode``: a decode step of one attention layer: the new tokens' K/V
  appended to the paged pool, then paged decode attention over it;
* ``prefill``: varlen causal attention over contiguous prompts;
* ``chunk``: chunked prefill through the pool: the chunks' K/V appended, then
  attention of the chunks' queries to the cached prefix and themselves;
* ``gather``: a decode step that hands contiguous padded K/V to the caller;
* ``fp8``: a prefill chunk quantised into an fp8 pool, then the packed
  dequantised window of every sequence;
* ``gdn``: a GDN layer's decode step: states gathered with the decode conv
  fused, the updated states scattered back;
* ``admit``: prefix-cache admission: page hashes of the batch's prompts, one
  block-manager step (the previous batch released, this one admitted), and the
  copy-on-write of partial pages.

Sequence lengths and page placement are the workload's shape and come from the
case itself; the seed makes the values.
"""
import numpy as np
import torch

from muserve_amd import _lib
from muserve_amd.block_manager import BlockManager, admit_op, release_op
from muserve_amd.kernels.attention import (attn_decode, attn_decode_fp8, attn_prefill,
                                           attn_prefill_paged)
from muserve_amd.kv_cache import PagedKVCache
from muserve_amd.prefix_hash import page_hashes_range, page_offsets
from muserve_amd.state_pool import StatePool

D = 256      # head_dim
G = 4        # query heads per KV head
PAGE = 16    # tokens per page
STATE = 8 * 128 * 128   # fp32 values of one recurrent state slot
CHANNELS = 2048         # conv channels of one slot, 4 bf16 each
MAX_LEN = 32768         # longest decode context
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # one interactive user: latency and launches
        {"name": "decode one user", "kind": "decode", "dtype": "bf16", "batch": 1, "heads": 1,
         "median": 777, "sigma": 0.0, "shape": 1},
        # a small batch on a rank with both KV heads, in the default pool dtype
        {"name": "decode fp16 two heads", "kind": "decode", "dtype": "fp16", "batch": 17,
         "heads": 2, "median": 1024, "sigma": 1.0, "shape": 2},
        # the benchmark's decode batch: 256 sequences, lognormal contexts of median 4096
        {"name": "decode full batch", "kind": "decode", "dtype": "bf16", "batch": 256, "heads": 1,
         "median": 4096, "sigma": 1.0, "shape": 102},
        # the serving loop's decode batch over an fp8 pool
        {"name": "decode fp8", "kind": "decode", "dtype": "fp8", "batch": 192, "heads": 1,
         "median": 1500, "sigma": 1.0, "shape": 4},
        # a short chat turn: the smallest prefill
        {"name": "prefill short prompt", "kind": "prefill", "seqs": 1, "heads": 1, "median": 77,
         "sigma": 0.0, "shape": 5},
        # a mixed batch of prompts as users send them
        {"name": "prefill ragged prompts", "kind": "prefill", "seqs": 6, "heads": 1,
         "median": 1024, "sigma": 1.0, "shape": 6},
        # the benchmark's prompts: 8 x 4096
        {"name": "prefill long prompts", "kind": "prefill", "seqs": 8, "heads": 1, "median": 4096,
         "sigma": 0.0, "shape": 7},
        # a serving step's prefill share: two chunks of a 4096-token budget on cached prefixes
        {"name": "prefill chunks", "kind": "chunk", "seqs": 2, "heads": 1, "chunk": 1433,
         "prefix": 6000, "shape": 8},
        # contiguous K/V for a caller with its own dense attention
        {"name": "padded gather", "kind": "gather", "batch": 64, "heads": 1, "median": 2048,
         "sigma": 1.0, "shape": 9},
        # the fp8 benchmark's shape, fewer requests: 2048-token chunks, 8192-token windows
        {"name": "fp8 chunk and window", "kind": "fp8", "seqs": 8, "heads": 1, "chunk": 2048,
         "window": 8192, "shape": 10},
        # a GDN layer at the serving loop's batch
        {"name": "gdn decode step", "kind": "gdn", "batch": 256, "shape": 11},
        # an admission batch of prompts that share templates
        {"name": "prefix admission", "kind": "admit", "batch": 64, "templates": 16,
         "template": 2048, "suffix": 512, "shape": 12},
    ]


def _log(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "chunk",
                       "gather", "fp8", "gdn", "admit"])
    shape = rng.randrange(1 << 20)
    if kind == "decode":
        batch, median = _log(rng, 1, 256), _log(rng, 64, 8192)
        heads = rng.choice([1, 1, 2])
        median = min(median, (256 * 4096) // (batch * heads))
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "fp16", "fp8"]), "batch": batch,
                "heads": heads, "median": median, "sigma": rng.choice([0.0, 0.5, 1.0]),
                "shape": shape}
    if kind == "prefill":
        seqs, median = _log(rng, 1, 8), _log(rng, 16, 4096)
        return {"kind": kind, "seqs": seqs, "heads": rng.choice([1, 1, 2]) if seqs < 4 else 1,
                "median": median, "sigma": rng.choice([0.0, 0.5, 1.0]), "shape": shape}
    if kind == "chunk":
        seqs = rng.choice([1, 2, 3, 4])
        return {"kind": kind, "seqs": seqs, "heads": 1, "chunk": _log(rng, 16, 4096 // seqs),
                "prefix": _log(rng, 16, 16384), "shape": shape}
    if kind == "gather":
        batch = _log(rng, 4, 64)
        return {"kind": kind, "batch": batch, "heads": rng.choice([1, 1, 2]) if batch <= 32 else 1,
                "median": _log(rng, 128, 2048), "sigma": rng.choice([0.0, 0.5, 1.0]),
                "shape": shape}
    if kind == "fp8":
        return {"kind": kind, "seqs": _log(rng, 1, 8), "heads": 1, "chunk": _log(rng, 64, 2048),
                "window": _log(rng, 256, 8192), "shape": shape}
    if kind == "gdn":
        return {"kind": kind, "batch": _log(rng, 1, 256), "shape": shape}
    return {"kind": kind, "batch": _log(rng, 2, 64), "templates": _log(rng, 2, 16),
            "template": _log(rng, 64, 2048), "suffix": _log(rng, 32, 512), "shape": shape}


# --- the workload's shape, from the case alone -------------------------------------------


def _lengths(case, count, longest):
    g = np.random.default_rng(case["shape"])
    x = case["median"] * np.exp(case["sigma"] * g.standard_normal(count))
    return np.clip(np.rint(x), 1, longest).astype(np.int64)


def _prompt_lengths(case):
    # prompts of one call: at most 4096 tokens each
    return _lengths(case, case["seqs"], 4096)


def _chunks(case):
    """(queries, keys) of each sequence: a chunk and the cached prefix under it."""
    g = np.random.default_rng(case["shape"])
    n = case["seqs"]
    q = np.maximum(1, np.rint(case["chunk"] * g.uniform(0.7, 1.0, n))).astype(np.int64)
    p = np.rint(case["prefix"] * g.uniform(0.3, 1.0, n)).astype(np.int64)
    return q, p + q


def _pages(n):
    return -(-n // PAGE)


def _tables(case, lens, dev):
    """Block tables over shuffled pages: (tables [B, W] int32 on the device, host, pool pages)."""
    counts = _pages(lens)
    pool = int(counts.sum()) + 16
    ids = np.random.default_rng(case["shape"] + 1).permutation(pool).astype(np.int32)
    host = np.zeros((len(lens), int(counts.max())), dtype=np.int32)
    at = 0
    for b, c in enumerate(counts):
        host[b, :c] = ids[at:at + c]
        at += c
    return torch.from_numpy(host).to(dev), host, pool


def _slots(host, first, lens):
    """Slots of positions first[b] .. lens[b] - 1 of every sequence, concatenated."""
    out = []
    for b in range(len(lens)):
        pos = np.arange(first[b], lens[b], dtype=np.int64)
        out.append(host[b][pos // PAGE].astype(np.int64) * PAGE + pos % PAGE)
    return np.concatenate(out)


def _i32(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.int32)).to(dev)


def _cu(n):
    return np.concatenate([[0], np.cumsum(n)])


def _gen(seed, dev):
    return torch.Generator(device=dev).manual_seed(int(seed) & 0x7FFFFFFF)


def _randn(gen, shape, dtype):
    return torch.randn(shape, generator=gen, device=gen.device).to(dtype)


def _quantized(x):
    """(e4m3fn codes, fp32 scales): one absmax / 448 scale per row."""
    xf = x.float()
    scale = xf.abs().amax(dim=-1).clamp(min=1e-12) / 448.0
    return (xf / scale.unsqueeze(-1)).clamp(-448.0, 448.0).to(torch.float8_e4m3fn), scale


# --- inputs (plain tensors, shared by prepare and exact) ----------------------------------


def _decode_inputs(case, seed, dev):
    g = _gen(seed, dev)
    B, H = case["batch"], case["heads"]
    longest = min(MAX_LEN, max(64, (1 << 20) * 3 // 2 // (B * H))) if B < 256 else MAX_LEN
    lens = _lengths(case, B, longest)  # the new token included
    tables, host, pool = _tables(case, lens, dev)
    dt = torch.bfloat16 if case["dtype"] == "fp8" else DTYPES[case["dtype"]]
    kv = _randn(g, (2, pool, PAGE, H, D), dt)
    x = {"lens": lens, "tables": tables, "host": host, "pool": pool, "kv": kv,
         "q": _randn(g, (B, 1, G * H, D), dt),
         "k": _randn(g, (B, H, D), dt), "v": _randn(g, (B, H, D), dt),
         "slots": torch.from_numpy(_slots(host, lens - 1, lens)).to(dev)}
    return x


def _prefill_inputs(case, seed, dev):
    g = _gen(seed, dev)
    H, lens = case["heads"], _prompt_lengths(case)
    T = int(lens.sum())
    return {"lens": lens, "q": _randn(g, (T, G * H, D), torch.bfloat16),
            "k": _randn(g, (T, H, D), torch.bfloat16), "v": _randn(g, (T, H, D), torch.bfloat16)}


def _chunk_inputs(case, seed, dev):
    g = _gen(seed, dev)
    H = case["heads"]
    nq, nk = _chunks(case)
    tables, host, pool = _tables(case, nk, dev)
    T = int(nq.sum())
    return {"nq": nq, "nk": nk, "tables": tables, "host": host, "pool": pool,
            "kv": _randn(g, (2, pool, PAGE, H, D), torch.bfloat16),
            "q": _randn(g, (T, G * H, D), torch.bfloat16),
            "k": _randn(g, (T, H, D), torch.bfloat16), "v": _randn(g, (T, H, D), torch.bfloat16),
            "slots": torch.from_numpy(_slots(host, nk - nq, nk)).to(dev)}


def _gather_inputs(case, seed, dev):
    g = _gen(seed, dev)
    B, H = case["batch"], case["heads"]
    lens = _lengths(case, B, 8192)
    tables, host, pool = _tables(case, lens, dev)
    return {"lens": lens, "tables": tables, "host": host, "pool": pool,
            "kv": _randn(g, (2, pool, PAGE, H, D), torch.bfloat16),
            "k": _randn(g, (B, H, D), torch.bfloat16), "v": _randn(g, (B, H, D), torch.bfloat16),
            "slots": torch.from_numpy(_slots(host, lens - 1, lens)).to(dev)}


def _fp8_lengths(case):
    """Context lengths after the chunk; every sequence gives its last window."""
    n = np.random.default_rng(case["shape"]).uniform(0.5, 1.5, case["seqs"])
    return case["chunk"] + np.rint(case["window"] * n).astype(np.int64)


def _fp8_inputs(case, seed, dev):
    g = _gen(seed, dev)
    H, lens = case["heads"], _fp8_lengths(case)
    tables, host, pool = _tables(case, lens, dev)
    T = case["chunk"] * case["seqs"]
    starts = np.maximum(0, lens - case["window"])
    return {"lens": lens, "starts": starts, "tables": tables, "host": host, "pool": pool,
            "kv": _randn(g, (2, pool, PAGE, H, D), torch.bfloat16),
            "k": _randn(g, (T, H, D), torch.bfloat16), "v": _randn(g, (T, H, D), torch.bfloat16),
            "slots": torch.from_numpy(_slots(host, lens - case["chunk"], lens)).to(dev)}


def _gdn_inputs(case, seed, dev):
    g = _gen(seed, dev)
    B = case["batch"]
    S = 2 * B + 3
    slots = np.random.default_rng(case["shape"]).permutation(S)[:B]
    return {"S": S, "slots": _i32(slots, dev),
            "pool": _randn(g, (1, S, 8, 128, 128), torch.float32),
            "conv": _randn(g, (1, S, CHANNELS, 4), torch.bfloat16),
            "x": _randn(g, (B, CHANNELS), torch.bfloat16),
            "weight": _randn(g, (CHANNELS, 1, 4), torch.bfloat16),
            "new": _randn(g, (B, 8, 128, 128), torch.float32)}


# --- states -------------------------------------------------------------------------------


def _pool(x, case, dtype, dev):
    cache = PagedKVCache(x["pool"], num_layers=1, kv_heads=case["heads"], head_dim=D, dtype=dtype,
                         device=dev, verbose=False)
    if dtype == torch.float8_e4m3fn:
        codes, scales = _quantized(x["kv"])
        cache.cache[0].copy_(codes)
        cache.scales[0].copy_(scales)
    else:
        cache.cache[0].copy_(x["kv"])
    return cache


def _prepare_decode(case, seed, dev):
    x = _decode_inputs(case, seed, dev)
    x["cache"] = _pool(x, case, DTYPES.get(case["dtype"], torch.float8_e4m3fn), dev)
    x["seq_lens"] = _i32(x["lens"], dev)
    del x["kv"]
    return x


def _prepare_prefill(case, seed, dev):
    x = _prefill_inputs(case, seed, dev)
    x["cu"] = _i32(_cu(x["lens"]), dev)
    x["longest"] = int(x["lens"].max())
    return x


def _prepare_chunk(case, seed, dev):
    x = _chunk_inputs(case, seed, dev)
    x["cache"] = _pool(x, case, torch.bfloat16, dev)
    x["cu"], x["seq_lens"] = _i32(_cu(x["nq"]), dev), _i32(x["nk"], dev)
    x["longest_q"], x["longest_k"] = int(x["nq"].max()), int(x["nk"].max())
    del x["kv"]
    return x


def _prepare_gather(case, seed, dev):
    x = _gather_inputs(case, seed, dev)
    x["cache"] = _pool(x, case, torch.bfloat16, dev)
    x["seq_lens"] = _i32(x["lens"], dev)
    out_len = x["tables"].shape[1] * PAGE
    shape = (case["batch"], out_len, case["heads"], D)
    x["out"] = tuple(torch.empty(shape, dtype=torch.bfloat16, device=dev) for _ in range(2))
    del x["kv"]
    return x


def _prepare_fp8(case, seed, dev):
    x = _fp8_inputs(case, seed, dev)
    x["cache"] = _pool(x, case, torch.float8_e4m3fn, dev)
    x["seq_lens"], x["start"] = _i32(x["lens"], dev), _i32(x["starts"], dev)
    n = x["lens"] - x["starts"]
    x["cu"] = torch.from_numpy(_cu(n)).to(dev)
    x["longest"] = int(n.max())
    shape = (int(n.sum()), case["heads"], D)
    x["out"] = tuple(torch.empty(shape, dtype=torch.bfloat16, device=dev) for _ in range(2))
    del x["kv"]
    return x


def _prepare_gdn(case, seed, dev):
    x = _gdn_inputs(case, seed, dev)
    pool = StatePool(num_layers=1, num_slots=x["S"], device=dev)
    pool.state.copy_(x.pop("pool"))
    pool.conv.copy_(x.pop("conv"))
    x["pool"] = pool
    return x


_GROUPS = 4  # batches of requests admitted in turn


def _admit_shape(case):
    """(template of every request, its suffix length) for the batches admitted in turn."""
    g = np.random.default_rng(case["shape"])
    n = _GROUPS * case["batch"]
    rank = np.minimum(g.zipf(1.4, n) - 1, case["templates"] - 1)
    return rank, np.maximum(1, np.rint(case["suffix"] * g.uniform(0.125, 1.0, n))).astype(np.int64)


def _prepare_admit(case, seed, dev):
    g = np.random.default_rng(seed)
    B, n = case["batch"], _GROUPS * case["batch"]
    rank, suffix = _admit_shape(case)
    heads = g.integers(0, 1 << 17, (case["templates"], case["template"]))
    prompts = [np.concatenate([heads[r], g.integers(0, 1 << 17, s)])
               for r, s in zip(rank, suffix)]
    lens = np.array([len(p) for p in prompts], dtype=np.int64)
    cu_t = _cu(lens).astype(np.int64)
    cu_p = page_offsets(cu_t)
    pages = _pages(lens)
    # the pool holds the templates and about two batches' own pages: a batch
    # finds its templates cached and evicts an older batch's suffixes
    own = pages - case["template"] // PAGE + 2
    P = int(case["templates"] * _pages(case["template"]) + own.sum() * 5 // 8 + 64)
    x = {"tokens": torch.from_numpy(np.concatenate(prompts)).to(dev),
         "tok_off": torch.from_numpy(cu_t).to(dev), "page_off": torch.from_numpy(cu_p).to(dev),
         "ntok": _i32(lens, dev),
         "hashes": torch.zeros(int(cu_p[-1]), dtype=torch.int64, device=dev),
         "errors": _lib.DeviceErrors(torch.device(dev)), "turn": 0, "batch": B,
         "bm": BlockManager(P, n, int(pages.max()), dev),
         "cache": PagedKVCache(P, num_layers=2, kv_heads=1, head_dim=D, dtype=torch.bfloat16,
                               device=dev, verbose=False)}
    x["ops"] = []
    for t in range(_GROUPS):
        gone = [release_op(((t - 1) % _GROUPS) * B + i) for i in range(B)]
        x["ops"].append(torch.tensor(gone + [admit_op(t * B + i) for i in range(B)],
                                     dtype=torch.int32, device=dev))
    # a manager in service: the last batch is admitted when the first turn comes
    page_hashes_range(x["tokens"], x["tok_off"], x["page_off"], 0, n, x["hashes"], x["errors"])
    for t in range(_GROUPS):
        x["bm"].step(x["ops"][t] if t else x["ops"][0][B:].contiguous(), x["hashes"],
                     x["page_off"], x["ntok"])
    return x


def prepare(case, seed):
    dev = torch.device("cuda:0")
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "chunk": _prepare_chunk,
            "gather": _prepare_gather, "fp8": _prepare_fp8, "gdn": _prepare_gdn,
            "admit": _prepare_admit}[case["kind"]](case, seed, dev) | {"case": case}


# --- one pass -----------------------------------------------------------------------------


def _run_decode(s):
    cache = s["cache"]
    cache.append(s["slots"], s["k"], s["v"], layer=0)
    k, v = cache.get_kv_by_layer(0)
    if cache.scales is not None:
        out = attn_decode_fp8(s["q"], k, v, cache.scales[0, 0], cache.scales[0, 1], s["seq_lens"],
                              s["tables"])
        return {"out": out, "codes": cache.cache.view(torch.uint8), "scales": cache.scales}
    out = attn_decode(s["q"], k, v, s["seq_lens"], s["tables"])
    return {"out": out, "kv": cache.cache}


def _run_prefill(s):
    return {"out": attn_prefill(s["q"], s["k"], s["v"], s["cu"], s["cu"], s["longest"],
                                s["longest"])}


def _run_chunk(s):
    cache = s["cache"]
    cache.append(s["slots"], s["k"], s["v"], layer=0)
    k, v = cache.get_kv_by_layer(0)
    out = attn_prefill_paged(s["q"], k, v, s["cu"], s["seq_lens"], s["tables"], s["longest_q"],
                             max_seqlen_k=s["longest_k"])
    return {"out": out, "kv": cache.cache}


def _run_gather(s):
    s["cache"].append(s["slots"], s["k"], s["v"], layer=0)
    k, v = s["cache"].gather(0, s["tables"], s["seq_lens"], out=s["out"])
    return {"k": k, "v": v}


def _run_fp8(s):
    cache = s["cache"]
    cache.append(s["slots"], s["k"], s["v"], layer=0)
    k, v = cache.gather(0, s["tables"], s["seq_lens"], out_len=s["longest"], starts=s["start"],
                        out=s["out"], cu_out=s["cu"])
    return {"k": k, "v": v, "codes": cache.cache.view(torch.uint8), "scales": cache.scales}


def _run_gdn(s):
    pool = s["pool"]
    states, conv = pool.decode_gather(0, s["slots"], s["x"], s["weight"])
    pool.scatter(0, s["slots"], s["new"])
    return {"states": states, "conv": conv, "pool": pool.state, "conv_pool": pool.conv}


def _run_admit(s):
    B, t, bm = s["batch"], s["turn"], s["bm"]
    s["turn"] = (t + 1) % _GROUPS
    page_hashes_range(s["tokens"], s["tok_off"], s["page_off"], t * B, B, s["hashes"], s["errors"])
    bm.step(s["ops"][t], s["hashes"], s["page_off"], s["ntok"])
    bm.copy_on_write(s["cache"], t * B, (t + 1) * B)
    return {"hashes": s["hashes"], "tables": bm.tables, "hits": bm.hits, "status": bm.status,
            "child": bm.child_last}


def run(state):
    return {"decode": _run_decode, "prefill": _run_prefill, "chunk": _run_chunk,
            "gather": _run_gather, "fp8": _run_fp8, "gdn": _run_gdn,
            "admit": _run_admit}[state["case"]["kind"]](state)


# --- what a pass cannot do without --------------------------------------------------------


def work(case):
    kind = case["kind"]
    row = 2 * D
    if kind == "decode":
        B, H = case["batch"], case["heads"]
        longest = min(MAX_LEN, max(64, (1 << 20) * 3 // 2 // (B * H))) if B < 256 else MAX_LEN
        lens = _lengths(case, B, longest)
        n = int(lens.sum())
        cached = (D + 4) if case["dtype"] == "fp8" else row
        read = 2 * n * H * cached + 4 * int(_pages(lens).sum()) + B * (4 + 8)
        new = B * H * 2 * (row + cached)
        return {"bytes": read + new + 2 * B * H * G * row, "flops": 4 * n * H * G * D}
    if kind == "prefill":
        lens, H = _prompt_lengths(case), case["heads"]
        pairs = int((lens * (lens + 1) // 2).sum())
        return {"bytes": int(lens.sum()) * H * row * (2 * G + 2), "flops": 4 * pairs * H * G * D}
    if kind == "chunk":
        (nq, nk), H = _chunks(case), case["heads"]
        pairs = int((nq * (nk - nq) + nq * (nq + 1) // 2).sum())
        T = int(nq.sum())
        return {"bytes": H * row * (2 * int(nk.sum()) + 4 * T + 2 * G * T),
                "flops": 4 * pairs * H * G * D}
    if kind == "gather":
        B, H = case["batch"], case["heads"]
        lens = _lengths(case, B, 8192)
        out = B * int(_pages(lens).max()) * PAGE
        return {"bytes": 2 * H * row * (int(lens.sum()) + out + 2 * B) +
                4 * int(_pages(lens).sum()), "flops": 0}
    if kind == "fp8":
        lens, H = _fp8_lengths(case), case["heads"]
        T = case["chunk"] * case["seqs"]
        n = int(np.minimum(lens, case["window"]).sum())
        return {"bytes": 2 * H * (T * (row + D + 4) + n * (D + 4 + row)) + 8 * T, "flops": 0}
    if kind == "gdn":
        B = case["batch"]
        return {"bytes": B * (4 * 4 * STATE + 2 * 8 * CHANNELS + 2 * 2 * CHANNELS),
                "flops": 2 * 4 * B * CHANNELS}
    B = case["batch"]
    rank, suffix = _admit_shape(case)
    pages = _pages(case["template"] + suffix) / _GROUPS
    # per page: 16 ids read, its hash written and read, its table entry and
    # page record for the admission and for the release of an earlier batch;
    # a copy-on-write page of two layers per request
    return {"bytes": float(pages.sum()) * (8 * PAGE + 16 + 2 * (4 + 32)) +
            B * 2 * 2 * 2 * PAGE * row, "flops": 0}


def tolerance(case):
    # byte moves, integer work, codes: exact. Attention outputs are rounded
    # to 16 bits (2^-9 of the value, rms about 1.7e-3 with bf16 probabilities in
    # the prefill product); four times the error measured against float64.
    if case["kind"] in ("decode", "prefill", "chunk"):
        return {"rel": 1e-3 if case.get("dtype") == "fp16" else 8e-3}
    if case["kind"] == "gdn":
        return {"rel": 8e-3}
    return "exact"


# --- the same in 64 bits, in plain torch --------------------------------------------------


def _attend(q, k, v, first):
    """q [n, H*G, D], k/v [m, H, D] float64; query t sees keys 0 .. first + t (first None: all)."""
    out = torch.empty_like(q)
    n, m = q.shape[0], k.shape[0]
    for h in range(q.shape[1]):
        kh, vh = k[:, h // G].contiguous(), v[:, h // G].contiguous()
        for a in range(0, n, 4096):
            s = (q[a:a + 4096, h] @ kh.t()) * D ** -0.5
            if first is not None:
                at = torch.arange(a, a + s.shape[0], device=q.device) + first
                s.masked_fill_(torch.arange(m, device=q.device)[None, :] > at[:, None],
                               float("-inf"))
            out[a:a + 4096, h] = torch.softmax(s, dim=-1) @ vh
    return out


def _rows(plane, host, b, n):
    """The first n cached rows of sequence b of one plane [P, 16, H, ...]."""
    ids = torch.from_numpy(host[b][:_pages(n)].astype(np.int64)).to(plane.device)
    return plane[ids].reshape(-1, *plane.shape[2:])[:n]


def exact(case, seed):
    dev = torch.device("cuda:0")
    kind = case["kind"]
    if kind == "decode":
        x = _decode_inputs(case, seed, dev)
        kv = x["kv"]
        flat = kv.view(2, -1, case["heads"], D)
        flat[0, x["slots"]], flat[1, x["slots"]] = x["k"], x["v"]
        if case["dtype"] == "fp8":
            codes, scales = _quantized(kv)
        out = torch.empty(x["q"].shape, dtype=torch.float64, device=dev)
        for b, n in enumerate(int(y) for y in x["lens"]):
            if case["dtype"] == "fp8":
                k, v = (_rows(codes[i].view(torch.uint8), x["host"], b, n)
                        .view(torch.float8_e4m3fn).double() *
                        _rows(scales[i], x["host"], b, n).double().unsqueeze(-1)
                        for i in range(2))
            else:
                k, v = (_rows(kv[i], x["host"], b, n).double() for i in range(2))
            out[b] = _attend(x["q"][b].double(), k, v, None)
        if case["dtype"] == "fp8":
            return {"out": out, "codes": None, "scales": scales.double().unsqueeze(0)}
        return {"out": out, "kv": kv.unsqueeze(0)}
    if kind == "prefill":
        x = _prefill_inputs(case, seed, dev)
        cu, out = _cu(x["lens"]), []
        for a, b in zip(cu[:-1], cu[1:]):
            out.append(_attend(*(x[t][a:b].double() for t in "qkv"), 0))
        return {"out": torch.cat(out)}
    if kind == "chunk":
        x = _chunk_inputs(case, seed, dev)
        kv = x["kv"]
        flat = kv.view(2, -1, case["heads"], D)
        flat[0, x["slots"]], flat[1, x["slots"]] = x["k"], x["v"]
        cu, out = _cu(x["nq"]), []
        for b, (n, m) in enumerate(zip(x["nq"], x["nk"])):
            k, v = (_rows(kv[i], x["host"], b, int(m)).double() for i in range(2))
            out.append(_attend(x["q"][cu[b]:cu[b + 1]].double(), k, v, int(m - n)))
        return {"out": torch.cat(out), "kv": kv.unsqueeze(0)}
    if kind == "gdn":
        x = _gdn_inputs(case, seed, dev)
        slots = x["slots"].long()
        conv = torch.cat([x["conv"][0, slots][..., 1:], x["x"].unsqueeze(-1)], dim=-1)
        y = (conv.double() * x["weight"][:, 0].double()).sum(-1)
        states = x["pool"][0, slots]
        x["pool"][0, slots] = x["new"]
        x["conv"][0, slots] = conv
        return {"states": states, "conv": y * torch.sigmoid(y), "pool": x["pool"],
                "conv_pool": x["conv"]}
    return None
