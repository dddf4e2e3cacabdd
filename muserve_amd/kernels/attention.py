"""Attention over the KV pool (muserve/kernels/attention.py): paged decode,
and varlen prefill over contiguous K/V or over the pool.

``attn_decode`` keeps the reference wrapper's signature and meaning
(muserve/kernels/attention.py:29-42): one query token per sequence attends to
its ``cache_seqlens[b]`` cached tokens, found through ``page_table``, with
query head h using KV head h // (Hq / Hkv) — the math of
muserve/model/qwen35_layer_v2.py:493-502, read straight from the pool by a
gfx950 kernel instead of a padded gather plus dense attention. Scores,
softmax and accumulation run in fp32; the output is bf16.

The call is asynchronous on the current stream. Data faults (a page id
outside the pool, a length beyond the table) set bits in a per-device error
word that ``check_errors(device)`` raises.
"""
from __future__ import annotations

import functools

import torch

from muserve_amd import _lib

HEAD_DIM = 256

_DECODE_FNS = {torch.bfloat16: "mkv_decode_attention_bf16",
               torch.float16: "mkv_decode_attention_f16"}

_errors: dict[torch.device, _lib.DeviceErrors] = {}


def _errword(dev: torch.device) -> _lib.DeviceErrors:
    if dev not in _errors:
        _errors[dev] = _lib.DeviceErrors(dev)
    return _errors[dev]


def check_errors(device: torch.device | str = "cuda") -> None:
    """Raises MkvDeviceError for faults flagged by earlier calls (synchronises)."""
    dev = torch.device(device)
    if dev in _errors:
        _errors[dev].check("attn_decode")


def _scratch(nbytes: int, dev: torch.device) -> torch.Tensor:
    """A call's workspace, from torch's allocator at each call, which orders
    its reuse by stream (and keeps it with the graph under capture). One buffer
    kept per device would be overwritten by a call on another stream while
    this one's kernels read it, and freed under them when a larger one is
    needed."""
    return torch.empty(nbytes, dtype=torch.uint8, device=dev)


def workspace_bytes(batch: int, num_kv_heads: int, num_q_heads: int, max_seqlen: int) -> int:
    n = _lib.load().mkv_decode_attention_workspace_bytes(batch, num_kv_heads, num_q_heads,
                                                         max_seqlen)
    if n < 0:
        raise ValueError("bad attention shape")
    return n


@functools.lru_cache(maxsize=1024)
def _decode_bytes(batch: int, num_kv_heads: int, num_q_heads: int, dev: torch.device) -> int:
    return workspace_bytes(batch, num_kv_heads, num_q_heads, 0)


def _decode_scratch(B: int, Hkv: int, Hq: int, max_seqlen: int, dev: torch.device) -> torch.Tensor:
    """The size depends on the shape and the device alone (asking the library
    again costs a decode call 1 us, as much as the allocation)."""
    if max_seqlen < 0:
        raise ValueError("bad attention shape")
    return _scratch(_decode_bytes(B, Hkv, Hq, dev), dev)


def attn_prefill(
    q: torch.Tensor,            # [total_tokens, NUM_Q_HEADS, HEAD_DIM] bf16
    k: torch.Tensor,            # [total_tokens, NUM_KV_HEADS, HEAD_DIM] bf16
    v: torch.Tensor,            # [total_tokens, NUM_KV_HEADS, HEAD_DIM] bf16
    cu_seqlens_q: torch.Tensor, # [num_seqs + 1] int32
    cu_seqlens_k: torch.Tensor, # [num_seqs + 1] int32
    max_seqlen_q: int,
    max_seqlen_k: int,
    softmax_scale: float | None = None,
    causal: bool = True,
    *,
    out: torch.Tensor | None = None,
) -> torch.Tensor:              # [total_tokens, NUM_Q_HEADS, HEAD_DIM] bf16
    """Varlen prefill attention (muserve/kernels/attention.py:6-25, the
    reference's flash_attn_varlen_func): sequence b's queries are rows
    cu_seqlens_q[b]..cu_seqlens_q[b+1] of q, its keys the same rows range of
    cu_seqlens_k in k/v; with causal masking aligned to the bottom-right
    corner (query t of nq sees keys 0 .. nk - nq + t). 4 query heads per KV
    head, head_dim 256; fp32 softmax and accumulation, probabilities rounded
    to bf16 for the P V product, one bf16 rounding of the output."""
    return _prefill(q, k, v, None, cu_seqlens_q, cu_seqlens_k, None, max_seqlen_q, softmax_scale,
                    causal, out, max_seqlen_k)


def attn_prefill_paged(
    q: torch.Tensor,              # [total_tokens, NUM_Q_HEADS, HEAD_DIM] bf16
    k_cache: torch.Tensor,        # [num_pages, PAGE_SIZE, NUM_KV_HEADS, HEAD_DIM] bf16
    v_cache: torch.Tensor,
    cu_seqlens_q: torch.Tensor,   # [num_seqs + 1] int32/int64: the step's query rows
    cache_seqlens: torch.Tensor,  # [num_seqs] int32: keys per sequence, the chunk included
    page_table: torch.Tensor,     # [num_seqs, max_pages] int32
    max_seqlen_q: int,
    softmax_scale: float | None = None,
    causal: bool = True,
    *,
    max_seqlen_k: int | None = None,
    out: torch.Tensor | None = None,
) -> torch.Tensor:
    """attn_prefill over the paged pool, for chunked prefill: a chunk's
    queries (its K/V appended to the pool first) attend to the sequence's
    cached prefix and to themselves, read through the block table — the
    prefill counterpart of attn_decode. With a scheduler plan, the prefill
    entries are plan.cu_seqlens / plan.seq_lens / plan.block_tables past the
    decode entries. ``max_seqlen_k`` (default: what the table holds) bounds
    cache_seqlens; a tight bound lets short steps split the keys better."""
    if page_table is None:
        raise ValueError("attn_prefill_paged reads the paged pool: page_table is required")
    return _prefill(q, k_cache, v_cache, page_table, cu_seqlens_q, None, cache_seqlens,
                    max_seqlen_q, softmax_scale, causal, out, max_seqlen_k)


PREFILL_Q_TILE = 64            # query tokens per workgroup of the prefill kernel
PREFILL_KV_TILE = 64           # keys per step of the prefill kernel (key ranges are multiples)
PREFILL_SPLIT_MIN = 256        # keys per range at least
PREFILL_DENSE_MAX = 8          # key tiles per range up to which a launch is not planned
PREFILL_RANGES = 64            # ranges of PREFILL_SPLIT_MIN keys; where more fit, twice the keys
PREFILL_PLAN_SEQS = 1024       # sequences, and query tiles x KV heads, of a planned launch
PREFILL_PLAN_TILES = 4096
_prefill_cu: dict[torch.device, int] = {}


def _prefill_cus(dev: torch.device) -> int:
    n = _prefill_cu.get(dev)
    if n is None:
        n = torch.cuda.get_device_properties(dev).multi_processor_count
        _prefill_cu[dev] = n
    return n


def prefill_schedule(tokens: int, max_q: int, max_k: int, batch: int, kv_heads: int, causal: bool,
                     cus: int) -> tuple[int, int, bool]:
    """(key ranges per query tile at most, keys a range aims at, planned).

    A CU runs one workgroup at a time, a key tile after the other, so a launch
    takes as long as the most key tiles that any CU gets. A grid sized on the
    host (every query tile that the longest sequence could have, times the
    batch, in ranges of the same number of keys) does while it fits the CUs at
    once with short ranges; a planned launch sorts the tasks that exist on the
    device, which costs a launch of 7-8 us and pays for itself where that
    grid's ranges would be long and its sequences differ (MI355X: six prompts
    of 80 to 4096 tokens 177 -> 143 us; 8 equal prompts of 4096, where the
    grid is balanced as it is, take 254-276 us without a plan).

    The line, PREFILL_DENSE_MAX, on 60 shapes (us without and with a plan): up
    to 8 key tiles per range the grid was faster on all of them (8 chunks of 1
    token on 6-14k cached ones 40, 51; 2 of 1 on 60k 73, 93; 500 tokens beside
    31 x 50 31, 33); at 9 to 16 by the shape (1200 on 7k cached 61, 73; 6
    prompts of 360 to 1240 45, 42; 4 of 265 to 1520 51, 42), but on all where
    up to 8 sequences have one query tile each: a plan has little to sort and
    more ranges to merge (2 x 1 on up to 120k 86, 114; 8 x 64 on up to 32k 69, 85).
    """
    units = -(-max_k // PREFILL_KV_TILE)
    if units <= PREFILL_SPLIT_MIN // PREFILL_KV_TILE:
        return 1, 0, False
    rows = -(-max_q // PREFILL_Q_TILE)
    dense = rows * batch
    tiles = min(dense, tokens // PREFILL_Q_TILE + batch)
    least = PREFILL_SPLIT_MIN // PREFILL_KV_TILE
    # twice that where a row would have more than PREFILL_RANGES ranges: the
    # merge walks them 8 at a time, about 0.3 us a range against 2.4 us a key
    # tile (64 tokens on 60000 cached ones in 235 ranges 108 us, in 118 76 us;
    # 200 on 16000 in 58, 46 or 23 ranges 48, 46 and 51 us)
    if units > PREFILL_RANGES * least:
        least *= 2
    # half of PREFILL_SPLIT_MIN for a few short workgroups (32 query tokens
    # each) with CUs to spare, whose chain of key tiles is most of the launch:
    # one prompt of 500 tokens 22.1 -> 18.2 us, 619 on 95 cached ones 27.2 ->
    # 24.6 us. With more ranges or more workgroups the merge costs it back
    # (2 x 600 tokens 40.7 -> 42.2 us, 40 tokens on 12000 cached ones 39 -> 44
    # us).
    fine = -(-2 * units // least)
    half = PREFILL_Q_TILE // 2
    few = min(-(-max_q // half) * batch, tokens // half + batch) * kv_heads * fine
    if least < units and fine <= 8 and few <= cus // 2:
        least //= 2
    fit = cus // max(1, dense * kv_heads)
    aim = max(least, -(-units // fit)) if fit else units
    dense_max = PREFILL_DENSE_MAX * (2 if batch <= 8 and rows == 1 else 1)
    if aim <= dense_max:
        splits = max(1, -(-units // aim)) if fit else 1
        per = -(-units // splits)
        # without a causal mask every row has all the ranges: they have to save
        # more key tiles (2.4 us each) than the merge of their partial rows
        # costs (8 x 300 tokens 22.2 us in one range, 28.6 in two; 8 x 500 31.3,
        # 33.9; 4 x 700 in one 38.6, in three 33.5)
        if not causal and (units - per) * 2.4 < 4 + splits * tokens * 4 * kv_heads * 2064 / 8e6:
            return 1, 0, False
        return (splits, per * PREFILL_KV_TILE, False) if splits > 1 else (1, 0, False)
    mean = units - (min(rows, units) - 1) / 2 if causal else units
    share = tiles * kv_heads * mean / cus  # key tiles per CU, at most
    if batch > PREFILL_PLAN_SEQS or tiles * kv_heads > PREFILL_PLAN_TILES:
        return 1, 0, False
    if share >= units:  # several rounds of whole tiles: long enough to balance by their order
        return 1, 0, dense > tiles + tiles // 8
    splits = -(-units // max(least, int(share * 3 / 4)))
    return min(splits, 65535 // kv_heads), 0, True


def _prefill(q, k, v, page_table, cu_q, cu_k, lens_k, max_seqlen_q, softmax_scale, causal, out,
             max_seqlen_k=None):
    dev = _lib.require_gpu(q, k, v, page_table, cu_q, cu_k, lens_k)
    if q.dtype != torch.bfloat16 or k.dtype != torch.bfloat16 or v.dtype != torch.bfloat16:
        raise TypeError("attn_prefill takes bf16 q, k and v")
    Tq, Hq, D = q.shape
    Hkv = k.shape[-2]
    if D != HEAD_DIM or k.shape[-1] != D or v.shape != k.shape or Hq != 4 * Hkv:
        raise ValueError(f"unsupported shapes q {tuple(q.shape)}, k {tuple(k.shape)} "
                         "(head_dim 256, 4 query heads per KV head)")
    if page_table is not None and (k.dim() != 4 or k.shape[1] != 16):
        raise ValueError("the paged pool must be [num_pages, 16, kv_heads, 256]")
    if page_table is None and k.dim() != 3:
        raise ValueError("contiguous k/v must be [total_tokens, kv_heads, 256]")
    if not (q.is_contiguous() and k.is_contiguous() and v.is_contiguous()):
        raise ValueError("q, k and v must be contiguous")
    cu_q = cu_q.to(device=dev, dtype=torch.int32).contiguous()
    batch = cu_q.numel() - 1
    if cu_k is not None:
        cu_k = cu_k.to(device=dev, dtype=torch.int32).contiguous()
        if cu_k.numel() != batch + 1:
            raise ValueError("cu_seqlens_k must have as many entries as cu_seqlens_q")
    if lens_k is not None:
        if lens_k.dtype != torch.int32 or page_table.dtype != torch.int32:
            raise TypeError("cache_seqlens and page_table must be int32")
        if lens_k.numel() != batch or page_table.shape[0] < batch or page_table.stride(1) != 1:
            raise ValueError("cache_seqlens / page_table rows do not match cu_seqlens_q")
        lens_k = lens_k.contiguous()
    if out is None:
        out = torch.empty_like(q)
    elif out.shape != q.shape or out.dtype != q.dtype or not out.is_contiguous():
        raise ValueError("out must be a contiguous tensor shaped like q")
    scale = D ** -0.5 if softmax_scale is None else float(softmax_scale)
    units = k.shape[0]
    # bounds that the rows already give: a caller's loose ones would buy a plan
    # and empty workgroups (one prompt of 64 tokens under bounds of 4096: 17.9
    # us, 11.0 under its own)
    max_q = min(int(max_seqlen_q), max(Tq, 1))  # (no rows: refused below)
    max_k = int(max_seqlen_k) if max_seqlen_k is not None else page_table.shape[1] * 16
    if page_table is None:
        max_k = min(max_k, units)
    sched = prefill_schedule(Tq, max_q, max_k, min(batch, PREFILL_PLAN_SEQS), Hkv, causal,
                             _prefill_cus(dev))
    some = batch
    if batch > PREFILL_PLAN_SEQS:
        # more than a plan holds are planned so many at a time (1500 tokens
        # beside 2000 x 16: one launch of 48000 workgroups, nearly all empty,
        # took 252 us)
        if sched[2] and batch <= 65535:  # (the library's limit for one call)
            some = PREFILL_PLAN_SEQS
        else:
            sched = prefill_schedule(Tq, max_q, max_k, batch, Hkv, causal, _prefill_cus(dev))
    splits, split_len, planned = sched
    ws, ws_bytes = None, 0
    if planned:
        ws_bytes = _lib.load().mkv_prefill_attention_plan_bytes(Tq, Hq, Hkv, some, max_q, splits)
    elif splits > 1:
        ws_bytes = _lib.load().mkv_prefill_attention_workspace_bytes(Tq, Hq, splits)
    if ws_bytes > 0:
        ws = _scratch(ws_bytes, dev)
    fn = "mkv_prefill_attention_planned_bf16" if planned else "mkv_prefill_attention_bf16"
    table, stride, width = None, 0, 0
    if page_table is not None:
        table, stride, width = page_table.data_ptr(), page_table.stride(0), page_table.shape[1]
    cu_qp, cu_kp, lens_kp = cu_q.data_ptr(), _lib.ptr(cu_k), _lib.ptr(lens_k)
    first = 0
    while True:
        _lib.call(fn, q.data_ptr(), k.data_ptr(), v.data_ptr(), units, Hkv, Hq, D, table, stride,
                  width, cu_qp, cu_kp, lens_kp, min(some, batch - first), Tq, max_q, scale,
                  1 if causal else 0, splits, *(() if planned else (split_len,)), out.data_ptr(),
                  _lib.ptr(ws), ws_bytes, _errword(dev).ptr(), _lib.stream_of(dev))
        first += some
        if first >= batch:
            return out
        cu_qp += 4 * some  # (int32 offsets, lengths and page ids)
        if table is None:
            cu_kp += 4 * some
        else:
            table += 4 * some * stride
            lens_kp += 4 * some


def attn_decode(
    q: torch.Tensor,                    # [B, 1, NUM_Q_HEADS, HEAD_DIM] bf16 / fp16
    k_cache: torch.Tensor,              # [num_pages, PAGE_SIZE, NUM_KV_HEADS, HEAD_DIM] same
    v_cache: torch.Tensor,              # [num_pages, PAGE_SIZE, NUM_KV_HEADS, HEAD_DIM] same
    cache_seqlens: torch.Tensor,        # [B] int32 — current kv length per seq
    page_table: torch.Tensor | None,    # [B, max_pages] int32 — paged kv index
    softmax_scale: float | None = None,
    *,
    max_seqlen: int | None = None,
    out: torch.Tensor | None = None,
    shared_pages: int = 0,
) -> torch.Tensor:                      # [B, 1, NUM_Q_HEADS, HEAD_DIM] bf16 / fp16
    """bf16 or fp16 caches (fp16 is the reference's default pool dtype,
    muserve/config.py:37), with q and the output in the caches' dtype.
    ``max_seqlen`` bounds ``cache_seqlens`` (default: what the page table
    holds). ``out`` may be given to write in place.

    ``shared_pages``: page ids below it may be read by several sequences of
    the batch (prompt pages shared through prefix reuse, e.g. a
    ``BlockManager``'s page range): they are loaded through the GPU caches so
    that their readers share them. Every other page streams past the caches,
    which is faster for pages one sequence reads (the default: 0, no page
    shared).

    With ``page_table=None`` the caches are contiguous per sequence,
    ``[B, S, NUM_KV_HEADS, HEAD_DIM]``, sequence b's first
    ``cache_seqlens[b]`` rows attended (the reference forwards None to its
    kernel the same way, muserve/kernels/attention.py:33-42): the padded
    layout ``PagedKVCache.gather`` writes."""
    if k_cache.dtype not in _DECODE_FNS or v_cache.dtype != k_cache.dtype:
        raise TypeError("attn_decode takes bf16 or fp16 caches (attn_decode_fp8 reads fp8 ones)")
    if q.dtype != k_cache.dtype:
        raise TypeError(f"q is {q.dtype}, the caches {k_cache.dtype}: they must match")
    return _decode(_DECODE_FNS[k_cache.dtype], q, k_cache, v_cache, None, None, cache_seqlens,
                   page_table, softmax_scale, max_seqlen, out, shared_pages)


def attn_decode_fp8(
    q: torch.Tensor,                    # [B, 1, NUM_Q_HEADS, HEAD_DIM] bf16
    k_cache: torch.Tensor,              # [num_pages, PAGE_SIZE, NUM_KV_HEADS, HEAD_DIM] e4m3fn
    v_cache: torch.Tensor,              # [num_pages, PAGE_SIZE, NUM_KV_HEADS, HEAD_DIM] e4m3fn
    k_scales: torch.Tensor,             # [num_pages, PAGE_SIZE, NUM_KV_HEADS] fp32
    v_scales: torch.Tensor,             # [num_pages, PAGE_SIZE, NUM_KV_HEADS] fp32
    cache_seqlens: torch.Tensor,
    page_table: torch.Tensor | None,
    softmax_scale: float | None = None,
    *,
    max_seqlen: int | None = None,
    out: torch.Tensor | None = None,
    shared_pages: int = 0,
) -> torch.Tensor:                      # [B, 1, NUM_Q_HEADS, HEAD_DIM] bf16
    """``attn_decode`` over an fp8 pool (codes plus one fp32 scale per token and
    KV head, as ``PagedKVCache`` appends them), with the dequantisation fused:
    a cached value is ``code * scale`` taken exactly (in fp32), not rounded to
    bf16 first as ``gather``'s dequantisation does. Same arguments otherwise."""
    if k_cache.dtype != torch.float8_e4m3fn or v_cache.dtype != torch.float8_e4m3fn:
        raise TypeError("attn_decode_fp8 takes float8_e4m3fn caches")
    for name, s in (("k_scales", k_scales), ("v_scales", v_scales)):
        if s.dtype != torch.float32 or s.shape != k_cache.shape[:3] or not s.is_contiguous():
            raise ValueError(f"{name} must be contiguous fp32 {tuple(k_cache.shape[:3])}")
    return _decode("mkv_decode_attention_fp8", q, k_cache, v_cache, k_scales, v_scales,
                   cache_seqlens, page_table, softmax_scale, max_seqlen, out, shared_pages)


def _decode_contig(q, k_cache, v_cache, cache_seqlens, softmax_scale, max_seqlen, out):
    dev = _lib.require_gpu(q, k_cache, v_cache, cache_seqlens)
    B, one, Hq, D = q.shape
    if k_cache.dim() != 4:
        raise ValueError("without a page table the caches are [B, S, kv_heads, 256]")
    Bk, S, Hkv, Dk = k_cache.shape
    if one != 1 or D != HEAD_DIM or Dk != D or Bk != B or v_cache.shape != k_cache.shape:
        raise ValueError(f"unsupported shapes q {tuple(q.shape)}, cache {tuple(k_cache.shape)}")
    if cache_seqlens.dtype != torch.int32 or cache_seqlens.numel() != B:
        raise TypeError("cache_seqlens must be int32 [B]")
    if not (q.is_contiguous() and k_cache.is_contiguous() and v_cache.is_contiguous()
            and cache_seqlens.is_contiguous()):
        raise ValueError("q, caches and cache_seqlens must be contiguous")
    if out is None:
        out = torch.empty_like(q)
    elif out.shape != q.shape or out.dtype != q.dtype or not out.is_contiguous():
        raise ValueError("out must be a contiguous tensor shaped like q")
    if max_seqlen is None:
        max_seqlen = S
    scale = D ** -0.5 if softmax_scale is None else float(softmax_scale)
    ws = _decode_scratch(B, Hkv, Hq, max_seqlen, dev)
    _lib.call("mkv_decode_attention_contig", q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
              1 if k_cache.dtype == torch.float16 else 0, Hkv, Hq, D, S,
              cache_seqlens.data_ptr(), B, int(min(max_seqlen, 1 << 24)), scale, out.data_ptr(),
              ws.data_ptr(), ws.numel(), _errword(dev).ptr(), _lib.stream_of(dev))
    return out


def _decode(fn, q, k_cache, v_cache, k_scales, v_scales, cache_seqlens, page_table,
            softmax_scale, max_seqlen, out, shared_pages=0):
    if page_table is None:
        if k_scales is not None:
            raise ValueError("attn_decode_fp8 reads the paged pool: page_table is required")
        return _decode_contig(q, k_cache, v_cache, cache_seqlens, softmax_scale, max_seqlen, out)
    dev = _lib.require_gpu(q, k_cache, v_cache, k_scales, v_scales, cache_seqlens, page_table)
    B, one, Hq, D = q.shape
    P, page, Hkv, Dk = k_cache.shape
    if one != 1 or page != 16 or D != HEAD_DIM or Dk != D or v_cache.shape != k_cache.shape:
        raise ValueError(f"unsupported shapes q {tuple(q.shape)}, cache {tuple(k_cache.shape)}")
    if q.dtype != (torch.float16 if k_cache.dtype == torch.float16 else torch.bfloat16):
        raise TypeError(f"attn_decode takes a {'fp16' if k_cache.dtype == torch.float16 else 'bf16'}"
                        " query")
    if cache_seqlens.dtype != torch.int32 or page_table.dtype != torch.int32:
        raise TypeError("cache_seqlens and page_table must be int32")
    if not (q.is_contiguous() and k_cache.is_contiguous() and v_cache.is_contiguous()
            and cache_seqlens.is_contiguous() and page_table.stride(1) == 1):
        raise ValueError("q, caches, cache_seqlens and page_table rows must be contiguous")
    width = page_table.shape[1]
    if max_seqlen is None:
        max_seqlen = width * 16
    if out is None:
        out = torch.empty_like(q)
    elif out.shape != q.shape or out.dtype != q.dtype or not out.is_contiguous():
        raise ValueError("out must be a contiguous tensor shaped like q")
    scale = D ** -0.5 if softmax_scale is None else float(softmax_scale)
    ws = _decode_scratch(B, Hkv, Hq, max_seqlen, dev)
    scales = () if k_scales is None else (k_scales.data_ptr(), v_scales.data_ptr())
    if shared_pages < 0:
        raise ValueError("shared_pages must be >= 0")
    _lib.call(fn, q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), *scales,
              P, int(shared_pages), Hkv, Hq, D, page_table.data_ptr(), page_table.stride(0), width,
              cache_seqlens.data_ptr(), B, max_seqlen, scale, out.data_ptr(),
              ws.data_ptr(), ws.numel(), _errword(dev).ptr(), _lib.stream_of(dev))
    return out
