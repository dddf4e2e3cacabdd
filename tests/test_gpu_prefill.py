"""GPU parity of the varlen prefill attention (attn_prefill over contiguous
K/V, attn_prefill_paged over the pool) vs the float64 oracle.

Tolerance, per output element: one bf16 ulp of the float64 value plus
2^-8 x the attended mass sum_j p_j |v_j| / sum_j p_j. The second term covers
the probabilities' rounding to bf16 for the P V product (relative 2^-9 each,
as in flash attention's bf16 path) with a factor of 2 for the fp32
evaluation."""
import numpy as np
import pytest
import torch

from muserve_amd import _lib
from muserve_amd.kernels import attention as A
from muserve_amd.kv_cache import PagedKVCache
from muserve_amd.scheduler import ContinuousBatchScheduler, InferenceRequest
from oracle import attention as att
from tests.gpu_util import DEV, case

pytestmark = pytest.mark.gpu


def within(got: torch.Tensor, want) -> None:
    want, mass = want
    got = got.float().cpu().numpy().astype(np.float64)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(want), 2.0 ** -126))) - 7)
    tol = ulp + 2.0 ** -8 * mass
    err = np.abs(got - want)
    bad = err > tol
    assert not bad.any(), (f"{bad.sum()} of {bad.size} elements out of tolerance; worst "
                           f"{err[bad].max()} at {np.argwhere(bad)[0]}")


def seqs(lens, seed):
    g = torch.Generator().manual_seed(seed)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    return g, cu


@pytest.mark.parametrize("causal", [True, False])
def test_contiguous_varlen_matches_oracle(causal):
    lens = [1, 5, 15, 16, 17, 31, 33, 64, 100, 257, 600]
    case(f"attn_prefill contiguous varlen causal={causal} lens {lens}")
    g, cu = seqs(lens, 31 + causal)
    T = int(cu[-1])
    q = torch.randn(T, 4, 256, generator=g).bfloat16()
    k = torch.randn(T, 1, 256, generator=g).bfloat16()
    v = torch.randn(T, 1, 256, generator=g).bfloat16()
    out = A.attn_prefill(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), cu.to(DEV), max(lens),
                         max(lens), causal=causal)
    torch.cuda.synchronize()
    A.check_errors(DEV)
    want = att.prefill_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(),
                                 cu.numpy(), 256 ** -0.5, causal, cu_k=cu.numpy(), stats=True)
    within(out, want)


def test_many_sequences_without_key_splits():
    """64 sequences of 256 queries fill 512 workgroups: one key range each,
    the output written by the attention kernel itself."""
    case("attn_prefill 64 x 256 tokens (no key splits)")
    lens = [256] * 64
    g, cu = seqs(lens, 33)
    T = int(cu[-1])
    q = torch.randn(T, 4, 256, generator=g).bfloat16()
    k = torch.randn(T, 1, 256, generator=g).bfloat16()
    v = torch.randn(T, 1, 256, generator=g).bfloat16()
    out = A.attn_prefill(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), cu.to(DEV), 256, 256)
    torch.cuda.synchronize()
    A.check_errors(DEV)
    sample = 4  # the oracle on the first sequences (each is independent)
    n = 256 * sample
    want = att.prefill_attention(q[:n].float().numpy(), k[:n].float().numpy(),
                                 v[:n].float().numpy(), cu[:sample + 1].numpy(), 256 ** -0.5, True,
                                 cu_k=cu[:sample + 1].numpy(), stats=True)
    within(out[:n], want)


def test_contiguous_with_prefix_two_kv_heads_and_scale():
    """nk > nq (a prefix before the queries), 2 KV heads (8 query heads), a
    softmax scale of 0.1, and a sequence with more queries than keys."""
    lq = [7, 40, 3, 129]
    lk = [20, 40, 1, 300]
    case(f"attn_prefill with prefix: nq {lq}, nk {lk}, 2 KV heads")
    g = torch.Generator().manual_seed(35)
    cu_q = torch.tensor(np.concatenate([[0], np.cumsum(lq)]), dtype=torch.int32)
    cu_k = torch.tensor(np.concatenate([[0], np.cumsum(lk)]), dtype=torch.int32)
    q = torch.randn(int(cu_q[-1]), 8, 256, generator=g).bfloat16()
    k = torch.randn(int(cu_k[-1]), 2, 256, generator=g).bfloat16()
    v = torch.randn(int(cu_k[-1]), 2, 256, generator=g).bfloat16()
    out = A.attn_prefill(q.to(DEV), k.to(DEV), v.to(DEV), cu_q.to(DEV), cu_k.to(DEV), max(lq),
                         max(lk), softmax_scale=0.1)
    torch.cuda.synchronize()
    A.check_errors(DEV)
    want = att.prefill_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(),
                                 cu_q.numpy(), 0.1, True, cu_k=cu_k.numpy(), stats=True)
    within(out, want)
    assert not out[int(cu_q[2]):int(cu_q[2]) + 2].float().abs().sum().item()  # saw nothing


def test_paged_chunks_match_oracle():
    """Chunked prefill over the pool: each sequence has a cached prefix and a
    chunk (appended first); queries are the chunk's tokens."""
    prefix = [0, 3, 16, 100, 1000]
    chunk = [17, 1, 32, 64, 300]
    case(f"attn_prefill_paged prefix {prefix} chunk {chunk}")
    g = torch.Generator().manual_seed(36)
    P = 256
    kc = torch.randn(P, 16, 1, 256, generator=g).bfloat16()
    vc = torch.randn(P, 16, 1, 256, generator=g).bfloat16()
    perm = torch.randperm(P, generator=g)
    lens = [p + c for p, c in zip(prefix, chunk)]
    width = max(-(-n // 16) for n in lens)
    table = torch.zeros(len(lens), width, dtype=torch.int32)
    at = 0
    for b, n in enumerate(lens):
        m = -(-n // 16)
        table[b, :m] = perm[at:at + m].to(torch.int32)
        at += m
    cu_q = torch.tensor(np.concatenate([[0], np.cumsum(chunk)]), dtype=torch.int32)
    q = torch.randn(int(cu_q[-1]), 4, 256, generator=g).bfloat16()
    seq_lens = torch.tensor(lens, dtype=torch.int32)
    out = A.attn_prefill_paged(q.to(DEV), kc.to(DEV), vc.to(DEV), cu_q.to(DEV), seq_lens.to(DEV),
                               table.to(DEV), max(chunk))
    torch.cuda.synchronize()
    A.check_errors(DEV)
    want = att.prefill_attention(q.float().numpy(), kc.float().numpy(), vc.float().numpy(),
                                 cu_q.numpy(), 256 ** -0.5, True, lens_k=seq_lens.numpy(),
                                 page_table=table.numpy(), stats=True)
    within(out, want)


def test_scheduler_prefill_entries_through_the_pool():
    """A scheduler step's prefill entries: their tokens' K/V appended through
    plan.slot_mapping, then attn_prefill_paged on plan.cu_seqlens /
    plan.seq_lens / plan.block_tables past the decode entries."""
    case("scheduler prefill chunks -> append -> attn_prefill_paged")
    rng = np.random.default_rng(7)
    g = torch.Generator(device=DEV).manual_seed(7)
    cache = PagedKVCache(1024, num_layers=1, dtype=torch.bfloat16, device=DEV, verbose=False)
    cache._free_pages = rng.permutation(1024).tolist()
    s = ContinuousBatchScheduler(max_batch_size=6, max_seq_len=2048, kv_cache=cache,
                                 chunked_prefill_size=300)
    for i in range(8):
        s.add_request(InferenceRequest(request_id=str(i), input_ids=[0] * int(rng.integers(20, 700)),
                                       max_new_tokens=int(rng.integers(2, 6))))
    checked = 0
    for _ in range(12):
        plan = s.plan_step()
        if plan is None:
            break
        T, nd, n = plan.num_tokens, plan.num_decode, plan.num_entries
        k = torch.randn(T, 1, 256, device=DEV, generator=g).bfloat16()
        v = torch.randn(T, 1, 256, device=DEV, generator=g).bfloat16()
        cache.append(plan.slot_mapping, k, v, layer=0)
        if n > nd:
            cu = plan.cu_seqlens[nd:] - plan.cu_seqlens[nd]
            t0 = int(plan.cu_seqlens[nd].item())
            q = torch.randn(T - t0, 4, 256, device=DEV, generator=g).bfloat16()
            width = plan.block_tables.shape[1]
            out = A.attn_prefill_paged(q, *cache.get_kv_by_layer(0), cu, plan.seq_lens[nd:],
                                       plan.block_tables[nd:], max(c for _, _, c in plan.prefill))
            torch.cuda.synchronize()
            A.check_errors(DEV)
            kc, vc = cache.get_kv_by_layer(0)
            want = att.prefill_attention(q.float().cpu().numpy(), kc.float().cpu().numpy(),
                                         vc.float().cpu().numpy(), cu.cpu().numpy(), 256 ** -0.5,
                                         True, lens_k=plan.seq_lens[nd:].cpu().numpy(),
                                         page_table=plan.block_tables[nd:].cpu().numpy(),
                                         stats=True)
            within(out, want)
            assert width >= 1
            checked += 1
        s.complete_step(plan)
    s.check_errors()
    assert checked >= 3


def test_bad_page_and_bad_offsets_are_flagged():
    case("attn_prefill_paged bad page id; attn_prefill offsets past the buffer")
    g = torch.Generator().manual_seed(37)
    kc = torch.randn(8, 16, 1, 256, generator=g).bfloat16().to(DEV)
    vc = torch.randn(8, 16, 1, 256, generator=g).bfloat16().to(DEV)
    q = torch.randn(20, 4, 256, generator=g).bfloat16().to(DEV)
    table = torch.tensor([[1, 99]], dtype=torch.int32, device=DEV)
    cu = torch.tensor([0, 20], dtype=torch.int32, device=DEV)
    A.attn_prefill_paged(q, kc, vc, cu, torch.tensor([30], dtype=torch.int32, device=DEV), table,
                         20)
    with pytest.raises(_lib.MkvDeviceError, match="page id"):
        A.check_errors(DEV)
    k = torch.randn(20, 1, 256, generator=g).bfloat16().to(DEV)
    cu_k = torch.tensor([0, 25], dtype=torch.int32, device=DEV)  # past the 20 key rows
    A.attn_prefill(q, k, k.clone(), cu, cu_k, 20, 25)
    with pytest.raises(_lib.MkvDeviceError, match="table"):
        A.check_errors(DEV)


def test_offsets_without_rows_are_refused():
    case("attn_prefill with no query rows and an offset past them")
    q = torch.empty(0, 4, 256, dtype=torch.bfloat16, device=DEV)
    k = torch.zeros(20, 1, 256, dtype=torch.bfloat16, device=DEV)
    cu_q = torch.tensor([0, 5], dtype=torch.int32, device=DEV)
    cu_k = torch.tensor([0, 20], dtype=torch.int32, device=DEV)
    with pytest.raises(_lib.MkvError, match="null pointer"):
        A.attn_prefill(q, k, k.clone(), cu_q, cu_k, 5, 20)


@pytest.mark.parametrize("split_len", [64, 128, 192])
def test_forced_key_splits_through_the_c_abi(split_len):
    """Key ranges of one, two and three 64-key tiles (the double-buffered
    loop's prologue-only, one-store and store-plus-prefetch cases), ranges
    that end inside a sequence or past its causal limit, and the merge, with
    the split chosen by the caller of the C ABI."""
    lens = [1, 63, 64, 65, 128, 129, 200, 383]
    case(f"mkv_prefill_attention_bf16 forced split_len {split_len}, lens {lens}")
    _forced_splits(lens, split_len, 38 + split_len)


@pytest.mark.parametrize("splits", [2, 3, 4, 5, 6, 7, 8, 9])
def test_every_merged_range_count(splits):
    """64-key ranges, as many as `splits`: the merge reads each count from 2
    to 8 with its own fixed number of loads and more than 8 through a loop;
    sequences end inside, at and past the ranges' edges."""
    lens = [1, 63, 64, 65, 64 * splits - 1, 64 * splits]
    case(f"mkv_prefill_attention_bf16 {splits} ranges of 64 keys, lens {lens}")
    _forced_splits(lens, 64, 60 + splits)


def _forced_splits(lens, split_len, seed):
    g, cu = seqs(lens, seed)
    T, max_k = int(cu[-1]), max(lens)
    q = torch.randn(T, 4, 256, generator=g).bfloat16().to(DEV)
    k = torch.randn(T, 1, 256, generator=g).bfloat16().to(DEV)
    v = torch.randn(T, 1, 256, generator=g).bfloat16().to(DEV)
    splits = -(-max_k // split_len)
    lib = _lib.load()
    ws_bytes = lib.mkv_prefill_attention_workspace_bytes(T, 4, splits)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=DEV)
    out = torch.empty_like(q)
    cu_d = cu.to(DEV)
    _lib.call("mkv_prefill_attention_bf16", q.data_ptr(), k.data_ptr(), v.data_ptr(), T, 1, 4, 256,
              None, 0, 0, cu_d.data_ptr(), cu_d.data_ptr(), None, len(lens), T, max_k,
              256 ** -0.5, 1, splits, split_len, out.data_ptr(), ws.data_ptr(), ws_bytes,
              A._errword(DEV).ptr(), _lib.stream_of(DEV))
    torch.cuda.synchronize()
    A.check_errors(DEV)
    want = att.prefill_attention(q.float().cpu().numpy(), k.float().cpu().numpy(),
                                 v.float().cpu().numpy(), cu.numpy(), 256 ** -0.5, True,
                                 cu_k=cu.numpy(), stats=True)
    within(out, want)


def _one_hot_keys(n_rows, heads=1):
    """V row j = e_(j mod 256) (bf16 ones): with a zero query every visible
    key has weight 1 / n, so output dim d is (visible keys j = d mod 256) / n
    and one key more or less changes a dim by about 1 / n, far above the
    rounding (the worst-case tolerance above cannot see a single key once a
    row attends to a few hundred)."""
    v = torch.zeros(n_rows, heads, 256)
    idx = torch.arange(n_rows)
    v[idx, :, idx % 256] = 1.0
    return v.bfloat16()


def _one_hot_want(nq, nk, causal):
    """Closed form for a zero query over one-hot keys: [nq, 256] float64."""
    out = np.zeros((nq, 256))
    d = np.arange(256)
    for t in range(nq):
        last = nk - nq + t if causal else nk - 1  # bottom-right causal alignment
        if last < 0:
            continue
        n = last + 1
        cnt = np.where(d <= last, (last - d) // 256 + 1, 0)
        out[t] = cnt / n
    return out


def _bf16_close(got, want):
    got = got.float().cpu().numpy().astype(np.float64)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(want), 2.0 ** -126))) - 7)
    err = np.abs(got - want)
    assert (err <= ulp).all(), f"worst {err.max()} at {np.unravel_index(err.argmax(), err.shape)}"


@pytest.mark.parametrize("causal", [True, False])
def test_understated_max_seqlen_k_keeps_every_key(causal):
    """A max_seqlen_k below the real key count (600 for 2000 keys): the split
    ranges cover 3 x 256 keys, and the last range must run to the end."""
    nq = nk = 2000
    case(f"attn_prefill one-hot keys, {nk} keys, max_seqlen_k 600, causal={causal}")
    q = torch.zeros(nq, 4, 256).bfloat16().to(DEV)
    k = torch.randn(nk, 1, 256, generator=torch.Generator().manual_seed(41)).bfloat16().to(DEV)
    v = _one_hot_keys(nk).to(DEV)
    cu = torch.tensor([0, nq], dtype=torch.int32, device=DEV)
    out = A.attn_prefill(q, k, v, cu, cu, nq, 600, causal=causal)
    torch.cuda.synchronize()
    A.check_errors(DEV)
    want = _one_hot_want(nq, nk, causal)
    for h in range(4):
        _bf16_close(out[:, h], want)


def test_one_hot_keys_pin_every_tile_and_split_boundary():
    """Sequences with a prefix (nk > nq) and lengths around the 64-key tiles
    and the split boundaries, with forced key splits through the C ABI: each
    output dim counts its visible keys exactly, so a key dropped or added at
    any tile or range boundary shows."""
    nqs = [1, 63, 64, 65, 129, 300]
    nks = [1, 64, 127, 65, 300, 777]
    case(f"mkv_prefill_attention_bf16 one-hot keys, forced splits of 128, nq {nqs} nk {nks}")
    cu_q = torch.tensor(np.concatenate([[0], np.cumsum(nqs)]), dtype=torch.int32)
    cu_k = torch.tensor(np.concatenate([[0], np.cumsum(nks)]), dtype=torch.int32)
    Tq, Tk = int(cu_q[-1]), int(cu_k[-1])
    q = torch.zeros(Tq + 7, 4, 256).bfloat16().to(DEV)  # 7 rows past every sequence
    k = torch.randn(Tk, 1, 256, generator=torch.Generator().manual_seed(42)).bfloat16().to(DEV)
    v = torch.cat([_one_hot_keys(n) for n in nks]).to(DEV)
    split_len, max_k = 128, max(nks)
    splits = -(-max_k // split_len)
    lib = _lib.load()
    ws_bytes = lib.mkv_prefill_attention_workspace_bytes(Tq + 7, 4, splits)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=DEV)
    canary = torch.full((Tq + 7, 4, 256), 0x1234, dtype=torch.int16, device=DEV)
    out = canary.clone().view(torch.bfloat16)
    cu_qd, cu_kd = cu_q.to(DEV), cu_k.to(DEV)
    _lib.call("mkv_prefill_attention_bf16", q.data_ptr(), k.data_ptr(), v.data_ptr(), Tk, 1, 4,
              256, None, 0, 0, cu_qd.data_ptr(), cu_kd.data_ptr(), None, len(nqs), Tq + 7,
              max(nqs), 256 ** -0.5, 1, splits, split_len, out.data_ptr(), ws.data_ptr(),
              ws_bytes, A._errword(DEV).ptr(), _lib.stream_of(DEV))
    torch.cuda.synchronize()
    A.check_errors(DEV)
    for b, (nq, nk) in enumerate(zip(nqs, nks)):
        want = _one_hot_want(nq, nk, True)
        rows = out[int(cu_q[b]):int(cu_q[b + 1])]
        for h in range(4):
            _bf16_close(rows[:, h], want)
    # rows outside every sequence's queries are left alone by the merge
    assert torch.equal(out[Tq:].view(torch.int16), canary[Tq:])


@pytest.mark.parametrize("lens,scale,grow", [
    ([31, 33, 97], 256 ** -0.5, 0.0),             # 4-wave workgroups: 32-query tiles
    ([63, 65, 129, 1], -0.07, 0.0),               # a negative scale (queries' signs flip)
    ([40, 300], 0.0, 0.0),                        # zero: every visible key weighs the same
    ([64] * 70 + [65, 127, 191], 0.05, 0.0),      # 8-wave workgroups: 64-query tiles
    ([1300, 700] + [64] * 60, 256 ** -0.5, 3e-3),  # maxima that keep rising
])
def test_query_tiles_scales_and_rising_maxima(lens, scale, grow):
    """Both workgroup sizes at the edges of their query tiles; scales whose
    sign and zero the kernel handles apart; and keys that grow along the
    sequence, so that the running maximum moves in every tile."""
    case(f"attn_prefill tiles: {len(lens)} sequences of {min(lens)}..{max(lens)}, scale {scale}")
    g, cu = seqs(lens, 71 + len(lens))
    T = int(cu[-1])
    pos = torch.cat([torch.arange(n) for n in lens]).float()
    q = torch.randn(T, 4, 256, generator=g).bfloat16()
    k = (torch.randn(T, 1, 256, generator=g) * (1.0 + grow * pos[:, None, None])).bfloat16()
    v = torch.randn(T, 1, 256, generator=g).bfloat16()
    out = A.attn_prefill(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), cu.to(DEV), max(lens),
                         max(lens), softmax_scale=scale)
    torch.cuda.synchronize()
    A.check_errors(DEV)
    want = att.prefill_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(),
                                 cu.numpy(), scale, True, cu_k=cu.numpy(), stats=True)
    within(out, want)


@pytest.mark.parametrize("lens", [[40, 97], [64] * 70 + [191, 320]])  # 4 and 8 waves
@pytest.mark.parametrize("c", [300.0, 6000.0, 20500.0, 21500.0, -20500.0, 3e6])
def test_large_finite_scores(c, lens):
    """Scores far past 2^24 in log2 units, where one fp32 step is more than
    the whole range of the exponential: the largest score's weight is still
    exactly 1. Every query is c in every dim; the keys are |c| and |c| / 2 in
    turn, so the visible keys of the larger product share the weight (the
    other's is 0 in float64 too; sums of 256 products of 8-bit mantissas are
    exact in fp32)."""
    case(f"attn_prefill: finite scores of about {256 * c * abs(c):.1e}, {len(lens)} sequences")
    g, cu = seqs(lens, 91)
    T = int(cu[-1])
    q = torch.full((T, 4, 256), c).bfloat16()
    odd = torch.cat([torch.arange(n) for n in lens]) % 2
    k = (abs(c) * (1.0 - 0.5 * odd))[:, None, None].expand(T, 1, 256).contiguous().bfloat16()
    v = torch.randn(T, 1, 256, generator=g).bfloat16()
    out = A.attn_prefill(q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV), cu.to(DEV), max(lens),
                         max(lens))
    torch.cuda.synchronize()
    A.check_errors(DEV)
    want = att.prefill_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(),
                                 cu.numpy(), 256 ** -0.5, True, cu_k=cu.numpy(), stats=True)
    within(out, want)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("splits,heads,nqs,nks", [
    # both sides of the 64-query and 64-key tiles, no queries, no visible keys
    (1, 1, [1, 0, 63, 64, 65, 129, 70], [1, 9, 64, 127, 65, 300, 20]),
    (2, 2, [1, 65, 0, 64, 200], [777, 65, 0, 640, 200]),
    (16, 1, [130, 1, 700, 64], [1500, 2049, 700, 64]),   # all tasks at once: ranges of 2 tiles up
    (40, 1, [20], [2560]),                               # many ranges of one query tile
    (3, 1, [1900, 1200] + [64] * 220, [1900, 1200] + [64] * 220),  # more tasks than CUs
    (5, 4, [300] * 30, [960] * 30),                      # 600 tasks of one length over 4 heads
])
def test_planned_launches_pin_every_task(splits, heads, nqs, nks, causal):
    """The schedule made on the device: with zero queries over one-hot keys a
    task dropped, doubled or cut in the wrong place changes what a row counts.
    Output rows past the queries stay as they were."""
    case(f"prefill planned: {len(nqs)} sequences, {heads} heads, {splits} ranges, causal={causal}")
    Tq, Tk = sum(nqs), sum(nks)
    cu_q = torch.tensor(np.cumsum([0] + nqs), dtype=torch.int32, device=DEV)
    cu_k = torch.tensor(np.cumsum([0] + nks), dtype=torch.int32, device=DEV)
    g = torch.Generator().manual_seed(43)
    q = torch.zeros(Tq, 4 * heads, 256).bfloat16().to(DEV)
    k = torch.randn(Tk, heads, 256, generator=g).bfloat16().to(DEV)
    v = torch.cat([_one_hot_keys(n, heads) for n in nks]).to(DEV)
    out = torch.full((Tq + 8, 4 * heads, 256), 7.0, dtype=torch.bfloat16, device=DEV)
    n = _lib.load().mkv_prefill_attention_plan_bytes(Tq, 4 * heads, heads, len(nqs), max(nqs),
                                                     splits)
    ws = torch.empty(n, dtype=torch.uint8, device=DEV)
    _lib.call("mkv_prefill_attention_planned_bf16", q.data_ptr(), k.data_ptr(), v.data_ptr(), Tk,
              heads, 4 * heads, 256, None, 0, 0, cu_q.data_ptr(), cu_k.data_ptr(), None, len(nqs),
              Tq, max(nqs), 256 ** -0.5, int(causal), splits, out.data_ptr(), ws.data_ptr(), n,
              A._errword(DEV).ptr(), _lib.stream_of(DEV))
    torch.cuda.synchronize()
    A.check_errors(DEV)
    off = 0
    for nq, nk in zip(nqs, nks):
        want = _one_hot_want(nq, nk, causal)
        for h in range(4 * heads):
            if nq:
                _bf16_close(out[off:off + nq, h], want)
        off += nq
    assert bool((out[Tq:] == 7.0).all())


def _paged_one_hot(nks, heads, seed, spare=5, width=None):
    """One-hot V rows (position j of a sequence is e_(j mod 256)) and random K
    on shuffled pages: k, v pools and the block table, on the device."""
    rng = np.random.default_rng(seed)
    pages = [-(-n // 16) for n in nks]
    P = sum(pages) + spare
    perm = rng.permutation(P)
    table = np.zeros((len(nks), width or max(1, max(pages))), dtype=np.int32)
    v = torch.zeros(P, 16, heads, 256).bfloat16()
    at = 0
    for b, n in enumerate(pages):
        table[b, :n] = perm[at:at + n]
        v[torch.from_numpy(perm[at:at + n])] = _one_hot_keys(16 * n, heads).view(n, 16, heads, 256)
        at += n
    k = torch.randn(P, 16, heads, 256, generator=torch.Generator().manual_seed(seed)).bfloat16()
    return k.to(DEV), v.to(DEV), torch.from_numpy(table).to(DEV)


def _planned_paged(k, v, table, cu_q, lens_k, Tq, max_q, splits, causal=True):
    """A planned launch over the pool through the C ABI, its workspace filled
    with ones (NaN, if read as partial rows) and followed by a canary, as its
    8 rows past Tq are: (out [Tq, 4 heads, 256], no canary touched)."""
    heads, batch = k.shape[2], len(lens_k)
    q = torch.zeros(Tq, 4 * heads, 256).bfloat16().to(DEV)
    out = torch.full((Tq + 8, 4 * heads, 256), 7.0, dtype=torch.bfloat16, device=DEV)
    n = _lib.load().mkv_prefill_attention_plan_bytes(Tq, 4 * heads, heads, batch, max_q, splits)
    assert n > 0
    ws = torch.full((n + 4096,), 0xFF, dtype=torch.uint8, device=DEV)
    cu = torch.tensor(cu_q, dtype=torch.int32, device=DEV)
    lens = torch.tensor(lens_k, dtype=torch.int32, device=DEV)
    _lib.call("mkv_prefill_attention_planned_bf16", q.data_ptr(), k.data_ptr(), v.data_ptr(),
              k.shape[0], heads, 4 * heads, 256, table.data_ptr(), table.stride(0),
              table.shape[1], cu.data_ptr(), None, lens.data_ptr(), batch, Tq, max_q,
              256 ** -0.5, int(causal), splits, out.data_ptr(), ws.data_ptr(), n,
              A._errword(DEV).ptr(), _lib.stream_of(DEV))
    torch.cuda.synchronize()
    assert bool((ws[n:] == 0xFF).all()) and bool((out[Tq:] == 7.0).all())
    return out[:Tq]


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("splits,heads,nqs,prefix", [
    (12, 2, [300, 1, 0, 129, 64], [3000, 777, 50, 9, 1500]),  # all at once, ranges over 2 heads
    (40, 1, [33, 65], [2527, 640]),                           # many ranges of few tiles
    (3, 1, [1200, 700] + [70] * 220, [600, 0] + [100] * 220),  # more tasks than CUs
    (4, 1, [500] + [20] * 300, [2000] + [30] * 300),          # more than 256 sequences
    (9, 1, [500] + [0] * 280 + [20] * 19, [2000] + [30] * 299),  # and all tasks at once
])
def test_planned_paged_chunks_pin_every_task(splits, heads, nqs, prefix, causal):
    """A planned launch over shuffled pages, with unequal chunks on unequal
    cached prefixes: the schedule and the page lookups at every range's start."""
    nks = [a + b for a, b in zip(nqs, prefix)]
    case(f"prefill planned, paged: {len(nqs)} sequences, {heads} heads, {splits} ranges, "
         f"causal={causal}")
    k, v, table = _paged_one_hot(nks, heads, 44)
    cu = np.cumsum([0] + nqs)
    out = _planned_paged(k, v, table, cu, nks, int(cu[-1]), max(nqs), splits, causal)
    A.check_errors(DEV)
    for b, (nq, nk) in enumerate(zip(nqs, nks)):
        want = _one_hot_want(nq, nk, causal)
        for h in range(4 * heads):
            if nq:
                _bf16_close(out[cu[b]:cu[b + 1], h], want)


def test_planned_paged_chunks_match_oracle():
    """Random values through attn_prefill_paged, at a shape that it plans."""
    chunk, prefix = [300, 40, 129], [3000, 500, 9000]
    lens = [p + c for p, c in zip(prefix, chunk)]
    case(f"attn_prefill_paged planned: prefix {prefix} chunk {chunk}")
    assert A.prefill_schedule(sum(chunk), max(chunk), max(lens), 3, 1, True,
                              A._prefill_cus(torch.device(DEV)))[2]
    g = torch.Generator().manual_seed(45)
    k, _, table = _paged_one_hot(lens, 1, 45)
    v = torch.randn(k.shape, generator=g).bfloat16().to(DEV)
    cu = torch.tensor(np.cumsum([0] + chunk), dtype=torch.int32)
    q = torch.randn(sum(chunk), 4, 256, generator=g).bfloat16()
    seq_lens = torch.tensor(lens, dtype=torch.int32)
    out = A.attn_prefill_paged(q.to(DEV), k, v, cu.to(DEV), seq_lens.to(DEV), table, max(chunk),
                               max_seqlen_k=max(lens))
    torch.cuda.synchronize()
    A.check_errors(DEV)
    want = att.prefill_attention(q.float().numpy(), k.float().cpu().numpy(),
                                 v.float().cpu().numpy(), cu.numpy(), 256 ** -0.5, True,
                                 lens_k=seq_lens.numpy(), page_table=table.cpu().numpy(),
                                 stats=True)
    within(out, want)


@pytest.mark.parametrize("what", ["page", "length", "negative length", "queries", "decreasing",
                                  "overlapping"])
def test_planned_launches_flag_bad_inputs(what):
    """Ids, lengths and offsets that the plan kernel (or a planned range)
    finds outside their buffers are flagged; the other sequences are served and
    nothing is written outside the queries, the output or the workspace."""
    case(f"prefill planned, paged: bad {what}")
    nqs, nks, splits = [100, 200, 70], [1500, 900, 640], 8
    k, v, table = _paged_one_hot(nks, 1, 46)
    cu, lens, Tq, max_q = list(np.cumsum([0] + nqs)), list(nks), sum(nqs), max(nqs)
    served = {0: (0, nqs[0], nks[0]), 1: (100, nqs[1], nks[1]), 2: (300, nqs[2], nks[2])}
    text = "table"
    if what == "page":
        table[1, 20] = k.shape[0] + 3  # keys 320 .. 335 of sequence 1 read as zeros
        text = "page id"
        del served[1]
    elif what == "length":  # 200 keys past the table's 94 pages: clamped to them
        lens[0] = 16 * table.shape[1] + 200
        served[0] = (0, nqs[0], 16 * table.shape[1])
    elif what == "negative length":
        lens[2] = -5
        del served[2]
    elif what == "queries":  # the last sequence would end 10 rows past the buffer
        cu[3] += 10
        del served[2]
    elif what == "decreasing":  # sequence 1 ends before it begins, 2 is empty
        cu[2] = cu[3] = 60
        del served[1], served[2]
    else:  # the same rows and keys four times: more tiles than the bounds expect
        nqs, nks = [640], [1500]
        cu, Tq, max_q = [0, 640, 0, 640, 0, 640, 0, 640], 640, 640
        lens, table = [1500] * 7, table[:1].expand(7, -1).contiguous()
        served = {}
    out = _planned_paged(k, v, table, cu, lens, Tq, max_q, splits)
    with pytest.raises(_lib.MkvDeviceError, match=text):
        A.check_errors(DEV)
    for first, nq, nk in served.values():
        want = _one_hot_want(nq, nk, True)
        for h in range(4):
            _bf16_close(out[first:first + nq, h], want)
    if what == "queries":
        assert bool((out[300:] == 7.0).all())
    elif what == "decreasing":
        assert bool((out[100:] == 7.0).all())
    elif what == "negative length":
        assert not out[300:].float().abs().sum().item()  # no key: zeros
    elif what == "page":  # each key's weight is 1 / n; those of the bad page count nothing
        want = _one_hot_want(200, 900, True)
        n = np.arange(701, 901)[:, None]
        want[:, 320 % 256:320 % 256 + 16] -= 1.0 / n
        for h in range(4):
            _bf16_close(out[100:300, h], want)


@pytest.mark.parametrize("tokens,max_q,max_k,batch,heads", [
    (1, 1, 1, 1, 1), (77, 77, 77, 1, 1), (13897, 4096, 4096, 6, 1), (32768, 4096, 4096, 8, 1),
    (2572, 1428, 6540, 2, 1), (3, 1, 1 << 20, 3, 2), (4096, 16, 64, 256, 1),
    (1 << 20, 1 << 20, 1 << 20, 1, 1), (5000, 4096, 4096, 1100, 1), (200, 200, 9000, 1, 8)])
def test_schedules_are_accepted(tokens, max_q, max_k, batch, heads):
    """Every schedule the host rule makes is one the entry points take."""
    splits, split_len, planned = A.prefill_schedule(tokens, max_q, max_k, batch, heads, True, 256)
    assert splits >= 1 and heads * splits <= 65535
    if planned:
        assert _lib.load().mkv_prefill_attention_plan_bytes(tokens, 4 * heads, heads, batch, max_q,
                                                            splits) > 0
    elif splits > 1:
        assert split_len > 0 and split_len % 64 == 0 and splits * split_len >= max_k


@pytest.mark.parametrize("paged", [False, True])
def test_more_sequences_than_a_plan_holds(paged, monkeypatch):
    """Ragged batches of more than 1024 sequences are planned 1024 at a time,
    whichever part the long ones are in."""
    lens = [3] * 1024 + [700] + [2] * 1100 + [300]
    case(f"attn_prefill {len(lens)} sequences of 2..700, paged={paged}")
    cu = np.cumsum([0] + lens)
    T = int(cu[-1])
    q = torch.zeros(T, 4, 256).bfloat16().to(DEV)
    cu_d = torch.tensor(cu, dtype=torch.int32, device=DEV)
    calls = []
    real = _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: calls.append(name) or real(name, *a))
    if paged:
        k, v, table = _paged_one_hot(lens, 1, 48)
        out = A.attn_prefill_paged(q, k, v, cu_d, torch.tensor(lens, dtype=torch.int32, device=DEV),
                                   table, max(lens), max_seqlen_k=max(lens))
    else:
        v = torch.cat([_one_hot_keys(n) for n in lens]).to(DEV)
        k = torch.randn(T, 1, 256, generator=torch.Generator().manual_seed(48)).bfloat16().to(DEV)
        out = A.attn_prefill(q, k, v, cu_d, cu_d, max(lens), max(lens))
    torch.cuda.synchronize()
    A.check_errors(DEV)
    assert calls == ["mkv_prefill_attention_planned_bf16"] * 3
    want = np.concatenate([_one_hot_want(n, n, True) for n in lens])
    for h in range(4):
        _bf16_close(out[:, h], want)


@pytest.mark.parametrize("lens", [[64], [40, 64, 7], [300, 20]])
def test_loose_bounds_cost_no_plan(lens, monkeypatch):
    """Bounds far above what the rows can hold: the schedule is made for the
    rows, and the output is that of tight bounds."""
    case(f"attn_prefill lens {lens} under bounds of 4096")
    g, cu = seqs(lens, 47)
    T = int(cu[-1])
    q, k, v = (torch.randn(T, h, 256, generator=g).bfloat16().to(DEV) for h in (4, 1, 1))
    cu = cu.to(DEV)
    made = []
    rule = A.prefill_schedule
    monkeypatch.setattr(A, "prefill_schedule", lambda *a: made.append(rule(*a)) or made[-1])
    got = A.attn_prefill(q, k, v, cu, cu, 4096, 4096)
    want = A.attn_prefill(q, k, v, cu, cu, T, T)
    torch.cuda.synchronize()
    A.check_errors(DEV)
    assert made[0] == made[1] and not made[0][2]
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


def test_planned_calls_on_two_streams():
    """Calls of different lengths at once on two streams: neither reads the
    other's plan or partial rows."""
    case("attn_prefill: two streams, ragged prompts of different lengths")
    jobs = []
    for seed, lens in ((1, [1500, 90, 700, 2000] * 4), (2, [300, 2500, 64, 1100] * 4)):
        g = torch.Generator().manual_seed(seed)
        T = sum(lens)
        q, k, v = (torch.randn(T, h, 256, generator=g).bfloat16().to(DEV) for h in (4, 1, 1))
        cu = torch.tensor(np.cumsum([0] + lens), dtype=torch.int32, device=DEV)
        want = A.attn_prefill(q, k, v, cu, cu, max(lens), max(lens))
        jobs.append((torch.cuda.Stream(DEV), (q, k, v, cu, cu, max(lens), max(lens)), want, []))
    torch.cuda.synchronize()
    for _ in range(6):
        for stream, args, _, outs in jobs:
            with torch.cuda.stream(stream):
                outs.append(A.attn_prefill(*args))
    torch.cuda.synchronize()
    A.check_errors(DEV)
    for _, _, want, outs in jobs:
        for out in outs:
            assert torch.equal(out.view(torch.int16), want.view(torch.int16))
