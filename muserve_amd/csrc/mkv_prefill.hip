// mkv_prefill.hip — varlen prefill attention (gfx950, MFMA): the math of
// attn_prefill (muserve/kernels/attention.py:6-25, flash_attn_varlen_func)
// over contiguous K/V, and the same over the paged pool for chunked prefill
// (a chunk's queries attend to the sequence's cached prefix and to
// themselves).
//
// Sequence b has nq queries and nk keys; query t sits at position nk - nq + t
// (causal masking aligned to the bottom-right corner) and, when causal,
// attends to positions 0 .. nk - nq + t. Query head h reads KV head h / 4.
//
// A workgroup (8 waves) takes 64 query tokens of one sequence and KV head;
// wave w holds query head 4*hk + w % 4 for tokens 32 (w / 4) .. +31, so the 8
// waves share every K/V tile through LDS. Per 64-token KV tile:
//   * K and V rows go straight into LDS (global_load_lds_dwordx4), in blocks
//     of 8 rows x 128 bytes (below); the next tile's loads are in flight in
//     the other buffer while this one is computed, one barrier per tile;
//   * the scores are computed transposed, S^T = K Q^T, on MFMA
//     (v_mfma_f32_32x32x16_bf16): A = 32 K rows from LDS, B = the wave's 32
//     queries, held in registers for the whole loop. A lane then holds scores
//     of one query only (column lane % 32), so the online softmax (fp32, exp2,
//     log2(e) folded into the scale) has one running maximum per lane and
//     reduces over registers, with one exchange between the half waves;
//   * the P^T operand of O^T += V^T P^T is those same registers rounded to
//     bf16: the sum over keys runs in the order in which the score tile's
//     rows lie in a lane, and V^T is read to match by gfx950's transposing
//     LDS load (ds_read_b64_tr_b16). P never passes through LDS.
// The output is O / l, rounded to bf16 once, turned to rows through LDS.
//
// What bounds it: a K or V byte read from LDS feeds 32 query rows, so a tile
// is 4096 cycles of a CU's matrix cores against 512 KiB of LDS reads; with 16
// rows per wave (v_mfma_f32_16x16x32_bf16, P through LDS, tiles through
// registers) the LDS reads and the passes of P bounded it, 560 us against
// 380 us for 8 x 4096 causal tokens of one KV head on MI355X. What then set
// the time was which CU ran which tile: workgroups are dealt to the 8 XCDs in
// turn, and with a sequence's tiles in consecutive workgroups an XCD had 113
// key tiles on its fullest CU against 65 on average. With the order below
// (prefill_attn_kernel) the same launch takes 254-276 us (1.00-1.08 PFLOP/s
// of the visible pairs, by the clock it gets); six prompts of 80 to 4096
// tokens, planned on the device (prefill_plan_kernel), 177 -> 142-149 us. While a
// CU is busy its matrix cores are so 59 % of the time, at 1.9 GHz.
#include <float.h>
#include <limits.h>
#include <math.h>

#include "mkv_device.h"

namespace mkv {
namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) u32x2v lds_u32x2;

// ds_read_b64_tr_b16: within each group of 16 lanes, lane j names an 8-byte
// row R_j of 4 bf16; lane i receives R_{4e + i/4}[i % 4] as element e (a
// layout probed on the device). Lane j of the group naming
// V[t0 + j/4][d0 + 4 (j % 4) ..] therefore hands lane i the 4 values
// V[t0 .. t0+3][d0 + i]: one dim of 4 tokens, the MFMA A-operand order of V^T.
__device__ __forceinline__ s16x4 lds_read_tr16(uint32_t addr) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(uintptr_t)addr);
}

constexpr int kPD = 256;           // head_dim
constexpr int kPRow = kPD * 2;     // bytes of one bf16 row
constexpr int kPG = 4;             // query heads per KV head
constexpr int kWTok = 32;          // query tokens per wave
constexpr int kQTok = 64;          // query tokens per workgroup of 8 waves
constexpr int kKvTile = 64;        // KV tokens per step
constexpr int kTileB = kKvTile * kPRow;     // bytes of one staged K (or V) tile
constexpr int kCus = 256;          // MI355X's, the most a plan counts; LDS holds one workgroup per CU
constexpr int kXcds = 8;           // MI355X: workgroups go round robin over 8 XCDs

// One workgroup's task of a planned launch: range z of p of the query tile
// from query qt of a sequence, for KV head hk (zp = z + 65536 p).
struct PlanItem {
  int32_t qs, nq, kbase, nk;
  int32_t b, hk, qt;
  uint32_t zp;
};
static_assert(sizeof(PlanItem) == 32, "two 16-byte loads");
struct Plan {
  int32_t items, cuts;  // tasks; (query tile, KV head) pairs of several ranges
  int32_t pad[14];
};
constexpr int kPlanThreads = 1024, kPlanSmall = 256;  // (the small form: quicker barriers)
constexpr int kPlanSlots = 4;                          // query tiles per thread
constexpr int kPlanTiles = kPlanThreads * kPlanSlots;  // query tiles at most
constexpr int kPlanSeqs = kPlanThreads;                // sequences at most
static_assert(kCus <= kPlanSmall, "tasks that run at once have a bin each, and a tile per thread");
constexpr int kPlanLeast = 2;                          // key tiles per range at least
constexpr int kPlanTries = 16;                         // range lengths that a plan tries

struct PrefillArgs {
  const uint8_t* q;      // [Tq, Hq, 256] bf16
  const uint8_t* k;      // paged [P, 16, Hkv, 256] or contiguous [Tk, Hkv, 256] bf16
  const uint8_t* v;
  const int32_t* table;  // paged: [B, tstride] page ids; null: contiguous
  int64_t tstride;
  int32_t twidth;
  int64_t kv_units;      // pages (paged) or token rows (contiguous)
  const int32_t* cu_q;   // [B + 1]
  const int32_t* cu_k;   // contiguous: [B + 1]
  const int32_t* lens_k; // paged: [B]
  int64_t num_q;         // query rows Tq
  int32_t max_q;         // the launch's bound on a sequence's queries
  uint8_t* out;          // [Tq, Hq, 256] bf16
  int32_t hkv;
  int32_t causal;
  int32_t tok;           // query tokens per workgroup of this launch (a power of two)
  uint32_t ranks;        // query tiles of the longest sequence the launch covers
  uint32_t rank0;        // the first tile rank of this launch
  int32_t turn;          // ranks turn over the XCDs
  int32_t cus;           // the device's CUs (kCus at most)
  int32_t splits;        // key ranges per (query tile, KV head) at most
  int32_t split_len;     // keys a range aims at (a multiple of the KV tile)
  Plan* plan;            // null: the grid is the schedule
  PlanItem* items;       // the plan's tasks, longest first
  PlanItem* cut;         // its pairs of several ranges (z unused)
  int32_t max_items, max_cuts;
  float* part;           // splits > 1: [Tq, Hq, splits, 256] unnormalised outputs
  float* ml;             // splits > 1: [Tq, Hq, splits, 2] (max, sum), log2 units
  float scale_log2;      // |softmax scale| * log2(e), positive
  uint32_t q_sign;       // 0x80008000 when the scale is negative: flips the queries' signs
  int32_t* err;
};

__device__ __forceinline__ uint16_t bf16_bits(float x) { return f32_to_bf16_rne(x); }

// two floats to bf16 (round to nearest even) by one v_cvt_pk_bf16_f32
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t bf16_pack(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
}

// A lane's value and that of the other half wave's lane of the same query,
// combined.
__device__ __forceinline__ float2 both_halves(float x) {
  const uint32_t w = __builtin_bit_cast(uint32_t, x);
  const u32x2v r = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  const uint32_t lo = r.x, hi = r.y;
  return float2{__builtin_bit_cast(float, lo), __builtin_bit_cast(float, hi)};
}
__device__ __forceinline__ float half_max(float x) {
  const float2 y = both_halves(x);
  return fmaxf(y.x, y.y);
}
__device__ __forceinline__ float half_sum(float x) {
  const float2 y = both_halves(x);
  return y.x + y.y;
}

// The queries of sequence b, from row qs: offsets outside the buffer, or more
// queries than the launch covers, are bad; nothing of the sequence (or nothing
// past the bound) is touched.
__device__ __forceinline__ int32_t seq_queries(const PrefillArgs& a, int64_t b, int32_t& qs,
                                               bool& bad) {
  qs = a.cu_q[b];
  const int32_t n = a.cu_q[b + 1] - qs;
  const bool ok = qs >= 0 && n >= 0 && (int64_t)qs + n <= a.num_q;
  bad = !ok || n > a.max_q;
  return ok ? (n < a.max_q ? n : a.max_q) : 0;
}

// The keys of sequence b: a length checked against what the table (or the
// buffer) holds; a bad one is flagged and clamped.
__device__ __forceinline__ int64_t seq_keys(const PrefillArgs& a, int64_t b, int64_t& kbase,
                                            bool& bad) {
  int64_t nk;
  kbase = 0;
  bad = false;
  if (a.table) {
    nk = a.lens_k[b];
    const int64_t cap = (int64_t)a.twidth * 16;
    if (nk < 0 || nk > cap) {
      bad = true;
      nk = nk < 0 ? 0 : cap;
    }
  } else {
    kbase = a.cu_k[b];
    nk = (int64_t)a.cu_k[b + 1] - kbase;
    if (kbase < 0 || nk < 0 || kbase + nk > a.kv_units) {
      bad = true;
      nk = 0;
    }
  }
  return nk;
}

// The end of the keys that the query tile from qt sees (0: none).
__device__ __forceinline__ int64_t tile_end(const PrefillArgs& a, int64_t nk, int32_t nq,
                                            int32_t qt) {
  if (!a.causal) return nk;
  const int32_t last_q = (qt + a.tok < nq ? qt + a.tok : nq) - 1;
  const int64_t end = nk - nq + last_q + 1;  // <= nk
  return end > 0 ? end : 0;
}

// Key ranges of a query tile that sees `units` key tiles: as many as keep a
// range at `cap` key tiles, at most the launch's count. The ranges differ by at
// most one key tile, the longer ones first. A query tile of one range is
// written by its workgroup, with no partial rows and no merge.
__device__ __forceinline__ int32_t tile_ranges(int32_t units, int32_t cap, int32_t splits) {
  if (units <= cap) return 1;
  const int32_t p = (int32_t)((uint32_t)(units + cap - 1) / (uint32_t)cap);
  return p > splits ? splits : p;
}
__device__ __forceinline__ int32_t units_of(int64_t keys) {
  return (int32_t)((keys + kKvTile - 1) / kKvTile);
}

// 16 bytes per lane from base + voff into LDS at lds + 16 * lane. Issued from
// inline assembly: the compiler neither waits for it nor moves LDS accesses
// across it; the waits are explicit (dma_wait before the tile's barrier). M0
// holds the destination; nothing else in this file uses M0 (to the compiler a
// reserved register, which it writes only right before an instruction that
// reads it and refuses in a clobber list).
__device__ __forceinline__ void dma16(const uint8_t* base, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(__builtin_amdgcn_readfirstlane(lds)), "v"(voff), "s"(base)
               : "memory");
}
__device__ __forceinline__ void dma_wait() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

// Keeps values derived from x out of registers held across the loop:
// recomputing them costs a few instructions, holding them costs registers.
__device__ __forceinline__ void opaque(uint32_t& x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void opaque(float& x) { asm volatile("" : "+v"(x)); }

// The largest running maximum (absolute, log2 units) up to which a residue of
// half an fp32 step, 2^-10, leaves the largest weight a bf16 1.
constexpr float kFusedMax = 32768.f;

// Instruction classes of __builtin_amdgcn_sched_group_barrier, and how many
// matrix operands are read ahead of their use.
constexpr int kSchedValu = 0x002, kSchedMfma = 0x008, kSchedDsRead = 0x100, kAhead = 3;

// WAVES: 8 (64 query tokens per workgroup) or 4 (32).
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void prefill_attn_kernel(PrefillArgs a) {
  constexpr int kTok = 8 * WAVES;      // query tokens of the workgroup
  constexpr int kGroups = 8 / WAVES;   // 8-row groups of a tile that a wave loads
  // K tiles 0 and 1, V tiles 0 and 1; after the loop 16 KiB per wave of
  // output rows. A tile is 8 groups of 8 rows, a group 4 blocks of 8 rows x 8
  // 16-byte chunks (1 KiB, one load instruction, whole 128-byte lines). In a
  // K block of row group rg, row r's chunk c lies at 8 (c ^ (rg & 1)) + r; in
  // a V block at 32 (r / 4) + 16 (c / 4) + 4 (r % 4) + c % 4. So the 16 lanes
  // of a score operand read and the 32 of a transposing one fall on distinct
  // banks, and every operand lies at a constant from one lane address: an
  // XOR swizzle of whole rows needs an address register per chunk, which the
  // kernel has not got (it spilled).
  __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * kTileB];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)lds;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int n = lane & 31, hf = lane >> 5;
  int64_t b, hk, kbase, nk;
  int32_t qs, nq, qt, split, ranges;
  if (a.plan) {
    if ((int32_t)blockIdx.x >= ld_const(&a.plan->items)) return;  // uniform
    const PlanItem* it = a.items + blockIdx.x;
    qs = ld_const(&it->qs);
    nq = ld_const(&it->nq);
    kbase = ld_const(&it->kbase);
    nk = ld_const(&it->nk);
    b = ld_const(&it->b);
    hk = ld_const(&it->hk);
    qt = ld_const(&it->qt);
    const uint32_t zp = (uint32_t)ld_const(reinterpret_cast<const int32_t*>(&it->zp));
    split = (int32_t)(zp & 0xffffu);
    ranges = (int32_t)(zp >> 16);
    if (ranges == 0) return;  // uniform: a gap in the list
  } else {
    // Workgroups come in the order of their tile's rank, the sequences' last
    // tiles (which see the most keys, if causal) first, and all (sequence, KV
    // head, range) triples of a rank before the next rank. The dispatcher
    // hands consecutive workgroups to the 8 XCDs in turn, whatever their
    // load, so a triple moves one XCD on with every 8 workgroups: each XCD
    // gets tiles of all ranks of every sequence. (Most grids no larger than
    // the CUs, which run at once, do without: no divisions for it. In a larger
    // one, sequences of 79, 76, 731 and 916 tokens took 28.4 us with the turn
    // and 42 us without.)
    const uint32_t rank = a.rank0 + blockIdx.z;
    uint32_t at = blockIdx.x;
    b = blockIdx.y;
    if (a.turn) {
      const uint32_t triples = gridDim.x * gridDim.y;
      const uint32_t turn =
          triples >= kXcds ? rank % triples : (uint32_t)((uint64_t)rank * triples / kXcds) % triples;
      uint64_t to = (uint64_t)blockIdx.y * gridDim.x + blockIdx.x + turn;
      to = to >= triples ? to - triples : to;
      b = (uint32_t)to / gridDim.x;
      at = (uint32_t)to - (uint32_t)b * gridDim.x;
    }
    hk = a.splits == 1 ? at : at / (uint32_t)a.splits;
    split = (int32_t)(at - (uint32_t)hk * (uint32_t)a.splits);
    bool bad_q, bad_k;
    nq = seq_queries(a, b, qs, bad_q);
    nk = seq_keys(a, b, kbase, bad_k);  // (its loads go out with the queries')
    if (bad_q && tid == 0 && rank == 0 && split == 0 && hk == 0) raise_err(a.err, MKV_DEVERR_TABLE);
    const int64_t q = (int64_t)(a.ranks - 1 - rank) * kTok;  // the workgroup's first query
    if (q >= nq) return;  // uniform
    qt = (int32_t)q;
    if (bad_k && tid == 0 && qt == 0) raise_err(a.err, MKV_DEVERR_TABLE);
    ranges = tile_ranges(units_of(tile_end(a, nk, nq, qt)), a.split_len / kKvTile, a.splits);
    if (split >= ranges) return;  // uniform
  }
  const int64_t hq = (int64_t)a.hkv * kPG;
  const int64_t h = hk * kPG + (wave & 3);      // this wave's query head
  const int32_t q0 = qt + kWTok * (wave >> 2);  // this wave's first query

  const int64_t shift = nk - nq;  // query t sits at position shift + t
  // this workgroup's key range
  int64_t kv_end = tile_end(a, nk, nq, qt), kv_begin = 0;
  if (ranges > 1) {
    const uint32_t units = (uint32_t)units_of(kv_end);
    const uint32_t each = units / (uint32_t)ranges, more = units - each * (uint32_t)ranges;
    const uint32_t z = (uint32_t)split;
    kv_begin = (int64_t)(z * each + (z < more ? z : more)) * kKvTile;
    if (split + 1 < ranges) kv_end = kv_begin + (int64_t)(each + (z < more ? 1 : 0)) * kKvTile;
  }
  // the last key any of this wave's queries sees (-1: it has none), and the
  // last one that all of them see
  int64_t wlast = -1, wfull = -1;
  if (q0 < nq) {
    const int64_t wq = q0 + kWTok < nq ? q0 + kWTok - 1 : nq - 1;
    wlast = a.causal && shift + wq < nk - 1 ? shift + wq : nk - 1;
    wfull = a.causal && shift + q0 < nk - 1 ? shift + q0 : nk - 1;
  }
  // The wave's share of a tile: kGroups groups of 8 rows, all on one page, a
  // block per instruction. Rows past the keys repeat the last key's row
  // (scores are masked, V is zeroed after arrival).
  const int32_t* trow = a.table ? a.table + b * a.tstride : nullptr;
  const uint32_t stride = (uint32_t)a.hkv * kPRow;  // bytes between token rows
  const uint32_t wrow = (uint32_t)wave * (8 * kGroups);
  auto page_of = [&](int64_t kv0) __attribute__((always_inline)) {
    int64_t t = kv0 + wrow;
    if (t >= nk) t = nk - 1;
    return trow ? ld_const(trow + (t >> 4)) : 0;
  };
  auto page_ok = [&](int32_t page) __attribute__((always_inline)) {
    return !trow || (page >= 0 && page < a.kv_units);
  };
  auto issue = [&](int64_t kv0, int32_t page, uint32_t buf) __attribute__((always_inline)) {
    const int64_t t0 = kv0 + wrow;
    if (t0 >= nk || !page_ok(page)) return;
    const int64_t row = trow ? (int64_t)page * 16 + (t0 & 15) : kbase + t0;
    const int64_t off = (row * a.hkv + hk) * kPRow;
    const uint32_t last = (uint32_t)(nk - t0 < 8 * kGroups ? nk - t0 : 8 * kGroups) - 1;
    uint32_t ln = lane;
    opaque(ln);
    const uint32_t dst = lds0 + buf * kTileB + wrow * kPRow;
#pragma unroll
    for (uint32_t g = 0; g < kGroups; ++g) {
      const uint32_t kr = 8 * g + (ln & 7), kc = (ln >> 3) ^ ((wave * kGroups + g) & 1);
      const uint32_t vr = 8 * g + (ln >> 5) * 4 + ((ln >> 2) & 3);
      const uint32_t vc = ((ln >> 4) & 1) * 4 + (ln & 3);
      const uint32_t kvo = (kr < last ? kr : last) * stride + kc * 16;
      const uint32_t vvo = (vr < last ? vr : last) * stride + vc * 16;
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        dma16(a.k + off + u * 128, kvo, dst + g * 4096 + u * 1024);
        dma16(a.v + off + u * 128, vvo, dst + 2 * kTileB + g * 4096 + u * 1024);
      }
    }
  };
  // after the wave's loads of a tile have arrived: zero V rows past the keys,
  // and both planes' rows of a page outside the pool (flagged)
  auto patch = [&](int64_t kv0, int32_t page, uint32_t buf) __attribute__((always_inline)) {
    const int64_t t0 = kv0 + wrow;
    if (t0 + 8 * kGroups <= nk && page_ok(page)) return;  // uniform: the usual case
    const bool wrong = t0 < nk && !page_ok(page);
    const int32_t left = (int32_t)(nk > t0 ? nk - t0 : 0);  // valid rows
    uint32_t ln = lane;
    opaque(ln);
    if (wrong && lane == 0) raise_err(a.err, MKV_DEVERR_PAGE);
    const int32_t vr = (int32_t)((ln >> 5) * 4 + ((ln >> 2) & 3));
    const uint32_t at = lds0 + buf * kTileB + wrow * kPRow + ln * 16;
#pragma unroll
    for (uint32_t u = 0; u < 4 * kGroups; ++u) {
      if (wrong) *(lds_u32x4*)(uintptr_t)(at + u * 1024) = u32x4{0u, 0u, 0u, 0u};
      if (wrong || vr + 8 * (int32_t)(u >> 2) >= left)
        *(lds_u32x4*)(uintptr_t)(at + 2 * kTileB + u * 1024) = u32x4{0u, 0u, 0u, 0u};
    }
  };

  int32_t page = 0, page_next = 0;
  if (kv_end > kv_begin) {
    page = page_of(kv_begin);
    issue(kv_begin, page, 0);
    page_next = page_of(kv_begin + kKvTile);
  }

  // Q^T as the B operand: column n = query q0 + n, dims 16 s + 8 hf .. +7
  bf16x8 qb[16];
  {
    // lanes past the queries repeat the last one (their output is dropped)
    const int64_t t = q0 + n < nq ? q0 + n : nq - 1;
    const uint8_t* row = a.q + ((qs + t) * hq + h) * kPRow + hf * 16;
#pragma unroll
    for (int s = 0; s < 16; ++s)
      qb[s] = __builtin_bit_cast(bf16x8, ld16(row + 32 * s) ^ a.q_sign);
  }
  float m_run = -INFINITY, l_run = 0.f;  // l_run: this half wave's keys only
  bool past_fused = false;  // uniform: some query's maximum is past kFusedMax
  f32x16 o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[j][i] = 0.f;

  // lane addresses in the current K tile (row n, chunk hf) and V tile (token
  // 4 hf + j / 4, dims 16 (g & 1) + 4 (j % 4) ..)
  const int j16 = lane & 15;
  uint32_t ka = lds0 + (uint32_t)((n >> 3) * 4096 + ((hf ^ ((n >> 3) & 1)) * 8 + (n & 7)) * 16);
  uint32_t va = lds0 + 2 * kTileB +
                (uint32_t)(hf * 512 +
                           ((j16 >> 2) * 4 + 2 * ((lane >> 4) & 1) + ((j16 & 3) >> 1)) * 16 +
                           (j16 & 1) * 8);

  uint32_t buf = 0;
  for (int64_t kv0 = kv_begin; kv0 < kv_end; kv0 += kKvTile) {
    dma_wait();
    patch(kv0, page, buf);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kv0 + kKvTile < kv_end) {
      issue(kv0 + kKvTile, page_next, buf ^ 1);
      page = page_next;
      page_next = page_of(kv0 + 2 * kKvTile);
    }
    if (kv0 <= wlast) {
      // S^T of the tile's two 32-key blocks: lane holds query n, keys
      // 32 kb + 8 (r / 4) + 4 hf + r % 4
      f32x16 sq[2];
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 16; ++i) sq[kb][i] = 0.f;
#pragma unroll
      for (int s = 0; s < 16; ++s)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const bf16x8 kk = __builtin_bit_cast(
              bf16x8, *(lds_u32x4*)(uintptr_t)(ka + kb * 32 * kPRow + (s >> 2) * 1024 +
                                               (s & 3) * 256));
          sq[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kk, qb[s], sq[kb], 0, 0, 0);
        }
      // operand reads run kAhead ahead of the matrix instructions
      __builtin_amdgcn_sched_group_barrier(kSchedDsRead, kAhead, 0);
#pragma unroll
      for (int s = 0; s < 32 - kAhead; ++s) {
        __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
        __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(kSchedMfma, kAhead, 0);
      if (kv0 + kKvTile - 1 > wfull) {  // uniform: keys some query does not see
        // the last key this lane's query sees, from the tile's start
        uint32_t ln = lane;
        opaque(ln);
        const int32_t first = (int32_t)(shift + q0 - kv0), end = (int32_t)(nk - 1 - kv0);
        const int32_t at = first + (int32_t)(ln & 31);
        const int32_t rel = (a.causal && at < end ? at : end) - 4 * (int32_t)(ln >> 5);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            sq[kb][r] = 32 * kb + 8 * (r >> 2) + (r & 3) <= rel ? sq[kb][r] : -INFINITY;
      }
      __builtin_amdgcn_s_setprio(0);
      float mx = sq[0][0];
#pragma unroll
      for (int i = 1; i < 32; ++i) mx = fmaxf(mx, sq[i >> 4][i & 15]);
      mx = half_max(mx) * a.scale_log2;
      // O and l are rescaled whenever some query's maximum moved (uniform
      // branch). Letting the maximum lag by a few powers of two skips most of
      // these (5 % of the kernel's time over 4096-token prompts), but then a
      // row's largest probability is no longer exactly 1 and is itself rounded
      // to bf16: the error against float64 grew from 0.00205 to 0.00208.
      if (__builtin_amdgcn_ballot_w64(mx > m_run)) {
        const float m_new = fmaxf(m_run, mx);
        const float ref = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m_run - ref);
        m_run = m_new;
        past_fused = __builtin_amdgcn_ballot_w64(fabsf(ref) > kFusedMax) != 0;
        l_run *= alpha;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[j][i] *= alpha;
      }
      const float m_ref = m_run == -INFINITY ? 0.f : m_run;  // a row with nothing seen yet
      // The exponents below are fused, score * scale - m_ref, while m_ref is the
      // rounded product: the largest score's exponent is that rounding's
      // residue, at most half an fp32 step of m_ref. Up to kFusedMax its
      // weight still rounds to a bf16 1. Past it (a step grows to more than
      // the exponential's range) the products are rounded first, as m_ref was.
      float mul = a.scale_log2;
      if (__builtin_expect(past_fused, 0)) {
#pragma unroll
        for (int i = 0; i < 32; ++i) {
          float x = sq[i >> 4][i & 15] * a.scale_log2;
          opaque(x);  // (or the product and the subtraction are fused again)
          sq[i >> 4][i & 15] = x;
        }
        mul = 1.f;
      }
      // O^T += V^T P^T in 16-key steps: half wave hf takes keys
      // 16 t + 4 hf .. +3 (elements 0-3) and 16 t + 8 + 4 hf .. +3. While the
      // matrix cores run step t, the vector unit makes step t + 1's
      // probabilities; operand reads run kAhead ahead.
      auto probs = [&](int t) __attribute__((always_inline)) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 8 * (t & 1) + 2 * i;
          const float p0 = __builtin_amdgcn_exp2f(fmaf(sq[t >> 1][r], mul, -m_ref));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(sq[t >> 1][r + 1], mul, -m_ref));
          l_run += p0 + p1;
          w[i] = bf16_pack(p0, p1);
        }
        return __builtin_bit_cast(bf16x8, u32x4{w[0], w[1], w[2], w[3]});
      };
      auto v_read = [&](int i) __attribute__((always_inline)) {  // operand i = 8 t + j
        const int t = i >> 3, j = i & 7;
        const uint32_t at = va + 16 * t * kPRow + (j >> 1) * 1024 + (j & 1) * 256;
        const s16x4 lo = lds_read_tr16(at), hi = lds_read_tr16(at + 8 * kPRow);
        return __builtin_bit_cast(bf16x8,
                                  (s16x8){lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w});
      };
      __builtin_amdgcn_s_setprio(1);
      bf16x8 vf[kAhead];
      bf16x8 pp = probs(0), pn = pp;
#pragma unroll
      for (int i = 0; i < kAhead; ++i) vf[i] = v_read(i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < kKvTile / 16; ++t) {
        if (t + 1 < kKvTile / 16) pn = probs(t + 1);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int i = 8 * t + j;
          o[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i % kAhead], pp, o[j], 0, 0, 0);
          if (i + kAhead < 8 * (kKvTile / 16)) vf[i % kAhead] = v_read(i + kAhead);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          __builtin_amdgcn_sched_group_barrier(kSchedMfma, 1, 0);
          __builtin_amdgcn_sched_group_barrier(kSchedDsRead, 2, 0);
          __builtin_amdgcn_sched_group_barrier(kSchedValu, 4, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        pp = pn;
      }
    }
    __builtin_amdgcn_s_setprio(0);
    const uint32_t step = buf ? 0u - kTileB : (uint32_t)kTileB;  // to the other buffer
    ka += step;
    va += step;
    buf ^= 1;
  }

  // Output rows through LDS (the tiles' space, 16 KiB per wave): a lane holds
  // dims 32 j + 8 i + 4 hf .. +3 of query q0 + n; rows of 512 bytes are stored
  // with chunk c at c ^ (row & 15), then each half wave writes whole rows.
  // One range: O / l in bf16 (zeros for a row that saw nothing); several:
  // this range's (max, sum, O) for the merge, 128 dims at a time.
  const float L = half_sum(l_run);
  {
    uint32_t ln = lane;
    opaque(ln);
    n = ln & 31;
    hf = ln >> 5;
  }
  __syncthreads();
  const uint32_t wl = lds0 + (uint32_t)wave * kWTok * kPRow;
  auto rows_out = [&](uint8_t* base, int64_t row_bytes) __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int u = 0; u < kWTok / 2; ++u) {
      const int r = 2 * u + hf;
      const u32x4 x = *(lds_u32x4*)(uintptr_t)(wl + (uint32_t)(r * kPRow + ((n ^ (r & 15)) * 16)));
      if (q0 + r < nq) st16(base + r * row_bytes + n * 16, x);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  const int64_t row0 = ((int64_t)qs + q0) * hq + h;
  if (ranges == 1) {
    const float inv = L > 0.f ? 1.f / L : 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        u32x2v w;
#pragma unroll
        for (int e = 0; e < 2; ++e)
          w[e] = bf16_pack(o[j][4 * i + 2 * e] * inv, o[j][4 * i + 2 * e + 1] * inv);
        *(lds_u32x2*)(uintptr_t)(wl + (uint32_t)(n * kPRow + (((4 * j + i) ^ (n & 15)) * 16) +
                                                 hf * 8)) = L > 0.f ? w : u32x2v{0u, 0u};
      }
    rows_out(a.out + row0 * kPRow, hq * kPRow);
  } else {
    float* part = a.part + (row0 * a.splits + split) * kPD;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int jj = 4 * half + j;
          const f32x4 x = {o[jj][4 * i], o[jj][4 * i + 1], o[jj][4 * i + 2], o[jj][4 * i + 3]};
          *(lds_u32x4*)(uintptr_t)(wl + (uint32_t)(n * kPRow + (((8 * j + 2 * i + hf) ^ (n & 15)) * 16))) =
              __builtin_bit_cast(u32x4, x);
        }
      rows_out(reinterpret_cast<uint8_t*>(part + 128 * half), hq * a.splits * (kPD * 4));
    }
    if (hf == 0 && q0 + n < nq) {
      float* ml = a.ml + ((row0 + n * hq) * a.splits + split) * 2;
      ml[0] = m_run;
      ml[1] = L;
    }
  }
}

// Combines the key ranges of one query token's KV head: one workgroup of 256
// threads per query t < max_seqlen_q of sequence b (grid.y) and KV head
// (grid.z); its four waves take the head's four query heads, a lane four
// dims (16-byte loads of the fp32 partial rows). It writes exactly the rows
// the attention kernel wrote ranges for: the same query offsets and bounds
// decide, so rows of `out` outside every sequence's queries are left alone,
// as with one range; rows of a tile of one range are already there. Each
// output element is summed over the ranges in range
// order, as a thread per element did (one workgroup per query head was 4x
// the workgroups for the same bytes). Up to 8 ranges, every load
// is issued before the first is used (a loop over the ranges waited a round
// trip per range, twice); loads of ranges past the count are not issued, so
// the bytes read are the ranges' own.
template <int N>
__device__ __forceinline__ void merge_ranges(const float2* ml, const float* part, float& L,
                                             float (&O)[4]) {
  float2 x[N];
  f32x4 p[N];
#pragma unroll
  for (int u = 0; u < N; ++u) {
    x[u] = ml[u];
    p[u] = *reinterpret_cast<const f32x4*>(part + (int64_t)u * kPD);
  }
  float M = -INFINITY;
#pragma unroll
  for (int u = 0; u < N; ++u) M = fmaxf(M, x[u].x);
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const float f = x[u].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(x[u].x - M);
#pragma unroll
    for (int e = 0; e < 4; ++e) O[e] += f * p[u][e];
    L += f * x[u].y;
  }
}

__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a) {
  int32_t qs, t, ranges;
  int64_t hk;
  if (a.plan) {
    if ((int32_t)blockIdx.y >= ld_const(&a.plan->cuts)) return;
    const PlanItem* it = a.cut + blockIdx.y;
    qs = ld_const(&it->qs);
    hk = ld_const(&it->hk);
    t = ld_const(&it->qt) + (int32_t)blockIdx.x;
    if (t >= ld_const(&it->nq)) return;
    ranges = ld_const(reinterpret_cast<const int32_t*>(&it->zp)) >> 16;
  } else {
    const int32_t b = blockIdx.y;
    int64_t kbase;
    bool bad;
    const int32_t nq = seq_queries(a, b, qs, bad);
    const int64_t nk = seq_keys(a, b, kbase, bad);
    t = blockIdx.x;
    hk = blockIdx.z;
    if (t >= nq) return;
    ranges = tile_ranges(units_of(tile_end(a, nk, nq, t & -a.tok)), a.split_len / kKvTile,
                         a.splits);
    if (ranges == 1) return;
  }
  const int64_t row = ((int64_t)qs + t) * ((int64_t)a.hkv * kPG) +
                      hk * kPG + (threadIdx.x >> 6);
  const int d = (threadIdx.x & 63) * 4;
  const int64_t at0 = row * a.splits;
  float O[4] = {0.f, 0.f, 0.f, 0.f}, L = 0.f;
  const float2* ml = reinterpret_cast<const float2*>(a.ml) + at0;
  const float* part = a.part + at0 * kPD + d;
  switch (ranges) {
    case 2: merge_ranges<2>(ml, part, L, O); break;
    case 3: merge_ranges<3>(ml, part, L, O); break;
    case 4: merge_ranges<4>(ml, part, L, O); break;
    case 5: merge_ranges<5>(ml, part, L, O); break;
    case 6: merge_ranges<6>(ml, part, L, O); break;
    case 7: merge_ranges<7>(ml, part, L, O); break;
    case 8: merge_ranges<8>(ml, part, L, O); break;
    default: {
      // more than 8 ranges: batches of 8, each loaded at once, under a running
      // maximum (a loop over the ranges, twice, waited a round trip apiece:
      // 40 tokens on 12000 cached ones, 47 ranges, 39.0 -> 36.8 us a step)
      float M = -INFINITY;
      for (int s0 = 0; s0 < ranges; s0 += 8) {
        float2 x[8];
        f32x4 p[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {  // past the last range: it again, unused
          const int at = s0 + u < ranges ? s0 + u : ranges - 1;
          x[u] = ml[at];
          p[u] = *reinterpret_cast<const f32x4*>(part + (int64_t)at * kPD);
        }
        float mb = M;
#pragma unroll
        for (int u = 0; u < 8; ++u) mb = fmaxf(mb, x[u].x);
        const float alpha = M == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(M - mb);
        L *= alpha;
#pragma unroll
        for (int e = 0; e < 4; ++e) O[e] *= alpha;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if (s0 + u >= ranges) break;  // uniform
          const float f = x[u].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(x[u].x - mb);
#pragma unroll
          for (int e = 0; e < 4; ++e) O[e] += f * p[u][e];
          L += f * x[u].y;
        }
        M = mb;
      }
    }
  }
  uint32_t w[2];
#pragma unroll
  for (int e = 0; e < 2; ++e)
    w[e] = (uint32_t)bf16_bits(L > 0.f ? O[2 * e] / L : 0.f) |
           ((uint32_t)bf16_bits(L > 0.f ? O[2 * e + 1] / L : 0.f) << 16);
  *reinterpret_cast<uint2*>(a.out + row * kPRow + d * 2) = uint2{w[0], w[1]};
}

// The plan of a launch: the (query tile, KV head, key range) tasks, longest
// first, and the pairs of several ranges for the merge. A CU runs one
// workgroup at a time, a key tile after the other, so what decides a launch is
// the most key tiles that any CU gets. Key tiles per range:
//   * the fewest with which all tasks run at once, one per CU, if that is not
//     far above the key tiles per CU (1.5 times + 2);
//   * else 1.2 times the key tiles per CU: the longest tasks start first, and
//     the shorter ones fill the CUs as they come free.
// Only the lengths on the device say which; a grid sized on the host cuts all
// sequences as the longest, or not at all. Whole calls, planned and with the
// best such grid of at most one task per CU: 6 prompts of 190 to 2180 tokens
// 50 and 107 us, 4 of 400 to 2280 52 and 113, two chunks of 1.0-1.4k on 3-6k
// tokens 84 and 83 (the rule in prefill_schedule draws the line). Sorted by
// length alone, without the XCDs' grouping, those chunks' attention took 66 us
// instead of 64. The plan takes 7-9 us.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void prefill_plan_kernel(PrefillArgs a, int32_t batch) {
  __shared__ int32_t pre[THREADS];          // the sequences' first tiles
  __shared__ int4 seq[THREADS];             // qs, nq, kbase, nk
  __shared__ int32_t bins[THREADS];         // tasks by their key tiles, then where they start
  __shared__ int32_t red[THREADS / 64][2];
  __shared__ uint16_t tile_units[THREADS];  // of the first tiles, for the search
  __shared__ int2 group[THREADS];           // a sequence's first bin, ranges of its last tile
  __shared__ int32_t cuts, found;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr int kWaves = THREADS / 64;
  // the exclusive prefix of x over the workgroup, and the total
  auto block_scan = [&](int32_t x, int32_t& total) __attribute__((always_inline)) {
    int32_t incl = x;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t o = __shfl_up(incl, d);
      if (lane >= d) incl += o;
    }
    __syncthreads();  // red's earlier readers are done
    if (lane == 63) red[wave][0] = incl;
    __syncthreads();
    int32_t at = incl - x;
    total = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      at += w < wave ? red[w][0] : 0;
      total += red[w][0];
    }
    return at;
  };
  int32_t mine = 0;
  if (tid < batch) {
    int32_t qs;
    int64_t kbase;
    bool bad_q, bad_k;
    const int32_t nq = seq_queries(a, tid, qs, bad_q);
    const int64_t nk = seq_keys(a, tid, kbase, bad_k);
    if (bad_q || (bad_k && nq > 0)) raise_err(a.err, MKV_DEVERR_TABLE);
    seq[tid] = int4{qs, nq, (int32_t)kbase, (int32_t)nk};
    mine = (nq + kQTok - 1) / kQTok;
  }
  bins[tid] = 0;
  if (tid == 0) {
    cuts = 0;
    found = INT_MAX;
  }
  int32_t tiles;
  const int32_t first = block_scan(mine, tiles);
  pre[tid] = first;  // (sequences past the batch repeat the total)
  // offsets that overlap (flagged above: some count is then negative) can
  // hold more tiles than the launch's bound; the ones past it are dropped
  if (tiles > (THREADS * kPlanSlots)) tiles = (THREADS * kPlanSlots);
  __syncthreads();

  int32_t sq[kPlanSlots], unit[kPlanSlots];
  int32_t sum = 0, most = 0;
#pragma unroll
  for (int k = 0; k < kPlanSlots; ++k) {
    const int32_t i = tid + k * THREADS;
    sq[k] = -1;
    unit[k] = 0;
    if (i >= tiles) continue;
    int lo = 0, hi = batch - 1;  // the last sequence that starts at or before tile i
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (pre[mid] <= i) lo = mid; else hi = mid - 1;
    }
    sq[k] = lo;
    const int4 x = seq[lo];
    // (as many as 16 bits hold: past 4 M keys the split needs no more)
    unit[k] = units_of(tile_end(a, x.w, x.y, (i - pre[lo]) * kQTok));
    unit[k] = unit[k] < 65535 ? unit[k] : 65535;
    if (k == 0) tile_units[tid] = (uint16_t)unit[k];
    sum += unit[k];
    most = unit[k] > most ? unit[k] : most;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    sum += __shfl_xor(sum, d);
    const int32_t o = __shfl_xor(most, d);
    most = o > most ? o : most;
  }
  if (lane == 0) {  // (red's earlier readers passed the barrier above)
    red[wave][0] = sum;
    red[wave][1] = most;
  }
  __syncthreads();
  sum = 0;
  most = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    sum += red[w][0];
    most = red[w][1] > most ? red[w][1] : most;
  }
  // key tiles of all tasks (the bounds on tiles and their keys keep it far
  // below the clamp, which offsets that overlap could pass)
  const uint64_t all64 = (uint64_t)(uint32_t)sum * (uint32_t)a.hkv;
  const uint32_t all = all64 < (1u << 30) ? (uint32_t)all64 : 1u << 30, cus = (uint32_t)a.cus;
  // key tiles per range: no less than the key tiles per CU (so the tasks are
  // at most the query tiles and one more per CU) and than the launch's bound
  int32_t least = (int32_t)((all + cus - 1) / cus);
  const int32_t bound = a.splits > 1 ? (most + a.splits - 1) / a.splits : most;
  least = least < bound ? bound : least;
  least = least < kPlanLeast ? kPlanLeast : least;
  int32_t cap = most;
  if (a.splits > 1 && least < most) {
    cap = (int32_t)((all + all / 5 + cus - 1) / cus);
    cap = cap < least ? least : cap > most ? most : cap;
    // kPlanTries candidates, evenly from the least to `far`
    int32_t far = (int32_t)(all * 3 / (2 * cus)) + 2;
    far = far < least ? least : far > most ? most : far;
    if ((int64_t)tiles * a.hkv <= a.cus) {  // (so tile_units holds them all)
      const int32_t step = (far - least + kPlanTries - 1) / kPlanTries;
      for (int c = wave; c < kPlanTries; c += kWaves) {
        int32_t tried = least + c * (step > 1 ? step : 1);
        tried = tried < far && c + 1 < kPlanTries ? tried : far;
        int32_t n = 0;
        for (int i = lane; i < tiles; i += 64) n += tile_ranges(tile_units[i], tried, a.splits);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) n += __shfl_xor(n, d);
        if (lane == 0 && (int64_t)n * a.hkv <= a.cus) atomicMin(&found, tried);
      }
      __syncthreads();
      if (found != INT_MAX) cap = found;
    }
  }
  if (cap < 1) cap = 1;

  // A counting sort of the tasks. All running at once: by (sequence, KV head,
  // range), each XCD taking a contiguous eighth (workgroup w runs on XCD
  // w % 8), so that the query tiles reading the same keys share an L2.
  // Else by key tiles, the longest first.
  const bool once = found != INT_MAX;  // uniform
  if (once) {
    int32_t keys = 0, most_p = 0, unused;
    if (tid < batch && seq[tid].y > 0) {
      const int32_t u = units_of(seq[tid].w);  // its last tile's
      most_p = tile_ranges(u < 65535 ? u : 65535, cap, a.splits);
      keys = most_p * a.hkv;
    }
    const int32_t base = block_scan(keys, unused);
    group[tid] = int2{base, most_p};
    __syncthreads();
  }
  // the task's bin; consecutive tasks of a tile share one unless `once`
  auto bin_of = [&](int k, int32_t p, int32_t hk, int32_t z) __attribute__((always_inline)) {
    if (once) {
      const int2 g = group[sq[k]];
      return g.x + hk * g.y + z;
    }
    const int32_t len = (unit[k] + p - 1) / p;
    return THREADS - 1 - (len < THREADS ? len : THREADS - 1);
  };
#pragma unroll
  for (int k = 0; k < kPlanSlots; ++k) {
    if (sq[k] < 0) continue;
    const int32_t p = tile_ranges(unit[k], cap, a.splits);
    if (once) {
      for (int32_t hk = 0; hk < a.hkv; ++hk)
        for (int32_t z = 0; z < p; ++z) atomicAdd(&bins[bin_of(k, p, hk, z)], 1);
    } else {
      atomicAdd(&bins[bin_of(k, p, 0, 0)], p * a.hkv);
    }
  }
  __syncthreads();
  int32_t total;
  const int32_t start = block_scan(bins[tid], total);
  bins[tid] = start;  // (each thread rewrites the entry that it alone read)
  __syncthreads();
  const int32_t per = (total + kXcds - 1) / kXcds;  // tasks per XCD
  auto place = [&](int32_t at) __attribute__((always_inline)) {
    return once ? at % per * kXcds + at / per : at;
  };
#pragma unroll
  for (int k = 0; k < kPlanSlots; ++k) {
    if (sq[k] < 0) continue;
    const int32_t p = tile_ranges(unit[k], cap, a.splits);
    const int4 x = seq[sq[k]];
    const int32_t qt = (tid + k * THREADS - pre[sq[k]]) * kQTok;
    int32_t at = once ? 0 : atomicAdd(&bins[bin_of(k, p, 0, 0)], p * a.hkv);
    int32_t c = p > 1 ? atomicAdd(&cuts, a.hkv) : 0;
    for (int32_t hk = 0; hk < a.hkv; ++hk) {
      PlanItem it = {x.x, x.y, x.z, x.w, sq[k], hk, qt, (uint32_t)p << 16};
      if (p > 1) {
        if (c < a.max_cuts) a.cut[c] = it;
        ++c;
      }
      for (int32_t z = 0; z < p; ++z) {
        it.zp = ((uint32_t)p << 16) | (uint32_t)z;
        const int32_t to = place(once ? atomicAdd(&bins[bin_of(k, p, hk, z)], 1) : at++);
        if (to < a.max_items) a.items[to] = it;
      }
    }
  }
  if (once && tid < per * kXcds - total) {  // the gaps
    const int32_t to = place(total + tid);
    if (to < a.max_items) a.items[to] = PlanItem{0, 0, 0, 0, 0, 0, 0, 0u};
  }
  if (once) total = per * kXcds;
  __syncthreads();
  if (tid == 0) {
    a.plan->items = total < a.max_items ? total : a.max_items;
    a.plan->cuts = cuts < a.max_cuts ? cuts : a.max_cuts;
  }
}

inline int64_t align16(int64_t n) { return (n + 15) / 16 * 16; }

// Sizes of a planned launch, from what the host knows: query tiles are
// bounded by the longest sequence's times the batch, and by the rows.
struct PlanSizes {
  int64_t tiles, items, cuts, bytes;
};
inline PlanSizes plan_sizes(int64_t num_q, int32_t hkv, int32_t batch, int32_t max_q,
                            int32_t splits, int32_t cus) {
  PlanSizes s;
  const int64_t dense = ((int64_t)max_q + kQTok - 1) / kQTok * batch;
  const int64_t rows = num_q / kQTok + batch;
  s.tiles = dense < rows ? dense : rows;
  // a range is no shorter than the key tiles per CU, so cutting adds at most
  // one task per CU, and at most that many pairs are cut
  const int64_t pairs = s.tiles * hkv;
  s.items = pairs * splits < pairs + cus ? pairs * splits : pairs + cus;
  s.items = (s.items + kXcds - 1) / kXcds * kXcds;  // with the gaps of a list dealt to the XCDs
  s.cuts = splits == 1 ? 0 : pairs < cus ? pairs : cus;
  s.bytes = (int64_t)sizeof(Plan) + (s.items + s.cuts) * (int64_t)sizeof(PlanItem);
  return s;
}

}  // namespace
}  // namespace mkv

using namespace mkv;

extern "C" int64_t mkv_prefill_attention_workspace_bytes(int64_t num_q_tokens, int32_t num_q_heads,
                                                         int32_t splits) {
  if (num_q_tokens < 0 || num_q_heads <= 0 || splits <= 0) return -1;
  if (splits == 1) return 0;
  return num_q_tokens * num_q_heads * splits * (kPD + 2) * 4;
}

namespace {

// Shared by the entry points: `planned` launches take their schedule from the
// plan kernel (split_len unused), others from the grid.
int prefill_attention(const char* fn, bool planned, const void* q, const void* k, const void* v,
                      int64_t kv_units, int32_t num_kv_heads, int32_t num_q_heads,
                      int32_t head_dim, const int32_t* page_table, int64_t table_stride,
                      int32_t table_width, const int32_t* cu_seqlens_q,
                      const int32_t* cu_seqlens_k, const int32_t* seq_lens_k, int32_t batch,
                      int64_t num_q_tokens, int32_t max_seqlen_q, float softmax_scale,
                      int32_t causal, int32_t splits, int32_t split_len, void* out,
                      void* workspace, int64_t workspace_bytes, int32_t* err, void* stream) {
  clear_error();
  MKV_REQUIRE(batch >= 0 && kv_units >= 0 && num_kv_heads > 0 && num_q_heads > 0 &&
                  max_seqlen_q >= 0 && num_q_tokens >= 0 && table_width >= 0 &&
                  table_stride >= table_width,
              MKV_E_INVALID, "%s: bad sizes", fn);
  MKV_REQUIRE(head_dim == kPD, MKV_E_UNSUPPORTED,
              "%s: head_dim %d unsupported (256)", fn,
              head_dim);
  MKV_REQUIRE(num_q_heads == kPG * num_kv_heads, MKV_E_UNSUPPORTED,
              "%s: %d query heads per KV head unsupported (4)", fn,
              num_q_heads / num_kv_heads);
  MKV_REQUIRE(num_q_heads <= 65535 && batch <= 65535, MKV_E_UNSUPPORTED,
              "%s: batch or query heads above 65535", fn);
  MKV_REQUIRE(splits >= 1 &&
                  (splits == 1 || planned || (split_len > 0 && split_len % kKvTile == 0)) &&
                  (int64_t)num_kv_heads * splits <= 65535,
              MKV_E_INVALID, "%s: bad key split (%d x %d)", fn, splits, split_len);
  if (batch == 0 || max_seqlen_q == 0) return MKV_OK;
  const int64_t part = mkv_prefill_attention_workspace_bytes(num_q_tokens, num_q_heads, splits);
  const PlanSizes plan = plan_sizes(num_q_tokens, num_kv_heads, batch, max_seqlen_q, splits, kCus);
  MKV_REQUIRE(!planned || (plan.tiles * num_kv_heads <= kPlanTiles && batch <= kPlanSeqs),
              MKV_E_UNSUPPORTED, "%s: %lld query tiles or %d sequences unsupported (%d, %d)", fn,
              (long long)plan.tiles * num_kv_heads, batch, kPlanTiles, kPlanSeqs);
  const int64_t need = planned ? align16(part) + plan.bytes : part;
  MKV_REQUIRE(need == 0 || (workspace && workspace_bytes >= need && aligned16(workspace)),
              MKV_E_INVALID,
              "%s: workspace of %lld bytes (16-byte aligned) required", fn, (long long)need);
  MKV_REQUIRE(q && k && v && cu_seqlens_q && out && err &&
                  (page_table ? seq_lens_k != nullptr : cu_seqlens_k != nullptr),
              MKV_E_INVALID, "%s: null pointer", fn);
  MKV_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out), MKV_E_ALIGN,
              "%s: q, k, v and out must be 16-byte aligned", fn);
  PrefillArgs a;
  a.q = static_cast<const uint8_t*>(q);
  a.k = static_cast<const uint8_t*>(k);
  a.v = static_cast<const uint8_t*>(v);
  a.table = page_table;
  a.tstride = table_stride;
  a.twidth = table_width;
  a.kv_units = kv_units;
  a.cu_q = cu_seqlens_q;
  a.cu_k = cu_seqlens_k;
  a.lens_k = seq_lens_k;
  a.num_q = num_q_tokens;
  a.max_q = max_seqlen_q;
  a.out = static_cast<uint8_t*>(out);
  a.hkv = num_kv_heads;
  a.causal = causal ? 1 : 0;
  a.cus = device_cus() < kCus ? device_cus() : kCus;
  a.splits = splits;
  a.split_len = splits > 1 && !planned ? split_len : INT_MAX / kKvTile * kKvTile;
  a.part = static_cast<float*>(workspace);
  a.ml = splits > 1 ? a.part + num_q_tokens * num_q_heads * splits * kPD : nullptr;
  a.plan = nullptr;
  a.items = a.cut = nullptr;
  a.max_items = (int32_t)plan.items;
  a.max_cuts = (int32_t)plan.cuts;
  // the kernel scales the row maximum, so its scale is positive: a negative
  // one flips the queries' signs, zero becomes the smallest normal number (the
  // masked scores stay -infinity under it)
  a.scale_log2 = fabsf(softmax_scale) * 1.4426950408889634f;
  if (a.scale_log2 < FLT_MIN) a.scale_log2 = FLT_MIN;
  a.q_sign = softmax_scale < 0.f ? 0x80008000u : 0u;
  a.err = err;
  const hipStream_t st = as_stream(stream);
  a.rank0 = 0;
  if (planned) {
    a.plan = reinterpret_cast<Plan*>(static_cast<uint8_t*>(workspace) + align16(part));
    a.items = reinterpret_cast<PlanItem*>(a.plan + 1);
    a.cut = a.items + plan.items;
    a.tok = kQTok;
    a.ranks = 0;
    a.turn = 0;
    if (batch <= kPlanSmall && plan.tiles <= kPlanSmall * kPlanSlots)
      hipLaunchKernelGGL(prefill_plan_kernel<kPlanSmall>, dim3(1), dim3(kPlanSmall), 0, st, a, batch);
    else
      hipLaunchKernelGGL(prefill_plan_kernel<kPlanThreads>, dim3(1), dim3(kPlanThreads), 0, st, a,
                         batch);
    if (plan.items > 0)
      hipLaunchKernelGGL(prefill_attn_kernel<8>, dim3((unsigned)plan.items), dim3(512), 0, st, a);
    if (plan.cuts > 0)
      hipLaunchKernelGGL(prefill_merge_kernel, dim3(kQTok, (unsigned)plan.cuts), dim3(256), 0, st,
                         a);
    return check_launch(fn);
  }
  // Workgroups of 4 waves (32 query tokens) while the ones with work fit the CUs
  // at once: each SIMD then has one wave to serve, so a key tile takes about
  // half as long. Past that, 8 waves share a tile's loads and overlap one
  // another's softmax with matrix work. The rows bound the tiles that exist
  // (sequences of 79, 76, 731 and 916 tokens in 4 ranges: 464 workgroups of 4
  // waves, at most 240 with work).
  auto ranks = [&](int tok) { return (max_seqlen_q + (int64_t)tok - 1) / tok; };
  const int64_t dense = ranks(kQTok / 2) * batch, rows = num_q_tokens / (kQTok / 2) + batch;
  const bool small = (dense < rows ? dense : rows) * num_kv_heads * splits <= a.cus;
  const int64_t triples = (int64_t)batch * num_kv_heads * splits;
  a.tok = small ? kQTok / 2 : kQTok;
  a.ranks = (uint32_t)ranks(a.tok);
  // Grids no larger than the CUs take their place from the grid, except where
  // that puts each key range on one XCD and the later ranges have few of the
  // tiles (causal prompts with no long prefix: the first range's XCD had 32
  // tiles, the last one's 4). One prompt of 2000 tokens in 8 ranges 40.0 ->
  // 34.5 us; on a long prefix every range has all tiles, and its keys are
  // better read by one XCD (4 x 200 tokens on 3600 in 8 ranges 41.5 us, turned
  // 43.9).
  const bool uneven = splits % kXcds == 0 && causal &&
                      2 * (int64_t)max_seqlen_q >= (int64_t)splits * split_len;
  a.turn = (int64_t)a.ranks * triples > a.cus || uneven;
  constexpr uint32_t kMaxZ = 65535;
  for (a.rank0 = 0; a.rank0 < a.ranks; a.rank0 += kMaxZ) {
    const dim3 grid((unsigned)(num_kv_heads * splits), (unsigned)batch,
                    a.ranks - a.rank0 < kMaxZ ? a.ranks - a.rank0 : kMaxZ);
    if (small)
      hipLaunchKernelGGL(prefill_attn_kernel<4>, grid, dim3(256), 0, st, a);
    else
      hipLaunchKernelGGL(prefill_attn_kernel<8>, grid, dim3(512), 0, st, a);
  }
  if (splits > 1 && num_q_tokens > 0)
    hipLaunchKernelGGL(prefill_merge_kernel,
                       dim3((unsigned)max_seqlen_q, (unsigned)batch, (unsigned)num_kv_heads),
                       dim3(256), 0, st, a);
  return check_launch(fn);
}

}  // namespace

extern "C" int mkv_prefill_attention_bf16(const void* q, const void* k, const void* v,
                                          int64_t kv_units, int32_t num_kv_heads,
                                          int32_t num_q_heads, int32_t head_dim,
                                          const int32_t* page_table, int64_t table_stride,
                                          int32_t table_width, const int32_t* cu_seqlens_q,
                                          const int32_t* cu_seqlens_k, const int32_t* seq_lens_k,
                                          int32_t batch, int64_t num_q_tokens, int32_t max_seqlen_q,
                                          float softmax_scale, int32_t causal, int32_t splits,
                                          int32_t split_len, void* out, void* workspace,
                                          int64_t workspace_bytes, int32_t* err, void* stream) {
  return prefill_attention("mkv_prefill_attention_bf16", false, q, k, v, kv_units, num_kv_heads,
                           num_q_heads, head_dim, page_table, table_stride, table_width,
                           cu_seqlens_q, cu_seqlens_k, seq_lens_k, batch, num_q_tokens,
                           max_seqlen_q, softmax_scale, causal, splits, split_len, out, workspace,
                           workspace_bytes, err, stream);
}

extern "C" int mkv_prefill_attention_planned_bf16(
    const void* q, const void* k, const void* v, int64_t kv_units, int32_t num_kv_heads,
    int32_t num_q_heads, int32_t head_dim, const int32_t* page_table, int64_t table_stride,
    int32_t table_width, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
    const int32_t* seq_lens_k, int32_t batch, int64_t num_q_tokens, int32_t max_seqlen_q,
    float softmax_scale, int32_t causal, int32_t splits, void* out, void* workspace,
    int64_t workspace_bytes, int32_t* err, void* stream) {
  return prefill_attention("mkv_prefill_attention_planned_bf16", true, q, k, v, kv_units,
                           num_kv_heads, num_q_heads, head_dim, page_table, table_stride,
                           table_width, cu_seqlens_q, cu_seqlens_k, seq_lens_k, batch,
                           num_q_tokens, max_seqlen_q, softmax_scale, causal, splits, 0, out,
                           workspace, workspace_bytes, err, stream);
}

extern "C" int64_t mkv_prefill_attention_plan_bytes(int64_t num_q_tokens, int32_t num_q_heads,
                                                    int32_t num_kv_heads, int32_t batch,
                                                    int32_t max_seqlen_q, int32_t splits) {
  if (num_q_tokens < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || batch < 0 ||
      max_seqlen_q < 0 || splits <= 0)
    return -1;
  const PlanSizes s =
      plan_sizes(num_q_tokens, num_kv_heads, batch, max_seqlen_q, splits, kCus);
  if (s.tiles * num_kv_heads > kPlanTiles || batch > kPlanSeqs) return -1;
  return align16(mkv_prefill_attention_workspace_bytes(num_q_tokens, num_q_heads, splits)) +
         s.bytes;
}
