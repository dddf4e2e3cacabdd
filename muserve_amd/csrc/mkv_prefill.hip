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
// registers) the LDS reads and the passes of P bounded it. On MI355X, 8 x 4096
// causal tokens of one KV head: 560 -> 380 us (0.49 -> 0.72 PFLOP/s of the
// visible pairs); two 1.3k-token chunks on 3-5k-token prefixes with their
// append and merge: 156 -> 80 us. While a CU is busy its matrix cores are so
// 60 % of the time.
#include <float.h>
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
constexpr int kCus = 256;          // MI355X; LDS holds one workgroup per CU

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
  int32_t splits;        // key ranges per (query tile, KV head); 1: output directly
  int32_t split_len;     // keys per range (a multiple of the KV tile)
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

// 16 bytes per lane from base + voff into LDS at lds + 16 * lane. Issued from
// inline assembly: the compiler neither waits for it nor moves LDS accesses
// across it; the waits are explicit (dma_wait before the tile's barrier). M0
// holds the destination; nothing else in this file uses M0.
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
  const int64_t b = blockIdx.y, hk = blockIdx.z / a.splits, split = blockIdx.z % a.splits;
  const int32_t qs = a.cu_q[b];
  const int32_t nq_raw = a.cu_q[b + 1] - qs;
  // query offsets outside the buffer, or more queries than the launch covers:
  // flagged; nothing of the sequence (or nothing past the bound) is touched
  const bool q_ok = qs >= 0 && nq_raw >= 0 && (int64_t)qs + nq_raw <= a.num_q;
  if ((!q_ok || nq_raw > a.max_q) && tid == 0 && blockIdx.x == 0 && blockIdx.z == 0)
    raise_err(a.err, MKV_DEVERR_TABLE);
  const int32_t nq = q_ok ? (nq_raw < a.max_q ? nq_raw : a.max_q) : 0;
  // the workgroup's first query; a causal sequence's last tiles see the most
  // keys and start first
  const int32_t qt = (int32_t)(gridDim.x - 1 - blockIdx.x) * kTok;
  if (qt >= nq) return;  // uniform
  const int64_t hq = (int64_t)a.hkv * kPG;
  const int64_t h = hk * kPG + (wave & 3);      // this wave's query head
  const int32_t q0 = qt + kWTok * (wave >> 2);  // this wave's first query

  // the sequence's keys: a length checked against what the table (or the
  // buffer) holds; a bad one is flagged and clamped
  int64_t nk, kbase = 0;
  bool bad = false;
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
  if (bad && tid == 0 && qt == 0) raise_err(a.err, MKV_DEVERR_TABLE);
  const int64_t shift = nk - nq;  // query t sits at position shift + t
  const int32_t last_q = (qt + kTok < nq ? qt + kTok : nq) - 1;  // the workgroup's last
  int64_t kv_end = a.causal ? shift + last_q + 1 : nk;
  if (kv_end > nk) kv_end = nk;
  // this workgroup's key range (the whole range with one split); the last
  // range runs to the sequence's end, so a split_len * splits below the real
  // key count never drops keys
  const int64_t kv_begin = split * (int64_t)a.split_len;
  if (split + 1 < a.splits && kv_begin + a.split_len < kv_end) kv_end = kv_begin + a.split_len;
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
        const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[j][i] *= alpha;
      }
      const float m_ref = m_run == -INFINITY ? 0.f : m_run;  // a row with nothing seen yet
      // O^T += V^T P^T in 16-key steps: half wave hf takes keys
      // 16 t + 4 hf .. +3 (elements 0-3) and 16 t + 8 + 4 hf .. +3. While the
      // matrix cores run step t, the vector unit makes step t + 1's
      // probabilities; operand reads run kAhead ahead.
      auto probs = [&](int t) __attribute__((always_inline)) {
        uint32_t w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 8 * (t & 1) + 2 * i;
          const float p0 = __builtin_amdgcn_exp2f(fmaf(sq[t >> 1][r], a.scale_log2, -m_ref));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(sq[t >> 1][r + 1], a.scale_log2, -m_ref));
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
  if (a.splits == 1) {
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
// as with one range. Each output element is summed over the ranges in range
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
  const int32_t b = blockIdx.y;
  const int32_t qs = a.cu_q[b];
  const int32_t nq_raw = a.cu_q[b + 1] - qs;
  const bool q_ok = qs >= 0 && nq_raw >= 0 && (int64_t)qs + nq_raw <= a.num_q;
  const int32_t nq = q_ok ? (nq_raw < a.max_q ? nq_raw : a.max_q) : 0;
  const int32_t t = blockIdx.x;
  if (t >= nq) return;
  const int64_t row = ((int64_t)qs + t) * ((int64_t)a.hkv * kPG) +
                      (int64_t)blockIdx.z * kPG + (threadIdx.x >> 6);
  const int d = (threadIdx.x & 63) * 4;
  const int64_t at0 = row * a.splits;
  float O[4] = {0.f, 0.f, 0.f, 0.f}, L = 0.f;
  const float2* ml = reinterpret_cast<const float2*>(a.ml) + at0;
  const float* part = a.part + at0 * kPD + d;
  switch (a.splits) {
    case 2: merge_ranges<2>(ml, part, L, O); break;
    case 3: merge_ranges<3>(ml, part, L, O); break;
    case 4: merge_ranges<4>(ml, part, L, O); break;
    case 5: merge_ranges<5>(ml, part, L, O); break;
    case 6: merge_ranges<6>(ml, part, L, O); break;
    case 7: merge_ranges<7>(ml, part, L, O); break;
    case 8: merge_ranges<8>(ml, part, L, O); break;
    default: {  // more than 8 ranges
      float M = -INFINITY;
      for (int sp = 0; sp < a.splits; ++sp) M = fmaxf(M, a.ml[(at0 + sp) * 2]);
      for (int sp = 0; sp < a.splits; ++sp) {
        const float m = a.ml[(at0 + sp) * 2];
        const float f = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
        const f32x4 p = *reinterpret_cast<const f32x4*>(a.part + (at0 + sp) * kPD + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) O[e] += f * p[e];
        L += f * a.ml[(at0 + sp) * 2 + 1];
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

}  // namespace
}  // namespace mkv

using namespace mkv;

extern "C" int64_t mkv_prefill_attention_workspace_bytes(int64_t num_q_tokens, int32_t num_q_heads,
                                                         int32_t splits) {
  if (num_q_tokens < 0 || num_q_heads <= 0 || splits <= 0) return -1;
  if (splits == 1) return 0;
  return num_q_tokens * num_q_heads * splits * (kPD + 2) * 4;
}

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
  clear_error();
  MKV_REQUIRE(batch >= 0 && kv_units >= 0 && num_kv_heads > 0 && num_q_heads > 0 &&
                  max_seqlen_q >= 0 && num_q_tokens >= 0 && table_width >= 0 &&
                  table_stride >= table_width,
              MKV_E_INVALID, "mkv_prefill_attention_bf16: bad sizes");
  MKV_REQUIRE(head_dim == kPD, MKV_E_UNSUPPORTED,
              "mkv_prefill_attention_bf16: head_dim %d unsupported (256)", head_dim);
  MKV_REQUIRE(num_q_heads == kPG * num_kv_heads, MKV_E_UNSUPPORTED,
              "mkv_prefill_attention_bf16: %d query heads per KV head unsupported (4)",
              num_q_heads / num_kv_heads);
  MKV_REQUIRE(num_q_heads <= 65535 && batch <= 65535, MKV_E_UNSUPPORTED,
              "mkv_prefill_attention_bf16: batch or query heads above 65535");
  MKV_REQUIRE(splits >= 1 && (splits == 1 || (split_len > 0 && split_len % kKvTile == 0)) &&
                  (int64_t)num_kv_heads * splits <= 65535,
              MKV_E_INVALID, "mkv_prefill_attention_bf16: bad key split (%d x %d)", splits,
              split_len);
  if (batch == 0 || max_seqlen_q == 0) return MKV_OK;
  const int64_t need = mkv_prefill_attention_workspace_bytes(num_q_tokens, num_q_heads, splits);
  MKV_REQUIRE(splits == 1 || (workspace && workspace_bytes >= need && aligned16(workspace)),
              MKV_E_INVALID,
              "mkv_prefill_attention_bf16: workspace of %lld bytes (16-byte aligned) required",
              (long long)need);
  MKV_REQUIRE(q && k && v && cu_seqlens_q && out && err &&
                  (page_table ? seq_lens_k != nullptr : cu_seqlens_k != nullptr),
              MKV_E_INVALID, "mkv_prefill_attention_bf16: null pointer");
  MKV_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out), MKV_E_ALIGN,
              "mkv_prefill_attention_bf16: q, k, v and out must be 16-byte aligned");
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
  a.splits = splits;
  a.split_len = splits > 1 ? split_len : 0;
  a.part = static_cast<float*>(workspace);
  a.ml = splits > 1 ? a.part + num_q_tokens * num_q_heads * splits * kPD : nullptr;
  // the kernel scales the row maximum, so its scale is positive: a negative
  // one flips the queries' signs, zero becomes the smallest normal number (the
  // masked scores stay -infinity under it)
  a.scale_log2 = fabsf(softmax_scale) * 1.4426950408889634f;
  if (a.scale_log2 < FLT_MIN) a.scale_log2 = FLT_MIN;
  a.q_sign = softmax_scale < 0.f ? 0x80008000u : 0u;
  a.err = err;
  // Workgroups of 4 waves (32 query tokens) while they all fit the CUs at once:
  // each SIMD then has one wave to serve, so a key tile takes about half as
  // long. Past that, 8 waves share a tile's loads and overlap one another's
  // softmax with matrix work.
  auto tiles = [&](int tok) {
    return dim3((unsigned)((max_seqlen_q + (int64_t)tok - 1) / tok), (unsigned)batch,
                (unsigned)(num_kv_heads * splits));
  };
  const dim3 small = tiles(kQTok / 2);
  if ((int64_t)small.x * small.y * small.z <= kCus)
    hipLaunchKernelGGL(prefill_attn_kernel<4>, small, dim3(256), 0, as_stream(stream), a);
  else
    hipLaunchKernelGGL(prefill_attn_kernel<8>, tiles(kQTok), dim3(512), 0, as_stream(stream), a);
  if (splits > 1 && num_q_tokens > 0)
    hipLaunchKernelGGL(prefill_merge_kernel,
                       dim3((unsigned)max_seqlen_q, (unsigned)batch, (unsigned)num_kv_heads),
                       dim3(256), 0, as_stream(stream), a);
  return check_launch("mkv_prefill_attention_bf16");
}
