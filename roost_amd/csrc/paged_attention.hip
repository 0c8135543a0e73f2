// PagedAttention (ROOST_OP_PAGED_ATTENTION) for gfx950: paged GQA decode and varlen causal chunked prefill over a
// block-tabled KV cache, behind the C1 workspace / plan / run entry points.
//
// Semantics are CpuOps.PagedAttention (reference: src/Starlings.Roost.Ops/CpuOps.cs:198-298): sequence b has
// n = q_indptr[b+1]-q_indptr[b] queries and kvLen = (pages-1)*page_size + kv_last_page_len[b] keys; query i sits at
// key position kvLen-n+i and (causal) sees keys j <= that position; a decode query sees every key; query head h reads
// KV head h / (q_heads / kv_heads); score = q.k * scale (scale 0 -> 1/sqrt(head_dim)); softmax; sum p*v; a query that
// sees no key outputs zeros. The entry-point contract is the reference's (kernels/src/paged_attention.cu:78-349):
// workspace() and plan() read the host batch tables, run() never does and refuses with NOT_PLANNED until plan() has
// written a plan record for this batch shape. The optional lse output is the base-2 log-sum-exp of the scaled scores,
// log2(sum_j 2^(s_j * log2 e)), which is the convention of the FlashInfer kernels the reference wraps.
//
// Decode (mode DECODE) -- HBM bound (DecodeMfmaKernel in bf16, DecodeF32Kernel, DecodeMergeKernel):
//   * plan() deals the batch's 16-token groups out evenly to one range per resident workgroup slot and cuts sequences
//     at range boundaries (so the variant is DETERMINISTIC but not BATCH_INVARIANT); a workgroup serves the KV heads
//     of its range, its wavefronts take alternate groups;
//   * bf16: a wavefront serves all the query heads of a KV head (up to 16), each K/V byte requested once; K and V rows are
//     loaded branch-free into one register buffer each, the next group's K in flight from the moment the scores have
//     read this one's; q.k on v_mfma_f32_16x16x32_bf16 (tokens on M, heads on N), P.V on v_mfma_f32_16x16x16_bf16 with P
//     rounded to bf16 and fp32 accumulation;
//   * f32: groups of 4 heads, a register double buffer, q.k as VALU products reduce-scattered across the lanes of a row;
//   * the wavefronts merge through LDS; a sequence cut into pieces writes fp32 partials (o, m, l) that
//     DecodeMergeKernel combines in key order.
// Prefill (mode PREFILL) -- MFMA bound (PrefillTileKernel + PrefillMergeKernel for page sizes that are powers of two
// and multiples of 16; PrefillKernel otherwise):
//   * one workgroup = 64 query tokens x the 4 query heads of one (virtual) KV head, 8 wavefronts; 64-key K and V
//     tiles are copied from the paged cache straight into LDS (global_load_lds), double-buffered;
//   * S^T = K Q^T and O^T = V^T P^T on v_mfma_f32_32x32x16_bf16 with fp32 accumulation; the softmax statistics of a
//     query live in one lane pair; P is rounded to bf16 before the P.V product (as FlashAttention-2 does);
//   * plan() cuts items longer than the average CU load into pieces (bf16 partials merged in key order) and orders the
//     work longest-first so the ragged causal tail does not set the makespan;
//   * single-token sequences of a prefill call run on the decode kernels, in one launch with the tile kernel when plan()
//     finds that cheaper (ChooseOverlap); an f32 prefill runs every query token as a row of
//     the f32 decode kernel.
// Output gate (roost_amd_paged_attention_gated_run): Qwen3.5's SigmoidMul on the attention output, applied by every
// kernel that stores an output element (decode, both prefill kernels, both merges) to the element already rounded to
// the output type, with the SigmoidMul op's arithmetic (GateMul in common.h), so it equals run() then SigmoidMul.

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <queue>
#include <type_traits>
#include <vector>

#include "common.h"

namespace {

using namespace roost_dev;

constexpr uint32_t kGroup = 4;                  // query heads per KV head (Qwen3.5: 8 over 2)
constexpr uint32_t kDecodeWgsPerCu = 2;        // decode workgroups resident per CU
constexpr int kMixedDecodeWaves = 8;           // wavefronts of a decode workgroup in the one-launch mixed step
constexpr int kDecodeRing = 2;                  // register ring depth: groups in flight per wavefront = ring - 1
constexpr uint32_t kMaxMergeSplits = 1024;      // partials one sequence may be split into
constexpr uint32_t kPrefillTileQ = 32;          // query tokens per workgroup of the general-page-size prefill
constexpr uint32_t kPrefillTileK = 64;          // keys per LDS tile
constexpr uint32_t kPfTokens = 64;              // query tokens per workgroup of the prefill for page sizes % 16 == 0
constexpr uint32_t kPfRows = kPfTokens * kGroup;  // query rows (token, head) of one such workgroup
// The 12-wavefront form of the tile kernel: 96 query tokens, so that each SIMD holds three wavefronts (153 of 168
// registers, no spills) and one's softmax has two others' multiplies to run beside, and each K/V tile is copied for
// half as many more queries. Four prompts around 3,800 tokens x 32 heads over 8, head dim 128: 533 -> 492 us. Head dim 64 is
// slower with it (83 -> 90 us); head dim 256 does not fit three wavefronts.
constexpr uint32_t kPfWideTokens = 96;
constexpr uint32_t kPfWideDim = 128;            // the head dim it is built for
// A 96-token tile's time over a 64-token one's, and what a piece of a cut item adds (partial rows, merge) in 64-token tiles:
// plan() takes the 12-wavefront form when its dispatch ends earlier in these terms. Ratios of the two dispatches and times
// (8 wavefronts, 12; us; head dim 128), no item cut: 4 prompts around 3,800 x 32 heads 1.45, 533 / 492; 8 ragged prompts to
// 4,000 1.45, 319 / 300; 7 of 3,500 x 16 heads 1.41, 349 / 330; 8 of 1,900 with a window of 1,023 1.38, 132 / 136. Cut: 5
// prompts to 2,800 x 8 heads 1.43 in 338 / 460 pieces, 87 / 95; 2 chunks of 1,100 in a window of 511 1.71 in 0 / 200, 36 / 42.
constexpr double kPfWideTileCost = 1.39;
constexpr double kPfCutPieceTiles = 0.02;
constexpr uint32_t kPfMinSplitTiles = 8;        // load balance cuts no piece below this many 64-key tiles
constexpr uint32_t kAlign = 256;
constexpr uint32_t kPlanMagic = 0x41504752;     // "RGPA"
constexpr float kLog2e = 1.4426950408889634f;

// Logit soft capping (CpuOps.cs:276: s -> cap tanh(s / cap) after the scale), applied to scores in log2 units:
// y -> capl tanh(y / capl) with capl = |cap| log2(e), through tanh(u) = 1 - 2 / (1 + e^(2u)) = 1 - 2 / (1 + 2^(y k)),
// k = 2 log2(e) / capl. capl = 0 turns it off. Masked scores are set to -inf after capping.
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

// Round-to-nearest-even pack of two floats (v_cvt_pk_bf16_f32): the softmax weights, which lie in [0, 256], and the
// tile kernel's outputs (the same rounding as PackBf16 for every finite value; only a NaN, which finite inputs never
// produce here, may keep another NaN pattern than 0x7FC0).
__device__ __forceinline__ uint32_t PackRne(float lo, float hi) {
  const bf16x2_t v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, v);
}

struct SoftCap {
  float capl;
  float k;
};
__device__ __forceinline__ float Capped(float y, SoftCap c) {
  return c.capl - 2.0f * c.capl * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(y * c.k));
}

// A decode row is one query token: the last token of its sequence (q_back 0: decode calls and the single-token
// sequences of a prefill call) or, in an f32 prefill, any token, q_back tokens before the sequence's last.
struct DecodeWork {
  int32_t seq;
  int32_t token_begin;  // first key of this piece (a multiple of 16)
  int32_t token_end;    // one past its last key
  int32_t slot;         // partial slot, or -1 when the piece is the whole row (written as the final row)
  int32_t q_back;       // the row's query token sits q_back tokens before its sequence's last token
};
struct DecodeMerge {
  int32_t seq;
  int32_t first;  // first partial slot; the row's pieces own slots first .. first + count - 1 in key order
  int32_t count;
  int32_t q_back;
};
// A prefill work item: query tokens q0 .. q0 + rows - 1 of sequence seq (all kGroup query heads of one KV head)
// against keys [kbeg, kend). slot >= 0 marks one piece of a split key range: it writes partials (its output divided
// by its own sum, in bf16 in the plan's first slots and in fp32 in the rest, and its fp32 running max and sum) that
// PrefillMergeKernel combines; slot -1 writes the final rows.
struct PrefillWork {
  int32_t seq;
  int32_t q0;
  int32_t kv_head;
  int32_t rows;
  int32_t kbeg;
  int32_t kend;
  int32_t slot;
  int32_t ends;  // kPieceFirst | kPieceLast: whether this piece starts / ends its item's key range
};
// The kernels re-derive an item's outer key bounds from the device's kv_last_page_len (plan() may have assumed full
// last pages when kv_last_page_len_host was NULL, or the lengths may have changed since): the first piece of an item
// starts at the device's first visible key and the last piece ends at the device's last one.
constexpr int32_t kPieceFirst = 1;
constexpr int32_t kPieceLast = 2;
struct PrefillMerge {
  int32_t seq;
  int32_t q0;
  int32_t kv_head;
  int32_t rows;
  int32_t first;  // the pieces own partial slots first .. first + count - 1
  int32_t count;
  int32_t reserved[2];
};

// What plan() leaves for run(); trivially copyable, read back with memcpy.
struct PlanRecord {
  uint32_t magic;
  uint32_t mode;
  uint32_t batch;
  uint32_t tokens;
  uint32_t page_size;
  uint32_t kv_layout;
  uint32_t head_dim;
  uint32_t kv_heads;
  int32_t window;        // WindowOf(params): the pieces start at the window
  uint32_t merges_two;   // prefill: the leading merge entries of exactly two pieces
  uint32_t overlap;      // prefill with single-token sequences: tile and decode kernels run side by side
  uint32_t dec_heads_per_wg;  // (virtual) KV heads per decode workgroup
  uint64_t pages;        // kv_indptr_host[batch]
  uint64_t work_items;   // decode pieces or prefill tiles
  uint64_t ranges;       // decode: workgroup ranges over the pieces
  uint64_t merges;       // decode: sequences whose pieces are merged
  uint64_t range_offset; // byte offsets in the int region
  uint64_t merge_offset;
  uint64_t counter_offset;
  uint64_t splits;       // decode partial slots
  uint64_t int_bytes;    // [work items | seq splits]
  uint64_t float_offset; // partials start here
  uint64_t float_bytes;
  // Single-token sequences of a prefill call run as decode: their pieces, ranges, merges and partials.
  uint64_t dec_items, dec_ranges, dec_merges, dec_splits;
  uint64_t dec_item_offset, dec_range_offset, dec_merge_offset, dec_float_offset;
  uint64_t splits_bf16;  // prefill: the leading partial slots, whose rows are bf16
  uint32_t q_heads;      // the partials' row stride and, in a prefill, the items' heads
  uint32_t dtype;        // PlanDtype(params): the kernels the tables were made for
  uint64_t item_tokens;  // prefill: query tokens per work item (kPfTokens or kPfWideTokens)
};

struct Layout {
  uint64_t work_items = 0;
  uint64_t ranges = 0;
  uint64_t merges = 0;
  uint64_t merges_two = 0;  // prefill: leading merge entries of two pieces
  uint32_t item_tokens = kPfTokens;  // prefill: query tokens per work item
  uint64_t splits_bf16 = 0;          // prefill: leading partial slots in bf16
  uint32_t overlap = 0;     // prefill: tile pieces and decode ranges side by side in one launch (ChooseOverlap)
  uint64_t range_offset = 0;
  uint64_t merge_offset = 0;
  uint64_t counter_offset = 0;
  uint64_t splits = 0;
  uint64_t int_bytes = 0;
  uint64_t float_offset = 0;
  uint64_t float_bytes = 0;
  uint64_t total = 0;
  // Decode region (decode calls: the whole plan; prefill calls: the single-token sequences).
  uint32_t dec_heads_per_wg = 1;
  uint64_t dec_items = 0, dec_ranges = 0, dec_merges = 0, dec_splits = 0;
  uint64_t dec_item_offset = 0, dec_range_offset = 0, dec_merge_offset = 0, dec_float_offset = 0;
};

// ---- Admission ---------------------------------------------------------------------------------------------------

// Query heads per KV head the kernels serve: 4, 8, 16 and 32 (the reference builds 4 only). The prefill and f32 kernels
// take larger groups as 2, 4 and 8 groups of kGroup = 4 that read the same KV rows.
bool GroupBuilt(uint32_t g) { return g == 4 || g == 8 || g == 16 || g == 32; }
// Groups of kGroup query heads ("virtual" KV heads) and the log2 of how many of them share one real KV head.
uint32_t VirtualHeads(const RoostPagedAttentionParams& p) { return p.q_heads / kGroup; }
uint32_t HeadShift(const RoostPagedAttentionParams& p) {
  return static_cast<uint32_t>(__builtin_ctz(p.q_heads / (p.kv_heads * kGroup)));
}

// Query heads one wavefront of the decode kernels serves: 4 in f32, the whole group of 4, 8 or 16 in bf16 (groups of 32
// as two of 16), so that a K/V row is requested once for up to 16 heads.
uint32_t DecodeGroupOf(const RoostPagedAttentionParams& p) {
  return p.q.dtype == ROOST_DTYPE_F32 ? kGroup : std::min(p.q_heads / p.kv_heads, 16u);
}
// Groups of DecodeGroupOf query heads.
uint32_t DecodeHeads(const RoostPagedAttentionParams& p) { return p.q_heads / DecodeGroupOf(p); }

// Shapes with a kernel here, per mode: head dims 64/128/256 decode; prefill on the tile kernel at 64, 128 and 256
// (64 and 128 need page sizes that are powers of two and multiples of 16), on the general kernel at 256.
bool PrefillShapeBuilt(const RoostPagedAttentionParams& p) {
  // f32 prefills run on the decode kernels (any page size); bf16 ones on the tile kernels.
  if (p.head_dim == 256 || p.q.dtype == ROOST_DTYPE_F32) return true;
  return (p.head_dim == 128 || p.head_dim == 64) && p.page_size % 16 == 0 && roost::IsPow2(p.page_size);
}

// The host batch tables, as workspace() and plan() read them: q_indptr over [0, tokens], both indptrs
// non-decreasing, last-page lengths in [1, page_size] for sequences that have pages, and (CpuOps.cs:326-329) a causal
// prefill sequence holding at least as many keys as queries.
void AdmitHostTables(const RoostPagedAttentionParams& p, roost::Gate& gate) {
  gate.Expect(p.q_indptr_host != nullptr && p.kv_indptr_host != nullptr, ROOST_STATUS_INVALID_ARGUMENT,
              "plan and workspace read q_indptr_host and kv_indptr_host; %s is NULL",
              p.q_indptr_host == nullptr ? "q_indptr_host" : "kv_indptr_host");
  if (!gate.ok()) return;
  const int32_t* qi = p.q_indptr_host;
  const int32_t* ki = p.kv_indptr_host;
  gate.Expect(qi[0] == 0 && qi[p.batch] == static_cast<int32_t>(p.tokens), ROOST_STATUS_INVALID_ARGUMENT,
              "q_indptr_host runs from %d to %d; it must run from 0 to tokens = %u", qi[0], qi[p.batch], p.tokens)
      .Expect(ki[0] == 0, ROOST_STATUS_INVALID_ARGUMENT, "kv_indptr_host[0] = %d, must be 0", ki[0]);
  for (uint32_t b = 0; b < p.batch && gate.ok(); ++b) {
    gate.Expect(qi[b + 1] >= qi[b] && ki[b + 1] >= ki[b], ROOST_STATUS_INVALID_ARGUMENT,
                "sequence %u: q_indptr_host or kv_indptr_host goes backwards", b);
    const int64_t pages = ki[b + 1] - ki[b];
    if (p.kv_last_page_len_host == nullptr || pages <= 0 || !gate.ok()) continue;
    const int32_t last = p.kv_last_page_len_host[b];
    gate.Expect(last >= 1 && last <= static_cast<int32_t>(p.page_size), ROOST_STATUS_INVALID_ARGUMENT,
                "sequence %u: kv_last_page_len_host = %d outside 1..page_size (%u)", b, last, p.page_size);
    if (p.mode == ROOST_ATTENTION_PREFILL && p.causal) {
      const int64_t keys = (pages - 1) * p.page_size + last;
      gate.Expect(keys >= qi[b + 1] - qi[b], ROOST_STATUS_INVALID_ARGUMENT,
                  "sequence %u: causal prefill of %d queries over only %lld keys", b, qi[b + 1] - qi[b],
                  static_cast<long long>(keys));
    }
  }
}

// The call's rules (the reference refuses a subset of these shapes: kernels/src/paged_attention.cu:78-130). `for_run`
// checks the device spans; otherwise (workspace, plan) the host tables.
RoostStatus Admit(const RoostPagedAttentionParams& p, bool for_run) {
  roost::Gate gate("paged_attention");
  const bool prefill = p.mode == ROOST_ATTENTION_PREFILL;
  gate.Expect(p.mode == ROOST_ATTENTION_DECODE || prefill, ROOST_STATUS_INVALID_ARGUMENT,
              "mode = %u is neither DECODE nor PREFILL", p.mode)
      .Expect(p.head_dim == 64 || p.head_dim == 128 || p.head_dim == 256, ROOST_STATUS_UNSUPPORTED,
              "head_dim = %u has no kernel here (built: 64, 128, 256)", p.head_dim)
      .Expect(!prefill || PrefillShapeBuilt(p), ROOST_STATUS_UNSUPPORTED,
              "bf16 prefill at head_dim = %u, page_size = %u has no kernel here (built: 256 at any page size; 64 and 128 "
              "at power-of-two page sizes that are multiples of 16)", p.head_dim, p.page_size)
      .Expect(p.kv_heads > 0 && p.q_heads % p.kv_heads == 0 && GroupBuilt(p.q_heads / std::max(p.kv_heads, 1u)),
              ROOST_STATUS_UNSUPPORTED, "q_heads = %u over kv_heads = %u: built for groups of 4, 8, 16 or 32 query "
              "heads per KV head", p.q_heads, p.kv_heads)
      // CpuOps.cs:180-186: a window of 0 keys is an error; -1 (any negative value) means no window.
      .Expect(p.window_left != 0, ROOST_STATUS_INVALID_ARGUMENT, "window_left = 0 is not a window; pass -1 for none")
      .Expect(std::isfinite(p.logits_soft_cap), ROOST_STATUS_INVALID_ARGUMENT,
              "logits_soft_cap = %g; a finite cap (0 for none) is required", p.logits_soft_cap)
      .Expect(p.kv_layout == ROOST_LAYOUT_PAGED_NHD || p.kv_layout == ROOST_LAYOUT_PAGED_HND,
              ROOST_STATUS_INVALID_ARGUMENT, "kv_layout = %u is not a paged layout (NHD or HND)", p.kv_layout)
      .Expect(p.batch > 0 && p.page_size > 0, ROOST_STATUS_INVALID_ARGUMENT,
              "batch = %u, page_size = %u: both must be positive", p.batch, p.page_size)
      .Expect(prefill || p.tokens == p.batch, ROOST_STATUS_INVALID_ARGUMENT,
              "decode of %u tokens over %u sequences; decode is one query token per sequence", p.tokens, p.batch);
  ROOST_GATE_RETURN(gate);
  if (!for_run) {
    AdmitHostTables(p, gate);
    return gate.status();
  }
  const uint32_t dt = p.q.dtype;
  gate.Expect(dt == ROOST_DTYPE_BF16 || dt == ROOST_DTYPE_F32, ROOST_STATUS_INVALID_ARGUMENT,
              "q is %s; attention reads bf16 or f32", roost::Describe(dt).name);
  ROOST_GATE_RETURN(gate);
  const uint64_t q_elems = static_cast<uint64_t>(p.tokens) * p.q_heads * p.head_dim;
  const uint64_t page_elems = static_cast<uint64_t>(p.page_size) * p.kv_heads * p.head_dim;
  gate.Tensor("q", p.q, dt, q_elems)
      .Tensor("output", p.output, dt, q_elems)
      .OptionalTensor("lse", p.lse, ROOST_DTYPE_F32, static_cast<uint64_t>(p.tokens) * p.q_heads)
      .Tensor("k_cache", p.k_cache, dt, page_elems)
      .Tensor("v_cache", p.v_cache, dt, page_elems)
      .Tensor("q_indptr", p.q_indptr, ROOST_DTYPE_I32, p.batch + 1ull)
      .Tensor("kv_indptr", p.kv_indptr, ROOST_DTYPE_I32, p.batch + 1ull)
      .Tensor("kv_last_page_len", p.kv_last_page_len, ROOST_DTYPE_I32, p.batch)
      .Aligned("q", p.q.address, 16)
      .Aligned("output", p.output.address, 16)
      .Aligned("k_cache", p.k_cache.address, 16)
      .Aligned("v_cache", p.v_cache.address, 16);
  return gate.status();
}

// ---- Host planning ---------------------------------------------------------------------------------------------------

// rows_per_split: partial rows one split slot holds (decode: the query heads of a sequence; prefill: kPfRows).
// splits_bf16: the prefill slots among them whose rows are bf16; the others are fp32.
Layout MakeLayout(uint64_t work_items, uint64_t ranges, uint64_t merges, uint64_t splits, uint64_t splits_bf16,
                  uint32_t rows_per_split, uint32_t head_dim, uint32_t mode) {
  Layout l;
  l.work_items = work_items;
  l.ranges = ranges;
  l.merges = merges;
  l.splits = splits;
  const bool decode = mode == ROOST_ATTENTION_DECODE;
  const uint64_t item_bytes = decode ? sizeof(DecodeWork) : sizeof(PrefillWork);
  const uint64_t merge_bytes = decode ? sizeof(DecodeMerge) : sizeof(PrefillMerge);
  l.range_offset = roost::RoundUp(work_items * item_bytes, 16);
  l.merge_offset = roost::RoundUp(l.range_offset + (ranges > 0 ? (ranges + 1) * sizeof(int32_t) : 0), 16);
  l.int_bytes = l.merge_offset + merges * merge_bytes;
  l.float_offset = roost::RoundUp(l.int_bytes, kAlign);
  // fp32 rows (a prefill's bf16 ones before them), then (max, sum) pairs
  l.splits_bf16 = splits_bf16;
  l.float_bytes = rows_per_split * (splits * (static_cast<uint64_t>(head_dim) + 2) * sizeof(float) -
                                    splits_bf16 * head_dim * sizeof(uint16_t));
  l.total = l.float_offset + l.float_bytes;
  return l;
}

uint32_t KvLenHost(const RoostPagedAttentionParams& p, uint32_t b) {
  const int64_t pages = p.kv_indptr_host[b + 1] - p.kv_indptr_host[b];
  if (pages <= 0) return 0;
  const int64_t last = p.kv_last_page_len_host != nullptr ? p.kv_last_page_len_host[b] : p.page_size;
  return static_cast<uint32_t>((pages - 1) * p.page_size + last);
}

// The sliding window: query position pos sees keys j >= pos - window (reference CpuOps.cs:180-197, 245-252); -1 (any
// negative window_left) means no window.
int32_t WindowOf(const RoostPagedAttentionParams& p) { return p.window_left < 0 ? -1 : p.window_left; }
// The soft cap as the kernels apply it (in log2 units); a cap of 0 is off and the sign of the cap does not matter
// (cap tanh(s / cap) is even in cap).
SoftCap CapOf(const RoostPagedAttentionParams& p) {
  const float cap = std::fabs(p.logits_soft_cap);
  if (cap == 0.0f) return SoftCap{0.0f, 0.0f};
  const float capl = cap * kLog2e;
  return SoftCap{capl, 2.0f * kLog2e / capl};
}
// First key a decode query (position kv - 1) sees.
int64_t DecodeFirstKey(int64_t kv, int32_t window) { return window < 0 ? 0 : std::max<int64_t>(0, kv - 1 - window); }

// Decode: the batch's 16-token groups are dealt out evenly to `ranges` workgroup ranges (kDecodeWgsPerCu workgroups
// per CU), each range cut at sequence boundaries into pieces. Every workgroup then streams the same number of bytes
// and the grid finishes together instead of in ragged rounds. A sequence cut into several pieces owns consecutive
// partial slots and one DecodeMerge entry (merged by DecodeMergeKernel); a sequence without keys is one empty piece
// that writes its zero rows.
// The split depends on the batch, so the variant is deterministic but not batch invariant.
// (Virtual) KV heads one decode workgroup serves: the largest of 4, 2 and 1 that divides their number, up to about 1 KB
// of an NHD token's row, which the workgroup's wavefronts then read side by side, and up to 2 where the heads lie in
// other places (HND). Measured at 4 / 2 / 1 heads (us): 32 heads over 8 at head dim 128, NHD 107 / 112 / 123; 16 over 4 at
// 256 109 / 105 / 105; 32 over 4 at 128, HND 110 / 107 / 105. With 8 or 16 heads per wavefront at head dim 256 one head per
// workgroup halves the partials: 67 against 70 us at 16 heads over 2, 74 against 79 at 32 over 2 (324 MB each).
uint32_t HeadsPerWorkgroup(const RoostPagedAttentionParams& p) {
  const uint32_t heads = DecodeHeads(p);
  const uint32_t most = p.head_dim == 256 ? (DecodeGroupOf(p) > kGroup ? 1 : 2) : p.kv_layout == ROOST_LAYOUT_PAGED_HND ? 2 : 4;
  return heads % 4 == 0 && most == 4 ? 4 : (heads % 2 == 0 && most >= 2 ? 2 : 1);
}

struct DecodePlan {
  uint32_t heads_per_wg = 1;       // (virtual) KV heads per workgroup
  std::vector<DecodeWork> items;
  std::vector<int32_t> range_ptr;  // ranges + 1 entries; empty when no sequence is planned
  std::vector<DecodeMerge> merges;
  int32_t slots = 0;
  uint64_t ranges() const { return range_ptr.empty() ? 0 : range_ptr.size() - 1; }
};

// One decode row: query token q_back tokens before the last of sequence seq, reading keys [first, end) (host lengths;
// the kernel clamps to the device's).
struct DecodeRow {
  uint32_t seq;
  int32_t q_back;
  int64_t first;
  int64_t end;
};

// How a call's rows are dealt to workgroups. Even: ranges of per_range groups, cut wherever a range is full, which fills
// the chip when there are more groups than slots. Aligned (per_range = the groups of a piece): each row cut by itself into
// pieces of at most per_range groups, a workgroup each, all of them resident at once.
struct DecodeDeal {
  bool aligned = false;
  uint64_t per_range = 1;
  uint32_t heads_per_wg = 1;
};

// Small calls are bound by latency: the steps a wavefront takes one after another (kStepUs each while HBM is not the
// limit), the merge launch (kMergeUs, none if no row is cut) and its pieces (kMergePieceUs each, read in turn). So few
// rows are cut into the piece count that balances the two, with fewer KV heads per workgroup where that gives a row more
// wavefronts; a call that fills the chip keeps the even deal. Fitted on the MI355X (8 heads over 2, head dim 256, cold):
// one context of 1,500 in pieces of 1 / 2 / 4 / 8 / 16 groups 13.5 / 11.7 / 11.9 / 13.1 / 17.8 us, one of 16,000 41 (2) /
// 26 / 21 / 23. Against the
// even deal (with the merge kernel below on both sides): one context of 1,500 13.5 -> 10.7 us, of 16,000 41 -> 18.6; three
// around 2,500 22.4 -> 12.4; 8 around 2,000 21.6 -> 14.1; 17 of 67 9.2 -> 7.0.
constexpr double kDecodeBytesPerUs = 5.6e6;  // the decode stream on the whole chip
constexpr double kLoneBytesPerUs = 4.0e6;    // of a long stream with at most one workgroup on a CU
constexpr double kLoneBytes = 200e6;
constexpr double kStepUs = 1.17;       // a 16-token group of a wavefront
constexpr double kMergeUs = 4.0;       // the merge launch
constexpr double kMergePieceUs = 0.05;
constexpr double kPieceUs = 2.5;       // a further piece of a range: its tables, query and first rows, one after the other
constexpr uint64_t kAlignMost = 16;    // groups per even range from which the even deal is kept unlooked-at

DecodeDeal ChooseDeal(const RoostPagedAttentionParams& p, uint32_t cus, const std::vector<uint64_t>& groups,
                      uint64_t total, uint64_t longest, bool may_align) {
  const uint32_t heads = DecodeHeads(p), most = HeadsPerWorkgroup(p);
  const uint64_t slots = static_cast<uint64_t>(cus) * kDecodeWgsPerCu;
  const double group_us = 16.0 * p.head_dim * 2 * (p.q.dtype == ROOST_DTYPE_F32 ? 4 : 2) / kDecodeBytesPerUs;
  // A long stream (from about 200 MB) with at most one workgroup per CU stays below kLoneBytesPerUs: 17 contexts of 6,960,
  // 8 heads over 2 x 256, took 65.5 us in 255 workgroups, 54 in the even deal's 493. With a second one on a few CUs those end
  // last, as if all had two, where the pieces are about equal: 44 of 1,024, 32 over 8 x 128, 47.7 us in 352 workgroups, 41.2
  // in 474; but 82 of 7 to 116 11.7 us in 328 and 15.1 in 164.
  const double bytes = static_cast<double>(total) * heads * group_us * kDecodeBytesPerUs;
  const double lone_us = bytes > kLoneBytes ? bytes / kLoneBytesPerUs : 0.0;
  auto cost = [&](uint64_t workgroups, uint32_t hpw, uint64_t piece, uint64_t pieces) {
    const double steps = static_cast<double>(roost::CeilDiv(piece, 4 / hpw));
    const bool lopsided = workgroups > cus && 2 * workgroups <= 3 * cus && 4 * workgroups * piece <= 5 * total * (heads / hpw);
    const double streams = static_cast<double>(lopsided ? 2 * cus : workgroups);
    return std::max(steps * std::max(kStepUs, streams * 4 * group_us), workgroups <= cus ? lone_us : 0.0) +
           (pieces > 1 ? kMergeUs + kMergePieceUs * pieces : 0.0);
  };
  DecodeDeal best;
  best.heads_per_wg = most;
  const uint64_t wanted = std::max<uint64_t>(1, slots / (heads / most));
  best.per_range = std::max<uint64_t>(1, roost::CeilDiv(total, std::max<uint64_t>(1, std::min(wanted, total))));
  // A row spans at most ceil(groups / per_range) + 1 pieces; keep that within what the merge kernel combines.
  best.per_range = std::max<uint64_t>(best.per_range, roost::CeilDiv(longest, kMaxMergeSplits - 2));
  // In f32 the kernel spills at head dim 256 and a step takes many times kStepUs: cut row by row, 30 rows of 1,200 keys took
  // 310 us (even: 122). At 64 and 128 the constants serve: one row of 1,500 13.5 -> 10.5 and 15.8 -> 13.8 us, 8 around 2,000
  // 19.6 -> 12.0 and 27.4 -> 19.4, a prompt of 100 10.9 -> 7.5 and 14.9 -> 15.0.
  if (p.q.dtype == ROOST_DTYPE_F32 && p.head_dim == 256) return best;
  if (!may_align || groups.size() > slots || best.per_range > kAlignMost) return best;
  const uint64_t ranges = roost::CeilDiv(total, best.per_range);
  double best_us = cost(ranges * (heads / most), most, best.per_range,
                        groups.size() == 1 && ranges == 1 ? 1 : roost::CeilDiv(longest, best.per_range) + 1);
  if (groups.size() > 1) best_us += kPieceUs;  // ranges that hold the end of one row and the start of the next
  for (uint64_t piece = 1; ; piece = std::min(longest, piece < 4 ? piece + 1 : piece + piece / 4)) {
    uint64_t n = 0;
    for (const uint64_t g : groups) n += roost::CeilDiv(g, piece);
    const uint64_t pieces = roost::CeilDiv(longest, piece);
    if (pieces <= kMaxMergeSplits) {
      for (uint32_t hpw = most; hpw >= 1; hpw /= 2) {
        const uint64_t workgroups = n * (heads / hpw);
        if (workgroups > slots) break;
        const double us = cost(workgroups, hpw, piece, pieces);
        if (us < best_us) {
          best_us = us;
          best = DecodeDeal{true, piece, hpw};
        }
      }
    }
    if (piece >= longest) break;
  }
  return best;
}

// Cuts the rows' keys into 16-token groups and deals them out (ChooseDeal); a row cut into pieces gets partial slots and a
// DecodeMerge entry.
DecodePlan BuildDecodeRows(const RoostPagedAttentionParams& p, uint32_t cus, const std::vector<DecodeRow>& rows,
                           bool may_align) {
  DecodePlan d;
  d.heads_per_wg = HeadsPerWorkgroup(p);
  if (rows.empty()) return d;
  std::vector<uint64_t> groups(rows.size()), first_group(rows.size());
  uint64_t total = 0;
  for (size_t r = 0; r < rows.size(); ++r) {
    // Keys before the window are never read (their pages may have been released); the first group keeps its
    // 16-alignment and the kernel masks its keys below the window.
    first_group[r] = static_cast<uint64_t>(rows[r].first) / 16;
    groups[r] = rows[r].end > rows[r].first ? roost::CeilDiv(static_cast<uint64_t>(rows[r].end), 16) - first_group[r] : 0;
    total += groups[r];
  }
  const uint64_t longest = *std::max_element(groups.begin(), groups.end());
  const DecodeDeal deal = ChooseDeal(p, cus, groups, total, std::max<uint64_t>(longest, 1), may_align);
  d.heads_per_wg = deal.heads_per_wg;
  d.items.reserve(rows.size() + total / deal.per_range + rows.size());
  d.range_ptr.push_back(0);
  uint64_t room = deal.per_range;  // groups left in the current range
  auto next_range = [&]() {
    d.range_ptr.push_back(static_cast<int32_t>(d.items.size()));
    room = deal.per_range;
  };
  for (size_t r = 0; r < rows.size(); ++r) {
    const auto seq = static_cast<int32_t>(rows[r].seq);
    const int32_t back = rows[r].q_back;
    if (groups[r] == 0) {
      d.items.push_back(DecodeWork{seq, 0, 0, -1, back});
      continue;
    }
    const uint64_t cuts = deal.aligned ? roost::CeilDiv(groups[r], deal.per_range) : 0;  // pieces of an aligned row
    if (deal.aligned && d.items.size() > static_cast<size_t>(d.range_ptr.back())) next_range();
    const size_t first_item = d.items.size();
    uint64_t g = 0;
    while (g < groups[r]) {
      if (room == 0 || (deal.aligned && g > 0)) next_range();
      const uint64_t done = d.items.size() - first_item;
      const uint64_t n = deal.aligned ? groups[r] * (done + 1) / cuts - g : std::min(room, groups[r] - g);
      d.items.push_back(DecodeWork{seq, static_cast<int32_t>((first_group[r] + g) * 16),
                                   static_cast<int32_t>(std::min<uint64_t>((first_group[r] + g + n) * 16,
                                                                           static_cast<uint64_t>(rows[r].end))),
                                   -1, back});
      g += n;
      room -= std::min(room, n);
    }
    const size_t pieces = d.items.size() - first_item;
    if (pieces > 1) {
      d.merges.push_back(DecodeMerge{seq, d.slots, static_cast<int32_t>(pieces), back});
      for (size_t i = first_item; i < d.items.size(); ++i) d.items[i].slot = d.slots++;
    }
  }
  d.range_ptr.push_back(static_cast<int32_t>(d.items.size()));
  return d;
}

// The last-token rows of the sequences b with take(b) (all of them in a decode call, the single-token ones in a
// prefill call).
template <typename Take>
DecodePlan BuildDecode(const RoostPagedAttentionParams& p, uint32_t cus, bool may_align, Take take) {
  std::vector<DecodeRow> rows;
  const int32_t window = WindowOf(p);
  for (uint32_t b = 0; b < p.batch; ++b) {
    if (!take(b)) continue;
    const int64_t kv = KvLenHost(p, b);
    rows.push_back(DecodeRow{b, 0, DecodeFirstKey(kv, window), kv});
  }
  return BuildDecodeRows(p, cus, rows, may_align);
}

// Every query token of every sequence as its own row (the f32 prefill, which runs on the VALU decode kernel): token i
// of a sequence of n tokens and kv keys sits at position kv - n + i and reads keys from its window start to itself
// (causal) or to the end.
DecodePlan BuildDecodeAllTokens(const RoostPagedAttentionParams& p, uint32_t cus) {
  std::vector<DecodeRow> rows;
  const int32_t window = WindowOf(p);
  for (uint32_t b = 0; b < p.batch; ++b) {
    const int64_t n = p.q_indptr_host[b + 1] - p.q_indptr_host[b];
    const int64_t kv = KvLenHost(p, b);
    for (int64_t i = 0; i < n; ++i) {
      const int64_t pos = kv - n + i;
      const int64_t end = p.causal ? std::max<int64_t>(0, pos + 1) : kv;
      const int64_t first = window < 0 ? 0 : std::max<int64_t>(0, pos - window);
      rows.push_back(DecodeRow{b, static_cast<int32_t>(n - 1 - i), std::min(first, end), end});
    }
  }
  return BuildDecodeRows(p, cus, rows, true);
}

// Places a decode plan at the end of the int region [0, l.int_bytes) and its partials at the end of the float region
// (which must not be laid out yet), then writes it to host when given.
void AppendDecode(const RoostPagedAttentionParams& p, const DecodePlan& d, Layout& l, unsigned char* host) {
  l.dec_heads_per_wg = d.heads_per_wg;
  l.dec_items = d.items.size();
  l.dec_ranges = d.ranges();
  l.dec_merges = d.merges.size();
  l.dec_splits = static_cast<uint64_t>(d.slots);
  l.dec_item_offset = roost::RoundUp(l.int_bytes, 16);
  l.dec_range_offset = roost::RoundUp(l.dec_item_offset + l.dec_items * sizeof(DecodeWork), 16);
  l.dec_merge_offset = roost::RoundUp(l.dec_range_offset + d.range_ptr.size() * sizeof(int32_t), 16);
  l.int_bytes = l.dec_merge_offset + l.dec_merges * sizeof(DecodeMerge);
  if (host != nullptr) {
    std::memcpy(host + l.dec_item_offset, d.items.data(), d.items.size() * sizeof(DecodeWork));
    std::memcpy(host + l.dec_range_offset, d.range_ptr.data(), d.range_ptr.size() * sizeof(int32_t));
    std::memcpy(host + l.dec_merge_offset, d.merges.data(), d.merges.size() * sizeof(DecodeMerge));
  }
  (void)p;
}

// Lays out the float region after the int region: the prefill partials (prefill_floats bytes), then the decode ones.
void PlaceFloats(const RoostPagedAttentionParams& p, uint64_t prefill_floats, Layout& l) {
  l.float_offset = roost::RoundUp(l.int_bytes, kAlign);
  l.dec_float_offset = l.float_offset + roost::RoundUp(prefill_floats, kAlign);
  l.float_bytes = (l.dec_float_offset - l.float_offset) +
                  l.dec_splits * p.q_heads * (static_cast<uint64_t>(p.head_dim) + 2) * sizeof(float);
  l.total = l.float_offset + l.float_bytes;
}

Layout PlanDecode(const RoostPagedAttentionParams& p, uint32_t cus, unsigned char* host) {
  const DecodePlan d = BuildDecode(p, cus, true, [](uint32_t) { return true; });
  Layout l;
  AppendDecode(p, d, l, host);
  PlaceFloats(p, 0, l);
  // The decode call's record fields name the same region.
  l.work_items = l.dec_items;
  l.ranges = l.dec_ranges;
  l.merges = l.dec_merges;
  l.splits = l.dec_splits;
  l.range_offset = l.dec_range_offset;
  l.merge_offset = l.dec_merge_offset;
  return l;
}

// Prefill work items: one per (query tile, KV head) -- 64-token tiles when the page size is a multiple of 16 (the
// DMA-fed kernel; 96-token ones at head dim 128 where that ends earlier), 32-token tiles otherwise. The DMA-fed kernel's
// key ranges are cut into pieces of whole 64-key tiles where they are longer than a share of the average load of a CU
// (at least kPfMinSplitTiles each, so that the longest causal tile does not set the makespan), where CUs would stay idle
// (SparsePieceTiles, down to 2 tiles) and beside decode ranges (ChooseOverlap); the pieces write partials merged by
// PrefillMergeKernel. Items are ordered longest first. The cuts depend on the whole batch, so the variant is deterministic
// but not batch invariant.
bool PrefillFastPath(const RoostPagedAttentionParams& p) {
  return p.page_size % 16 == 0 && (p.page_size & (p.page_size - 1)) == 0;
}

// The work items of a call by their key ranges in 64-key tiles: `tiles` holds one entry per query tile, of which `heads`
// items (one per group of kGroup query heads) are cut alike.
struct ItemList {
  std::vector<int64_t> tiles;
  int64_t heads = 1;
  int64_t count() const { return static_cast<int64_t>(tiles.size()) * heads; }
  int64_t longest() const { return tiles.empty() ? 0 : *std::max_element(tiles.begin(), tiles.end()); }
  int64_t total() const {
    int64_t sum = 0;
    for (int64_t t : tiles) sum += t;
    return sum * heads;
  }
};

// The pieces an item of `tiles` tiles is cut into with at most `target` each.
int64_t Pieces(int64_t tiles, int64_t target) { return std::min<int64_t>(roost::CeilDiv(tiles, target), kMaxMergeSplits); }

// The longest-first dispatch of the items cut at `target` onto `cus` workgroup slots, each piece costing its tiles
// plus kPfPieceCost (its set-up and epilogue): the finishing time of the last slot, in tiles.
constexpr int64_t kPfPieceCost = 2;
int64_t PrefillMakespan(const ItemList& items, int64_t target, uint32_t cus) {
  // Piece costs by counting (they are small integers), then longest first onto the least loaded slot.
  std::vector<int64_t> count;
  for (const int64_t tiles : items.tiles) {
    const int64_t n = Pieces(tiles, target);
    for (int64_t i = 0; i < n; ++i) {
      const auto c = static_cast<size_t>(tiles * (i + 1) / n - tiles * i / n + kPfPieceCost);
      if (c >= count.size()) count.resize(c + 1, 0);
      count[c] += items.heads;
    }
  }
  // Slots by load (at[L]: how many slots carry L tiles); loads only grow, so the least loaded level only moves up, and
  // pieces of one cost fill a level's slots together.
  std::vector<int64_t> at(1, std::max<uint32_t>(cus, 1));
  size_t lo = 0, end = 0;
  for (size_t c = count.size(); c-- > 0;) {
    for (int64_t left = count[c]; left > 0;) {
      while (at[lo] == 0) ++lo;
      const int64_t n = std::min(at[lo], left);
      left -= n;
      at[lo] -= n;
      const size_t load = lo + c;
      if (load >= at.size()) at.resize(load + 1, 0);
      at[load] += n;
      end = std::max(end, load);
    }
  }
  return static_cast<int64_t>(end);
}

// The piece size (in tiles, at least kPfMinSplitTiles) the 64-token kernel cuts key ranges at. Candidates: 3/4, 17/20
// and the whole of the average CU load, and the smallest sizes whose pieces fill the CUs exactly once or twice
// (config 5's two 512-token chunks: 256 pieces of 9 tiles instead of 288 of 8, whose last 32 ran in a second round);
// the one whose longest-first dispatch ends first wins. Config 3 keeps 3/4 (0.197 ms, against 0.203 at 17/20 and
// 0.234 at 13/20); a dense 4 x 4096 batch takes the whole average (1,095 against 950 TFLOP/s at 3/4).
struct PieceChoice {
  int64_t target;  // piece size in tiles
  int64_t end;     // the dispatch's finishing time in tiles
  int64_t cut;     // pieces of cut items
};

PieceChoice PrefillPieceTiles(const ItemList& items, uint32_t cus) {
  const uint32_t slots = std::max<uint32_t>(cus, 1);
  const int64_t total_tiles = items.total();
  auto of_avg = [&](int64_t num, int64_t den) {
    return std::max<int64_t>(kPfMinSplitTiles, roost::CeilDiv(total_tiles * num, den * int64_t{slots}));
  };
  std::vector<int64_t> cand{of_avg(3, 4), of_avg(17, 20), of_avg(1, 1)};
  const int64_t longest = items.longest();
  for (int64_t rounds = 1; rounds <= 2; ++rounds) {
    if (items.count() > rounds * slots) break;
    // Smallest target whose pieces number at most rounds x slots (the count only falls as the target grows).
    int64_t lo = kPfMinSplitTiles, hi = std::max<int64_t>(longest, kPfMinSplitTiles);
    auto count = [&](int64_t t) {
      int64_t n = 0;
      for (const int64_t tiles : items.tiles) n += Pieces(tiles, t);
      return n * items.heads;
    };
    if (count(hi) > rounds * slots) continue;
    while (lo < hi) {
      const int64_t mid = (lo + hi) / 2;
      if (count(mid) <= rounds * slots) hi = mid; else lo = mid + 1;
    }
    cand.push_back(lo);
  }
  int64_t best = cand[0], best_end = PrefillMakespan(items, cand[0], slots);
  for (size_t i = 1; i < cand.size(); ++i) {
    const int64_t end = PrefillMakespan(items, cand[i], slots);
    if (end < best_end || (end == best_end && cand[i] > best)) {
      best = cand[i];
      best_end = end;
    }
  }
  int64_t cut = 0;
  for (const int64_t tiles : items.tiles) {
    const int64_t n = Pieces(tiles, best);
    if (n > 1) cut += n * items.heads;
  }
  return {best, best_end, cut};
}

// Calls whose pieces do not fill the CUs once (a short prompt: 1,777 tokens x 2 KV heads made 128 pieces of up to 8
// tiles for 256 CUs): pieces below kPfMinSplitTiles, down to 2 tiles, while they still run in one round. Each is priced by
// what such calls measured: a tile on a chip with idle CUs 2.3 us at head dim 256, the merge launch 4.5 us, and 0.08 us
// per piece for its partial rows written and merged (both sides less at smaller head dims). Fresh prompts of 8 heads over 2,
// pieces of at least 8 tiles against this choice (us): head dim 256, 500 tokens 38.6 -> 29.2, 1,000 45.4 -> 37.8, 1,777
// 51.8 -> 47.1, 256 on 4,000 cached ones 48.1 -> 40.4; 128, 500 23.4 -> 17.4, 1,000 28.9 -> 21.6; 64, 500 17.0 -> 14.3,
// 1,000 23.0 -> 16.4. 200 tokens stay whole: 23.9 / 13.1 / 10.2 at 256 / 128 / 64 against 27.3 / 16.3 / 13.2 in pieces of 2.
// Over prompts of 100 to 1,777 tokens at the three head dims the choice was within 5% of the best of 2 to 8 tiles, but for
// chunks of 100 on 300 at 64 (12%, left whole).
constexpr double kSparseTileUs = 2.3;
constexpr double kPieceMergeUs = 0.08;
constexpr double kMergeLaunchUs = 4.5;

int64_t SparsePieceTiles(const ItemList& items, int64_t target, uint32_t head_dim, uint32_t cus) {
  if (items.count() >= static_cast<int64_t>(cus)) return target;
  const double rel = head_dim / 256.0;
  const double tile_us = kSparseTileUs * (0.25 + 0.75 * rel);
  int64_t best = target;
  double best_us = 0.0;
  for (int64_t t = target; t >= 2; t = std::min(t, static_cast<int64_t>(kPfMinSplitTiles)) - 1) {
    int64_t n = 0, longest = 0;
    for (const int64_t tiles : items.tiles) {
      const int64_t pieces = Pieces(tiles, t);
      n += pieces * items.heads;
      longest = std::max<int64_t>(longest, pieces > 0 ? (tiles + pieces - 1) / pieces : 0);
    }
    if (n > static_cast<int64_t>(cus)) break;  // one round: the longest piece ends last
    const double us = (longest + kPfPieceCost) * tile_us + n * kPieceMergeUs * rel +
                      (n > items.count() ? kMergeLaunchUs : 0.0);
    if (t == target || us < best_us) {
      best_us = us;
      best = t;
    }
  }
  return best;
}

// Side by side or one after the other. A prefill call that also holds single-token sequences (a mixed worker step)
// runs MFMA-bound tile pieces and HBM-bound decode ranges. A tile workgroup needs a whole CU (two 256-register
// wavefronts per SIMD and 128 KB of LDS), so the two kinds cannot share CUs; but when the tile items are cut into fewer,
// longer pieces they hold only as many CUs as there are pieces, and decode ranges sized for the remaining CUs stream
// K/V on those, both in one launch (MixedAttentionKernel). ChooseOverlap estimates both schedules with rates measured
// on the MI355X -- a 64-key tile at head dim 256 takes ~3.7 us of a CU (less at smaller head dims), the decode stream as
// below, and the merged launch costs ~3 us more than its longer side -- and keeps the cheaper. Config 5 (48 decode rows
// over 831 MB of K/V, two 512-token chunks): 64 pieces beside decode ranges for the other 191 CUs. The decode side needs
// page sizes that are multiples of 16 (its fast-page form).
// The decode stream with groups of 8 and more query heads: 28 KB a us and CU up to 5.6 TB/s, 4 us for every piece a CU
// takes in turn (an epilogue of up to 16 heads); 16 us for the further launches of the two schedules one after the other;
// 2 us for the merge of the pieces and 0.01 (bf16) or 0.04 us (fp32) for each at head dim 256. Fitted to 140 mixed calls of
// such groups (1 to 128 rows of 4 to 16,384 keys, 1 to 3 chunks, head dims 64 to 256): the choice is 1% above the best of 1
// to 16 cuts on average and 17% at worst. Priced as groups of 4 are, it was 11% and 3.4 times: 2 rows of 9,577 keys beside
// a chunk of 190 on 1,769, 32 heads over 2 x 256, 141 us (53 now).
// With groups of 4: 5.6 TB/s on 256 CUs, falling off as (CUs / 256)^0.26 (5.2 TB/s on 192, but with few CUs 64 reach 2.5
// TB/s and not 3.9). On 60 such calls the choice is 8% above the best on average and 65% at worst; where it goes wrong, too
// few CUs are left for the decode ranges.
struct OverlapChoice {
  bool use = false;
  int64_t target = 0;    // piece size (tiles) of the tile kernel
  uint32_t dec_cus = 0;  // CUs the decode ranges are sized for
  bool bf16 = true;      // the pieces' partials are bf16
};

constexpr double kTileUsD256 = 3.7;
constexpr double kMixedLaunchUs = 3.0;

double TileUs(uint32_t head_dim) { return kTileUsD256 * (0.25 + 0.75 * head_dim / 256.0); }
double DecodeUs(double bytes, uint32_t cus_used, uint32_t cus) {
  return bytes / (kDecodeBytesPerUs * std::pow(static_cast<double>(cus_used) / cus, 0.26));
}
constexpr double kBigGroupCuBytesPerUs = 28e3;
constexpr double kBigGroupPieceUs = 4.0;
constexpr double kBigGroupSerialUs = 16.0;
constexpr double kBigGroupMergeUs = 2.0;
constexpr double kBigGroupMergeBf16Us = 0.01, kBigGroupMergeF32Us = 0.04;

template <typename Single>
OverlapChoice ChooseOverlap(const RoostPagedAttentionParams& p, const ItemList& items, int64_t serial_target, uint32_t cus,
                            Single single) {
  OverlapChoice best;
  double dec_bytes = 0.0;
  uint64_t rows = 0;
  for (uint32_t b = 0; b < p.batch; ++b) {
    if (!single(b)) continue;
    ++rows;
    dec_bytes += static_cast<double>(KvLenHost(p, b)) * DecodeHeads(p) * p.head_dim * 2.0 * 2.0;
  }
  const bool big = DecodeGroupOf(p) > kGroup;
  const double blocks = static_cast<double>(rows) * (DecodeHeads(p) / HeadsPerWorkgroup(p));
  auto stream_us = [&](uint32_t n) {
    return big ? dec_bytes / std::min(kDecodeBytesPerUs, n * kBigGroupCuBytesPerUs) : DecodeUs(dec_bytes, n, cus);
  };
  if (dec_bytes == 0.0 || items.tiles.empty() || cus < 2 || p.page_size % 16 != 0) return best;
  const int64_t longest = items.longest();
  const double tile_us = TileUs(p.head_dim);
  double best_us = PrefillMakespan(items, serial_target, cus) * tile_us + stream_us(cus) + (big ? kBigGroupSerialUs : 0.0);
  for (int64_t k = 1; k <= 16; ++k) {
    const int64_t target = std::max<int64_t>(1, roost::CeilDiv(longest, k));
    int64_t pieces = 0, merged = 0, piece_max = 0;
    for (const int64_t tiles : items.tiles) {
      const int64_t n = Pieces(tiles, target);
      pieces += n * items.heads;
      if (n > 1) merged += n * items.heads;
      piece_max = std::max<int64_t>(piece_max, roost::CeilDiv(tiles, n));
    }
    if (pieces >= static_cast<int64_t>(cus)) break;
    const uint32_t left = cus - static_cast<uint32_t>(pieces);
    const double pieces_us = static_cast<double>(piece_max + kPfPieceCost) * tile_us;
    const double decode_us = stream_us(left) + (big ? kBigGroupPieceUs * blocks / left : 0.0);
    // The decode ranges of larger groups end early, and items are cut to end with them. Where the ranges take any share of
    // the time, such an item might as well run whole: its pieces keep fp32 partials (2 to 12% of a small call). In calls
    // that the pieces alone decide, every schedule cuts the items, and they stay in bf16.
    const bool bf16 = !big || 4 * stream_us(left) < pieces_us;
    double us = std::max(pieces_us, decode_us) + kMixedLaunchUs;
    if (big && merged > 0) {
      us += kBigGroupMergeUs + (bf16 ? kBigGroupMergeBf16Us : kBigGroupMergeF32Us) * merged * p.head_dim / 256.0;
    }
    if (us < best_us) {
      best_us = us;
      best.use = true;
      best.target = target;
      best.dec_cus = left;
      best.bf16 = bf16;
    }
  }
  return best;
}

Layout PlanPrefill(const RoostPagedAttentionParams& p, uint32_t cus, unsigned char* host) {
  if (p.q.dtype == ROOST_DTYPE_F32) {  // no f32 MFMA tile kernel: every query token is a row of the f32 decode kernel
    Layout l = MakeLayout(0, 0, 0, 0, 0, kPfRows, p.head_dim, ROOST_ATTENTION_PREFILL);
    AppendDecode(p, BuildDecodeAllTokens(p, cus), l, host);
    PlaceFloats(p, 0, l);
    return l;
  }
  const bool fast = PrefillFastPath(p);
  struct Item {
    PrefillWork w;
    int64_t cost;
  };
  const int32_t window = WindowOf(p);
  // A sequence with one query token (a decode row of a mixed step) sees every key whether causal or not: the decode
  // kernel streams it at HBM speed instead of a 64-row MFMA tile holding one row.
  auto single = [&](uint32_t b) { return p.q_indptr_host[b + 1] - p.q_indptr_host[b] == 1; };
  // Visits every query tile of tile_q tokens: (sequence, first token, tokens, key range).
  auto query_tiles = [&](int64_t tile_q, auto&& visit) {
    for (uint32_t b = 0; b < p.batch; ++b) {
      if (single(b)) continue;
      const int64_t n = p.q_indptr_host[b + 1] - p.q_indptr_host[b];
      const int64_t kv = KvLenHost(p, b);
      for (int64_t q0 = 0; q0 < n; q0 += tile_q) {
        const int64_t rows = std::min<int64_t>(tile_q, n - q0);
        int64_t kend = p.causal ? std::min<int64_t>(kv, kv - n + q0 + rows) : kv;
        if (kend < 0) kend = 0;
        // With a window the item's first query (position kv - n + q0) sees keys from kv - n + q0 - window on; the
        // range starts at that key rounded down to 16 (a 16-row group never straddles a page), and keys before it are
        // never read.
        int64_t kbeg = window < 0 ? 0 : std::max<int64_t>(0, kv - n + q0 - window) / 16 * 16;
        if (kbeg > kend) kbeg = kend;
        visit(b, q0, rows, kbeg, kend);
      }
    }
  };
  auto item_list = [&](int64_t tile_q) {
    ItemList l;
    l.heads = VirtualHeads(p);
    query_tiles(tile_q, [&](uint32_t, int64_t, int64_t, int64_t kbeg, int64_t kend) {
      l.tiles.push_back(roost::CeilDiv(kend - kbeg, 64));
    });
    return l;
  };
  int64_t tile_q = fast ? kPfTokens : kPrefillTileQ;
  int64_t target = 0;
  int64_t whole = 0;  // longest key range in tiles that load balance alone leaves whole
  OverlapChoice overlap;
  if (fast) {
    ItemList list = item_list(tile_q);
    const PieceChoice narrow = PrefillPieceTiles(list, cus);
    target = whole = narrow.target;
    overlap = ChooseOverlap(p, list, target, cus, single);
    if (overlap.use) {
      target = overlap.target;
    } else {
      if (p.head_dim == kPfWideDim) {
        ItemList wide_list = item_list(kPfWideTokens);
        const PieceChoice wide = PrefillPieceTiles(wide_list, cus);
        if (wide.end * kPfWideTileCost + wide.cut * kPfCutPieceTiles < narrow.end + narrow.cut * kPfCutPieceTiles) {
          tile_q = kPfWideTokens;
          target = wide.target;
          list = std::move(wide_list);
        }
      }
      target = SparsePieceTiles(list, target, p.head_dim, cus);
    }
  }
  std::vector<Item> items;
  query_tiles(tile_q, [&](uint32_t b, int64_t q0, int64_t rows, int64_t kbeg, int64_t kend) {
    for (uint32_t h = 0; h < VirtualHeads(p); ++h) {  // item per group of kGroup query heads
      items.push_back(Item{PrefillWork{static_cast<int32_t>(b), static_cast<int32_t>(q0), static_cast<int32_t>(h),
                                       static_cast<int32_t>(rows), static_cast<int32_t>(kbeg),
                                       static_cast<int32_t>(kend), -1, kPieceFirst | kPieceLast},
                           kend - kbeg + 64});
    }
  });
  // A bf16 partial row is one rounding more (2-norm error of a row against 64 bits: 0.0023 whole, 0.0029 merged from bf16,
  // however many pieces). Items that load balance cuts anyway take it: their merge would read twice the bytes. An item that
  // is cut only for idle CUs or under the wide form keeps fp32 partials: fresh prompts of 500 / 1,000 tokens (8 heads over 2,
  // head dim 256) 26.7 / 34.9 us in bf16 pieces, 29.5 / 37.3 in fp32, 38.5 / 45.3 not cut so.
  std::vector<PrefillMerge> merges;
  uint64_t splits_bf16 = 0, splits = 0;
  if (fast) {
    auto tiles_of = [](const Item& it) { return roost::CeilDiv(static_cast<int64_t>(it.w.kend - it.w.kbeg), 64); };
    // (The 64-token items under a 96-token one are at most a tile shorter.)
    auto bf16_partials = [&](const Item& it) {
      return overlap.use ? overlap.bf16 : tiles_of(it) - (tile_q == kPfWideTokens ? 1 : 0) > whole;
    };
    for (const Item& it : items) {
      const int64_t pieces = Pieces(tiles_of(it), target);
      if (pieces > 1) (bf16_partials(it) ? splits_bf16 : splits) += static_cast<uint64_t>(pieces);
    }
    splits += splits_bf16;
    auto slot16 = int32_t{0}, slot32 = static_cast<int32_t>(splits_bf16);
    std::vector<Item> cut;
    cut.reserve(items.size());
    for (const Item& it : items) {
      const int64_t tiles = tiles_of(it), pieces = Pieces(tiles, target);
      if (pieces <= 1) {
        cut.push_back(it);
        continue;
      }
      int32_t& slot = bf16_partials(it) ? slot16 : slot32;
      merges.push_back(PrefillMerge{it.w.seq, it.w.q0, it.w.kv_head, it.w.rows, slot, static_cast<int32_t>(pieces), {0, 0}});
      for (int64_t i = 0; i < pieces; ++i) {
        const int64_t t0 = tiles * i / pieces, t1 = tiles * (i + 1) / pieces;
        PrefillWork w = it.w;
        w.kbeg = static_cast<int32_t>(it.w.kbeg + t0 * 64);
        w.kend = static_cast<int32_t>(std::min<int64_t>(it.w.kbeg + t1 * 64, it.w.kend));
        w.slot = slot++;
        w.ends = (i == 0 ? kPieceFirst : 0) | (i == pieces - 1 ? kPieceLast : 0);
        cut.push_back(Item{w, (t1 - t0) * 64 + 64});
      }
    }
    items.swap(cut);
  }
  std::stable_sort(items.begin(), items.end(), [](const Item& a, const Item& b) { return a.cost > b.cost; });
  // Merges of exactly two pieces first: they run on the 8-rows-per-block form of the merge kernel.
  std::stable_partition(merges.begin(), merges.end(), [](const PrefillMerge& m) { return m.count == 2; });
  Layout l = MakeLayout(items.size(), 0, merges.size(), splits, splits_bf16,
                        static_cast<uint32_t>(tile_q) * kGroup, p.head_dim, ROOST_ATTENTION_PREFILL);
  l.item_tokens = fast ? static_cast<uint32_t>(tile_q) : kPfTokens;
  l.merges_two = static_cast<uint64_t>(
      std::count_if(merges.begin(), merges.end(), [](const PrefillMerge& m) { return m.count == 2; }));
  if (host != nullptr) {
    auto* w = reinterpret_cast<PrefillWork*>(host);
    for (size_t i = 0; i < items.size(); ++i) w[i] = items[i].w;
    std::memcpy(host + l.merge_offset, merges.data(), merges.size() * sizeof(PrefillMerge));
  }
  const uint64_t prefill_floats = l.float_bytes;
  l.overlap = overlap.use ? 1u : 0u;
  // Side by side, a decode workgroup has 8 wavefronts and a CU to itself: ranges for dec_cus / 2 CUs at
  // kDecodeWgsPerCu 4-wavefront workgroups each are one range per free CU.
  // With groups of 4 the even deal is kept there: cut row by row, calls of few rows took up to 12% longer. Larger groups,
  // whose pieces end in longer epilogues, gain (by 7% on average, 4% at most lost; 109 rows of 141 keys beside a prompt of
  // 68, 32 heads over 2 x 128: 20.9 -> 11.4 us).
  AppendDecode(p, BuildDecode(p, overlap.use ? std::max(1u, overlap.dec_cus / kDecodeWgsPerCu) : cus,
                              !overlap.use || DecodeGroupOf(p) > kGroup, single),
               l, host);
  PlaceFloats(p, prefill_floats, l);
  return l;
}

uint32_t ComputeUnits(const RoostContext* ctx) { return ctx != nullptr && ctx->compute_units > 0 ? ctx->compute_units : 256; }

Layout PlanLayout(const RoostPagedAttentionParams& p, uint32_t cus, unsigned char* host) {
  return p.mode == ROOST_ATTENTION_DECODE ? PlanDecode(p, cus, host) : PlanPrefill(p, cus, host);
}

// ---- Device helpers --------------------------------------------------------------------------------------------------

struct KvView {
  const void* k;
  const void* v;
  const int32_t* kv_indptr;
  const int32_t* kv_indices;
  const int32_t* last_len;
  uint64_t pool_pages;  // pages the pools hold; page ids outside [0, pool_pages) are skipped
  uint32_t page_size;
  uint32_t kv_heads;    // real KV heads of the pools (their row strides)
  uint32_t hnd;
  uint32_t head_shift;  // the kernels work on groups of kGroup query heads ("virtual" KV heads, q_heads / kGroup of
                        // them); virtual head v reads the K/V rows of real head v >> head_shift
  uint32_t vheads;      // q_heads / kGroup
  const void* out_gate;  // the output gate ([tokens, q_heads * head_dim] in the output's type), or NULL for none
};

__device__ __forceinline__ uint32_t SeqKvLen(const KvView& kv, int32_t b, int32_t* p0) {
  const int32_t a = kv.kv_indptr[b];
  const int32_t e = kv.kv_indptr[b + 1];
  *p0 = a;
  const int32_t pages = e - a;
  if (pages <= 0) return 0;
  int32_t last = kv.last_len[b];
  last = last < 1 ? 1 : (last > static_cast<int32_t>(kv.page_size) ? static_cast<int32_t>(kv.page_size) : last);
  return static_cast<uint32_t>((pages - 1) * static_cast<int32_t>(kv.page_size) + last);
}

// Element offset of key `j` of a sequence (page table starting at entry p0) for KV head h, or -1 when its page id is
// outside the pool (a released or corrupt entry: the key is treated as absent instead of faulting).
template <int D>
__device__ __forceinline__ int64_t KeyRow(const KvView& kv, int32_t p0, uint32_t j, uint32_t h) {
  const uint32_t pi = j / kv.page_size;
  const uint32_t off = j - pi * kv.page_size;
  const int32_t page = kv.kv_indices[p0 + pi];
  if (page < 0 || static_cast<uint64_t>(page) >= kv.pool_pages) return -1;
  const uint64_t pg = static_cast<uint64_t>(page);
  const uint32_t hr = h >> kv.head_shift;
  const uint64_t row = kv.hnd ? (pg * kv.kv_heads + hr) * kv.page_size + off : (pg * kv.page_size + off) * kv.kv_heads + hr;
  return static_cast<int64_t>(row * D);
}

// Branch-free form for the prefill tile loads: key j (clamped into [0, key_end)) always yields a loadable offset;
// *ok says whether the key exists (j < key_end and its page id is inside the pool).
template <int D>
__device__ __forceinline__ uint64_t KeyRowSafe(const KvView& kv, int32_t p0, int32_t j, int32_t key_end, uint32_t h,
                                               bool* ok) {
  const uint32_t jc = static_cast<uint32_t>(min(j, key_end - 1));
  const uint32_t pi = jc / kv.page_size;
  const uint32_t off = jc - pi * kv.page_size;
  const int32_t page = kv.kv_indices[p0 + pi];
  const bool good = j < key_end && page >= 0 && static_cast<uint64_t>(page) < kv.pool_pages;
  *ok = good;
  const uint64_t pg = good ? static_cast<uint64_t>(page) : 0;
  const uint32_t hr = h >> kv.head_shift;
  const uint64_t row = kv.hnd ? (pg * kv.kv_heads + hr) * kv.page_size + off : (pg * kv.page_size + off) * kv.kv_heads + hr;
  return good ? row * D : 0;
}

// A float as the output type stores it.
template <typename T>
__device__ __forceinline__ T Narrow(float x) {
  if constexpr (sizeof(T) == 2) return F32ToBf16(x); else return x;
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// The output gate (SigmoidMul folded into the epilogue): output element e, already rounded to the output type, times
// sigmoid(gate[e]) with SigmoidMul's own arithmetic; unchanged without a gate. GateOut2 takes two packed bf16 pairs.
__device__ __forceinline__ u32x2_t GateOut2(const void* gate, uint64_t e, u32x2_t v) {
  if (gate == nullptr) return v;
  const u32x2_t g = *reinterpret_cast<const u32x2_t*>(static_cast<const uint16_t*>(gate) + e);
  return u32x2_t{GateMulBf16x2(v[0], g[0]), GateMulBf16x2(v[1], g[1])};
}
template <typename T>
__device__ __forceinline__ T GateOut(const void* gate, uint64_t e, T v) {
  return gate == nullptr ? v : GateMul(v, static_cast<const T*>(gate)[e]);
}
// The same in two steps, for epilogues that request the gate before their own loads land: the raw gate words of
// element e (zero without a gate), then the product.
__device__ __forceinline__ u32x2_t GateFetch2(const void* gate, uint64_t e) {
  return gate == nullptr ? u32x2_t{0, 0} : *reinterpret_cast<const u32x2_t*>(static_cast<const uint16_t*>(gate) + e);
}
__device__ __forceinline__ u32x2_t GateApply2(const void* gate, u32x2_t g, u32x2_t v) {
  return gate == nullptr ? v : u32x2_t{GateMulBf16x2(v[0], g[0]), GateMulBf16x2(v[1], g[1])};
}
template <typename T>
__device__ __forceinline__ T GateFetch(const void* gate, uint64_t e) {
  return gate == nullptr ? T{} : static_cast<const T*>(gate)[e];
}
template <typename T>
__device__ __forceinline__ T GateApply(const void* gate, T g, T v) {
  return gate == nullptr ? v : GateMul(v, g);
}

// 16-byte load with the non-temporal hint, for data read exactly once in whole cache lines per instruction (f32 K and V).
__device__ __forceinline__ uint4 LoadStream16(const void* p) {
  const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// Partial dot product of a 16-byte f32 K vector with the matching 16 bytes of q.
__device__ __forceinline__ float Dot16(const uint4& k, const float* q, float acc) {
  acc = fmaf(__uint_as_float(k.x), q[0], acc);
  acc = fmaf(__uint_as_float(k.y), q[1], acc);
  acc = fmaf(__uint_as_float(k.z), q[2], acc);
  acc = fmaf(__uint_as_float(k.w), q[3], acc);
  return acc;
}

__device__ __forceinline__ float ShflXor(float v, int mask) { return __shfl_xor(v, mask, 64); }

// A lane's value combined with that of lane ^ 32 through v_permlane32_swap (registers only, no LDS round trip): the
// swap leaves each lane holding both values, so max and sum need no select and both lanes get the same bits.
__device__ __forceinline__ float MaxXor32(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float SumXor32(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// x[i] for a runtime i in [0, 4) without indexing a register array (which would spill it to scratch).
__device__ __forceinline__ float Pick4(const float* x, int i) {
  return i == 0 ? x[0] : (i == 1 ? x[1] : (i == 2 ? x[2] : x[3]));
}

// What the f32 decode kernel reads as the V row of a token that is not there, where no visible token's row is at hand: its
// weight is 0, but 0 times a row that nobody wrote may be NaN. 256 floats, the longest row.
__device__ __align__(16) uint32_t kZeroRow[256];

// ---- f32 decode kernel -----------------------------------------------------------------------------------------------

template <int D>
struct DecodeCfg {
  static constexpr int kVec = 4;                     // floats per 16-byte vector
  static constexpr int kLpr = D / kVec;              // lanes per K/V row
  static constexpr int kTpi = 64 / kLpr;             // rows (tokens) per wave-wide load
  static constexpr int kNi = 16 / kTpi;              // loads per 16-token group per lane
  static_assert(kLpr <= 64 && 64 % kLpr == 0 && 16 % kTpi == 0, "shape");
  static_assert(kNi * kGroup == kLpr, "each lane must end the reduce-scatter with one (token, head) score");
};

// One wavefront's running state: acc[h][e] is this lane's slice of sum_j p_j v_j for query head h, m[h] the running
// max of the head (wave-uniform), l_lane this lane's share of the head-(r % 4) denominator.
template <int D>
struct DecodeState {
  float acc[kGroup][DecodeCfg<D>::kVec];
  float m[kGroup];
  float l_lane;
};

// Folds one 16-token group (already in registers) into the state.
//
// Lane (ri, r) holds, for K, the 16-byte slice r of token slot i ^ (r >> 2) in register i, and q of head h ^ (r & 3)
// in register h; so its partial score register j = 4i + h stands for the logical (slot, head) index j ^ r. With that
// permutation the reduce-scatter needs no selects: at distance mk the partner's register j + mk stands for the same
// logical index as this lane's register j, so s[j] += partner.s[j + mk]; afterwards register 0 holds the complete score
// of index r (slot r / 4, head r % 4). V register i holds slot i in natural order.
// valid: bit s set when token slot s of this lane's row group is a real key.
template <int D>
__device__ __forceinline__ void DecodeGroup(DecodeState<D>& st, const uint4* kr, const uint4* vr, uint32_t valid,
                                            const float (*qr)[DecodeCfg<D>::kVec], float* x_row, int r, int ri, int lane,
                                            float scale_log2, SoftCap cap) {
  using C = DecodeCfg<D>;
  constexpr int kVec = C::kVec, kLpr = C::kLpr, kNi = C::kNi;
  float s[kLpr];
#pragma unroll
  for (int i = 0; i < kNi; ++i)
#pragma unroll
    for (int h = 0; h < (int)kGroup; ++h) s[i * kGroup + h] = Dot16(kr[i], qr[h], 0.0f);
#pragma unroll
  for (int mk = kLpr / 2; mk >= 1; mk >>= 1)
#pragma unroll
    for (int j = 0; j < mk; ++j) s[j] += ShflXor(s[j + mk], mk);
  const int my_head = r % kGroup;
  const bool my_valid = (valid >> (r / kGroup)) & 1u;
  float y = s[0] * scale_log2;
  if (cap.capl != 0.0f) y = Capped(y, cap);
  const float sc = my_valid ? y : -INFINITY;
  // Group max per head (lanes sharing r % 4), then every lane learns all 4.
  float gm = sc;
#pragma unroll
  for (int mk = 4; mk < 64; mk <<= 1) gm = fmaxf(gm, ShflXor(gm, mk));
  const float x1 = ShflXor(gm, 1), x2 = ShflXor(gm, 2), x3 = ShflXor(gm, 3);
  float corr[kGroup];
  bool rescale = false;
#pragma unroll
  for (int h = 0; h < (int)kGroup; ++h) {
    const int dd = h ^ my_head;
    const float hm = dd == 0 ? gm : (dd == 1 ? x1 : (dd == 2 ? x2 : x3));
    const float mn = fmaxf(st.m[h], hm);
    corr[h] = mn == -INFINITY ? 1.0f : exp2f(st.m[h] - mn);
    rescale |= mn != st.m[h];
    st.m[h] = mn;
  }
  const float pw = sc == -INFINITY ? 0.0f : exp2f(sc - Pick4(st.m, my_head));
  st.l_lane = st.l_lane * Pick4(corr, my_head) + pw;
  if (rescale) {
#pragma unroll
    for (int h = 0; h < (int)kGroup; ++h)
#pragma unroll
      for (int e = 0; e < kVec; ++e) st.acc[h][e] *= corr[h];
  }
  x_row[lane] = pw;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  float pv[kLpr];
#pragma unroll
  for (int i = 0; i < kLpr; i += 4) {
    const float4 t4 = *reinterpret_cast<const float4*>(&x_row[ri * kLpr + i]);
    pv[i] = t4.x; pv[i + 1] = t4.y; pv[i + 2] = t4.z; pv[i + 3] = t4.w;
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int i = 0; i < kNi; ++i) {
    const float vf[kVec] = {__uint_as_float(vr[i].x), __uint_as_float(vr[i].y), __uint_as_float(vr[i].z),
                            __uint_as_float(vr[i].w)};
#pragma unroll
    for (int h = 0; h < (int)kGroup; ++h) {
      const float w = pv[i * kGroup + h];
#pragma unroll
      for (int e = 0; e < kVec; ++e) st.acc[h][e] = fmaf(w, vf[e], st.acc[h][e]);
    }
  }
}

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// A workgroup barrier that orders LDS only: the wavefront's LDS operations complete, global loads and stores stay in
// flight. `__syncthreads()` also waits for every outstanding global access (`vmcnt(0)`); at a piece's end that is the
// round trip of its output stores and of the ring's loads past the piece's last group, none of which the barrier
// protects. The empty asm's memory clobber keeps the compiler from moving memory operations across it.
__device__ __forceinline__ void LdsBarrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0); vmcnt and expcnt left at their maxima
  asm volatile("s_barrier" ::: "memory");
}

// Split-K paged decode of f32 caches. kFastPage: page_size is a multiple of 16, so a 16-token group (16-aligned within its
// sequence) lies in one page and its page id is one wave-uniform scalar load; otherwise each lane looks its own
// token's page up. Loads are branch-free (an absent key reads a valid address and is masked) and the next group's
// K/V is fetched into a second register buffer while the current group is computed. Workgroup (range, KV head)
// processes the pieces of its range in turn; a piece that is not a whole sequence writes fp32 partials that
// DecodeMergeKernel combines in key order.
template <int D, bool kFastPage>
__global__ void __launch_bounds__(256, kDecodeWgsPerCu)
    DecodeF32Kernel(const float* __restrict__ q, float* __restrict__ out, float* __restrict__ lse, KvView kv,
                    const int32_t* __restrict__ kv_indices, const DecodeWork* __restrict__ work,
                    const int32_t* __restrict__ range_ptr, float* __restrict__ part_o, float* __restrict__ part_ml,
                    const int32_t* __restrict__ q_rows, uint32_t q_heads, uint32_t heads_per_wg, float scale_log2,
                    int32_t window, uint32_t causal, SoftCap cap) {
  using C = DecodeCfg<D>;
  constexpr int kVec = C::kVec, kLpr = C::kLpr, kTpi = C::kTpi, kNi = C::kNi;
  constexpr int kWaves = 4;
  __shared__ float x_lds[kWaves][64];
  __shared__ float m_lds[kWaves * kGroup];
  __shared__ float l_lds[kWaves * kGroup];
  __shared__ float o_lds[kWaves * kGroup * D];

  // Both KV heads of a range are adjacent in launch order, so the two halves of each NHD page row are read together.
  // A workgroup serves heads_per_wg (1, 2 or 4) KV heads of one range, 4 / heads_per_wg wavefronts per head, so the
  // KV heads of each page row (adjacent in an NHD pool) are read by one CU at the same time.
  const uint32_t hblocks = kv.vheads / heads_per_wg;
  const uint32_t range = blockIdx.x / hblocks;
  const int lane = threadIdx.x & 63;
  // The wavefront index is uniform within a wavefront; saying so lets the group's page id be a scalar load.
  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t kvh = (blockIdx.x % hblocks) * heads_per_wg + wave_id % heads_per_wg;
  const int wave = wave_id / static_cast<int>(heads_per_wg);           // index among this head's wavefronts
  const int waves_per_head = kWaves / static_cast<int>(heads_per_wg);
  const int r = lane % kLpr;   // which 16-byte slice of a row
  const int ri = lane / kLpr;  // which row of a wave-wide load
  const int kperm = r / static_cast<int>(kGroup);  // this lane's token-slot permutation for K
  const float* kbase = static_cast<const float*>(kv.k);
  const float* vbase = static_cast<const float*>(kv.v);

  const int32_t it_end = range_ptr[range + 1];
  for (int32_t it = range_ptr[range]; it < it_end; ++it) {
  const DecodeWork wk = work[it];
  int32_t p0 = 0;
  const uint32_t kv_len = SeqKvLen(kv, wk.seq, &p0);
  // The row's query token: its sequence's index in a decode call; in a prefill call q_back tokens before the
  // sequence's last, q_indptr[seq + 1] - 1 (the last token; the only one of a single-token sequence).
  // (Clamped into the sequence's own rows, so that device tables that disagree with the plan cannot move it outside.)
  const uint64_t tok = q_rows != nullptr
                           ? static_cast<uint64_t>(max(q_rows[wk.seq], q_rows[wk.seq + 1] - 1 - wk.q_back))
                           : static_cast<uint64_t>(wk.seq);
  // The query's position; it sees keys up to itself (causal) or all of them, and from its window start on.
  const int32_t qpos = static_cast<int32_t>(kv_len) - 1 - wk.q_back;
  const uint32_t t_begin = static_cast<uint32_t>(wk.token_begin);
  uint32_t t_end = min(kv_len, static_cast<uint32_t>(wk.token_end));
  if (causal) t_end = min(t_end, static_cast<uint32_t>(max(0, qpos + 1)));
  // The sliding window's first visible key; the piece may start up to 15 keys before it, which are masked.
  const uint32_t lo = window < 0 || kv_len == 0 ? 0u : static_cast<uint32_t>(max(0, qpos - window));

  float qr[kGroup][kVec];
  {
    const float* qrow = q + (tok * q_heads + kvh * kGroup) * D + r * kVec;
#pragma unroll
    for (int h = 0; h < (int)kGroup; ++h) {
      const float4 v = *reinterpret_cast<const float4*>(qrow + (h ^ (r & 3)) * D);
      qr[h][0] = v.x; qr[h][1] = v.y; qr[h][2] = v.z; qr[h][3] = v.w;
    }
  }

  DecodeState<D> st;
#pragma unroll
  for (int h = 0; h < (int)kGroup; ++h) {
    st.m[h] = -INFINITY;
#pragma unroll
    for (int e = 0; e < kVec; ++e) st.acc[h][e] = 0.0f;
  }
  st.l_lane = 0.0f;

  // Byte stride between the rows of consecutive tokens of one KV head inside a page.
  const uint32_t tok_bytes = (kv.hnd ? D : kv.kv_heads * D) * 4;
  // Group gi (0-based, 16 tokens) of this wavefront: key g = t_begin + 16 * (wave + waves_per_head * gi).
  const uint32_t ngroups = (t_end > t_begin) ? (t_end - t_begin + 15) / 16 : 0;
  const uint32_t nw = ngroups > static_cast<uint32_t>(wave)
                          ? (ngroups - wave + waves_per_head - 1) / waves_per_head : 0;
  // Every load is unconditional: a group index past the end is clamped to the wave's last group and its keys are
  // masked, so the number of loads in flight is the same on every path and the compiler can wait for exactly the
  // current group's data (vmcnt) while the next group's loads stay in flight.
  constexpr bool kZeroGroup = D <= 128;
  // Absent tokens read the V row of their group's first visible token. A group without any reads kZeroRow, or at head dim
  // 256, where the registers spill and the further address costs more (16 contexts around 4,000: 203 -> 224 us; 209 as it
  // is), is not computed.
  auto load = [&](uint32_t gi, uint4* kr, uint4* vr, uint32_t& valid) {
    valid = 0;
    const uint32_t g0 = t_begin + 16u * (wave + waves_per_head * min(gi, nw - 1));
    const bool live = gi < nw;
    if constexpr (kFastPage) {
      const uint32_t pi = g0 / kv.page_size;
      const uint32_t off0 = g0 - pi * kv.page_size;
      const int32_t page = kv_indices[p0 + pi];  // uniform address: a scalar load
      const bool page_ok = page >= 0 && static_cast<uint64_t>(page) < kv.pool_pages;
      const uint64_t pg = page_ok ? static_cast<uint64_t>(page) : 0;
      const uint32_t kvr = kvh >> kv.head_shift;  // the real KV head this group of query heads reads
      const uint64_t row0 = kv.hnd ? (pg * kv.kv_heads + kvr) * kv.page_size + off0
                                   : (pg * kv.page_size + off0) * kv.kv_heads + kvr;
      const char* kg = reinterpret_cast<const char*>(kbase + row0 * D);
      const uint32_t n = page_ok ? min(16u, t_end - g0) : 0u;
      const bool any = page_ok && max(lo, g0) < min(g0 + 16u, t_end);  // a visible token in the group
      const uint32_t first = any ? max(lo, g0) - g0 : 0;
      const uint32_t visible = any ? ((1u << n) - 1u) & ~((1u << first) - 1u) : 0u;  // bit t: token t
      const char* vg = reinterpret_cast<const char*>(vbase + row0 * D);
      if (kZeroGroup && !any) vg = reinterpret_cast<const char*>(kZeroRow);
#pragma unroll
      for (int i = 0; i < kNi; ++i) {
        const uint32_t tv = i * kTpi + ri;  // V register i: slot i
        const bool okv = kZeroGroup ? ((visible >> tv) & 1u) != 0 && live
                                    : live && page_ok && g0 + tv < t_end && g0 + tv >= lo;
        vr[i] = LoadStream16(vg + ((okv ? tv : first) * tok_bytes + r * 16));
        const uint32_t tk = (i ^ kperm) * kTpi + ri;  // K register i: slot i ^ kperm
        const uint32_t row = kZeroGroup ? min(tk, max(n, 1u) - 1) : (page_ok && g0 + tk < t_end ? tk : 0);
        kr[i] = LoadStream16(kg + (row * tok_bytes + r * 16));
        valid |= static_cast<uint32_t>(okv) << i;
      }
    } else {
#pragma unroll
      for (int i = 0; i < kNi; ++i) {
        bool okk, okv;
        const int32_t tk = static_cast<int32_t>(g0 + (i ^ kperm) * kTpi + ri);
        const uint64_t rowk = KeyRowSafe<D>(kv, p0, tk, static_cast<int32_t>(t_end), kvh, &okk);
        const uint64_t rowv = KeyRowSafe<D>(kv, p0, static_cast<int32_t>(g0 + i * kTpi + ri),
                                            static_cast<int32_t>(t_end), kvh, &okv);
        okv = okv && g0 + i * kTpi + ri >= lo;
        kr[i] = *reinterpret_cast<const uint4*>(kbase + rowk + r * kVec);
        vr[i] = LoadStream16((okv ? vbase + rowv : reinterpret_cast<const float*>(kZeroRow)) + r * kVec);
        valid |= static_cast<uint32_t>(okv && live) << i;
      }
    }
  };

  if (nw > 0) {
    // A ring of kDecodeRing register buffers: group gi is computed while groups gi+1 .. gi+kDecodeRing-1 are in
    // flight (kDecodeRing - 1 groups of 16 loads stay below the 63 outstanding vector loads a wavefront can count).
    uint4 kbuf[kDecodeRing][kNi], vbuf[kDecodeRing][kNi];
    uint32_t valid[kDecodeRing];
#pragma unroll
    for (int s = 0; s < kDecodeRing - 1; ++s) load(s, kbuf[s], vbuf[s], valid[s]);
    for (uint32_t gi = 0; gi < nw; gi += kDecodeRing) {
#pragma unroll
      for (int s = 0; s < kDecodeRing; ++s) {
        constexpr int kLast = kDecodeRing - 1;
        const int nxt = (s + kLast) % kDecodeRing;
        load(gi + s + kLast, kbuf[nxt], vbuf[nxt], valid[nxt]);
        if (gi + s < nw && (kZeroGroup || !kFastPage || __any(valid[s] != 0))) {
          DecodeGroup<D>(st, kbuf[s], vbuf[s], valid[s], qr, x_lds[wave_id], r, ri, lane, scale_log2, cap);
        }
      }
    }
  }

  // Wave: fold the row groups (lanes sharing r) and total the per-lane denominators per head.
#pragma unroll
  for (int mk = kLpr; mk < 64; mk <<= 1)
#pragma unroll
    for (int h = 0; h < (int)kGroup; ++h)
#pragma unroll
      for (int e = 0; e < kVec; ++e) st.acc[h][e] += ShflXor(st.acc[h][e], mk);
  // Per-lane denominators: lanes with r % 4 == h hold head h.
  float lsum = st.l_lane;
#pragma unroll
  for (int mk = 4; mk < 64; mk <<= 1) lsum += ShflXor(lsum, mk);
  if (lane < (int)kGroup) {
    m_lds[wave_id * kGroup + lane] = Pick4(st.m, lane);
    l_lds[wave_id * kGroup + lane] = lsum;  // lane h holds the total of head h
  }
  if (ri == 0) {
#pragma unroll
    for (int h = 0; h < (int)kGroup; ++h)
#pragma unroll
      for (int e = 0; e < kVec; ++e) o_lds[(wave_id * kGroup + h) * D + r * kVec + e] = st.acc[h][e];
  }
  LdsBarrier();

  // Workgroup: merge the wavefronts of each KV head, then write the final row or this piece's partial.
  const int split = wk.slot;
  for (int idx = threadIdx.x; idx < (int)(heads_per_wg * kGroup * D); idx += 64 * kWaves) {
    const int hk = idx / (kGroup * D);  // local KV head: wavefronts hk, hk + heads_per_wg, ...
    const int h = (idx / D) % kGroup;
    const int d = idx % D;
    float M = -INFINITY;
    for (int w = hk; w < kWaves; w += heads_per_wg) M = fmaxf(M, m_lds[w * kGroup + h]);
    float o = 0.0f, L = 0.0f;
    for (int w = hk; w < kWaves; w += heads_per_wg) {
      const float f = m_lds[w * kGroup + h] == -INFINITY ? 0.0f : exp2f(m_lds[w * kGroup + h] - M);
      o += o_lds[(w * kGroup + h) * D + d] * f;
      L += l_lds[w * kGroup + h] * f;
    }
    const uint32_t qh = ((blockIdx.x % hblocks) * heads_per_wg + hk) * kGroup + h;
    if (split < 0) {
      const uint64_t row = tok * q_heads + qh;
      out[row * D + d] = GateOut<float>(kv.out_gate, row * D + d, L > 0.0f ? o / L : 0.0f);
      if (lse != nullptr && d == 0) lse[row] = L > 0.0f ? M + log2f(L) : -INFINITY;
    } else {
      const uint64_t prow = static_cast<uint64_t>(split) * q_heads + qh;
      part_o[prow * D + d] = o;
      if (d == 0) {
        part_ml[prow * 2] = M;
        part_ml[prow * 2 + 1] = L;
      }
    }
  }
  LdsBarrier();  // the next piece reuses the LDS merge buffers
  }
}


// ---- bf16 decode kernel ----------------------------------------------------------------------------------------------
//
// A wavefront serves all NH = 4, 8 or 16 query heads of a KV head (padded to 16) and both products run on matrix
// instructions, with no exchange of the weights between lanes. Per group of 16 tokens, lane (c = lane % 16, g = lane / 16):
//   * q.k on v_mfma_f32_16x16x32_bf16 (tokens on M, heads on N): the lane gets the scores of tokens 4g .. 4g + 3 for head c;
//   * its four weights, packed, are the A operand (heads on M, tokens 4g + i in k-slots 4g + i) of
//     v_mfma_f32_16x16x16_bf16;
//   * it loads the D / 16 dims of slice c of tokens 4g .. 4g + 3 (whole rows per 16 lanes), and pairs of those rows
//     interleaved with v_perm are the B operands: one multiply per dim e of the slice gives heads 4g + j, dim (c, e).
// The running maximum is the exact one, so a head's largest weight is 1, which bf16 holds: kept up to 2^8 below the scores
// (as the prefill kernels do), it let a dominant weight be rounded where its denominator was not, and a whole peaked row
// came out up to 2^-8 off, or infinite for V past 1e36. It moves in a wavefront's first groups and rarely later; only then
// are a head's rescale factors brought to the lanes holding its sums.
//
// Bound by HBM. One register buffer each for a group's K and V rows: the next group's K rows are requested once the
// scores have read these, its V rows once P.V has, so one of the two is in flight at all times. Two buffers of each
// (the next group requested before this one is computed) were slower: 73 against 67 us at 16 heads over 2, head dim
// 256, 324 MB (they spill there), 113 against 112 at 32 over 4, head dim 128. V, read in whole rows, and K at head dims
// 64 and 128 take the non-temporal hint (V plain: 110 against 101 us at 8 over 2, head dim 256, 579 MB); K at 256, where
// an instruction reads half of each 128-byte line, is faster without (101 against 102.4).
// Measured against groups of 4 heads on v_dot2 with a double buffer, whose larger groups requested the rows again for
// every 4 heads (contexts cold): 8 over 2, 256: 107 -> 101 us (5.7 TB/s); 32 over 8, 128: 115 -> 107; 16 over 4, 64:
// 82 -> 72; 32 over 4, 128 (642 MB): 168 -> 112; 32 over 2, 128: 134 -> 64; 32 over 2, 256: 155 -> 74.
typedef short i16x4v_t __attribute__((ext_vector_type(4)));

template <int D, int NH, bool kFastPage, int kWaves>
__device__ __forceinline__ void DecodeMfmaBody(const uint16_t* __restrict__ q, uint16_t* __restrict__ out,
                                               float* __restrict__ lse, KvView kv,
                                               const int32_t* __restrict__ kv_indices,
                                               const DecodeWork* __restrict__ work,
                                               const int32_t* __restrict__ range_ptr, float* __restrict__ part_o,
                                               float* __restrict__ part_ml, const int32_t* __restrict__ q_rows,
                                               uint32_t q_heads, uint32_t heads_per_wg, float scale_log2,
                                               int32_t window, uint32_t causal, SoftCap cap, uint32_t block,
                                               float* m_lds, float* l_lds, float* o_lds) {
  // LDS (the caller's): m_lds and l_lds [kWaves][NH], o_lds [kWaves][NH][D] floats. kv.vheads and kv.head_shift count
  // groups of NH query heads.
  constexpr int kKc = D / 32;                // K operands (16 bytes per lane) of a group
  constexpr int kSlice = D >= 128 ? 8 : 4;   // dims of one V load per lane
  constexpr int kVh = D / 16 / kSlice;       // V loads per token: the row in kVh parts of 16 slices
  constexpr bool kQLds = D == 256 && NH > 4;
  static_assert(!kQLds || NH * D * 4 >= 64 * 16 * kKc, "q fits in the wavefront's share of o_lds");
  typedef uint32_t vword_t __attribute__((ext_vector_type(kSlice / 2)));

  const uint32_t hblocks = kv.vheads / heads_per_wg;
  const uint32_t range = block / hblocks;
  const int lane = threadIdx.x & 63;
  const int wave_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t kvh = (block % hblocks) * heads_per_wg + wave_id % heads_per_wg;
  const int wave = wave_id / static_cast<int>(heads_per_wg);
  const int waves_per_head = kWaves / static_cast<int>(heads_per_wg);
  const int c = lane & 15, g = lane >> 4;
  const uint16_t* kbase = static_cast<const uint16_t*>(kv.k);
  const uint16_t* vbase = static_cast<const uint16_t*>(kv.v);

  const int32_t it_end = range_ptr[range + 1];
  for (int32_t it = range_ptr[range]; it < it_end; ++it) {
    const DecodeWork wk = work[it];
    int32_t p0 = 0;
    const uint32_t kv_len = SeqKvLen(kv, wk.seq, &p0);
    // The row's query token and the keys it sees, as in DecodeF32Kernel.
    const uint64_t tok = q_rows != nullptr
                             ? static_cast<uint64_t>(max(q_rows[wk.seq], q_rows[wk.seq + 1] - 1 - wk.q_back))
                             : static_cast<uint64_t>(wk.seq);
    const int32_t qpos = static_cast<int32_t>(kv_len) - 1 - wk.q_back;
    const uint32_t t_begin = static_cast<uint32_t>(wk.token_begin);
    uint32_t t_end = min(kv_len, static_cast<uint32_t>(wk.token_end));
    if (causal) t_end = min(t_end, static_cast<uint32_t>(max(0, qpos + 1)));
    const uint32_t lo = window < 0 || kv_len == 0 ? 0u : static_cast<uint32_t>(max(0, qpos - window));

    // B operand of q.k: head c's dims 32 kc + 8 g .. +8 (columns past NH repeat the heads; their results are not used).
    // At head dim 256 it is kept in this wavefront's share of o_lds and read per group: in registers it spilled 48.
    u32x4_t qb[kQLds ? 1 : kKc];
    auto* q_lds = reinterpret_cast<u32x4_t*>(o_lds + wave_id * NH * D) + lane;
    {
      const uint16_t* qrow = q + (tok * q_heads + kvh * NH + c % NH) * D + g * 8;
#pragma unroll
      for (int kc = 0; kc < kKc; ++kc) {
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(qrow + kc * 32);
        if constexpr (kQLds) q_lds[64 * kc] = v; else qb[kc] = v;
      }
    }
    f32x4_t acc[D / 16];  // acc[kSlice * h + e][j]: head 4g + j, dim 16 kSlice h + kSlice c + e
#pragma unroll
    for (int e = 0; e < D / 16; ++e) acc[e] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    float m_run = -INFINITY;  // head c's running maximum (the same in the four lanes of a head)
    float l_lane = 0.0f;      // this lane's share of head c's denominator

    const uint32_t tok_bytes = (kv.hnd ? D : kv.kv_heads * D) * 2;
    const uint32_t ngroups = (t_end > t_begin) ? (t_end - t_begin + 15) / 16 : 0;
    const uint32_t nw = ngroups > static_cast<uint32_t>(wave)
                            ? (ngroups - wave + waves_per_head - 1) / waves_per_head : 0;
    // Where group gi (16 tokens) of this wavefront lies: key g0 = t_begin + 16 (wave + waves_per_head gi). A group past
    // the end is the last one again with no valid key, so that every load is unconditional.
    struct Place {
      uint64_t row;    // element offset of its first token's row; of token c's row when the group may cross pages
      uint32_t g0;
      uint32_t valid;  // bit t: token t is a real key of the window
      bool page_ok;    // its page id lies in the pool (a group in one page)
    };
    auto place = [&](uint32_t gi) {
      Place a;
      a.g0 = t_begin + 16u * (wave + waves_per_head * min(gi, nw - 1));
      if constexpr (kFastPage) {
        const uint32_t pi = a.g0 / kv.page_size;
        const uint32_t off0 = a.g0 - pi * kv.page_size;
        const int32_t page = kv_indices[p0 + pi];  // uniform address: a scalar load
        a.page_ok = page >= 0 && static_cast<uint64_t>(page) < kv.pool_pages;
        const uint64_t pg = a.page_ok ? static_cast<uint64_t>(page) : 0;
        const uint32_t kvr = kvh >> kv.head_shift;
        a.row = (kv.hnd ? (pg * kv.kv_heads + kvr) * kv.page_size + off0
                        : (pg * kv.page_size + off0) * kv.kv_heads + kvr) * D;
        const uint32_t n = gi < nw && a.page_ok ? min(16u, t_end - a.g0) : 0u;
        a.valid = (1u << n) - 1u;
      } else {
        bool ok;
        a.row = KeyRowSafe<D>(kv, p0, static_cast<int32_t>(a.g0 + c), static_cast<int32_t>(t_end), kvh, &ok);
        a.page_ok = true;
        a.valid = static_cast<uint32_t>(__ballot(ok && gi < nw)) & 0xFFFFu;  // lanes 0..15 hold tokens 0..15
      }
      if (a.g0 < lo) a.valid &= ~((1u << min(16u, lo - a.g0)) - 1u);  // before the window
      return a;
    };
    // Rows of absent tokens: K reads the group's first (general pages: the pool's first), whose score is masked. V reads
    // the group's first visible token's, since a weight of 0 times a row that nobody wrote may be NaN; a group without a
    // visible token is not folded.
    auto load_k = [&](const Place& a, u32x4_t* kr) {
      const char* kg = reinterpret_cast<const char*>(kbase + a.row);
      const uint32_t ko = (kFastPage && a.page_ok && a.g0 + c < t_end ? c : 0) * tok_bytes + g * 16;
#pragma unroll
      for (int i = 0; i < kKc; ++i) {
        const auto* kp = reinterpret_cast<const u32x4_t*>(kg + (ko + i * 64));
        kr[i] = D <= 128 ? __builtin_nontemporal_load(kp) : *kp;
      }
    };
    auto load_v = [&](const Place& a, vword_t (*vr)[4]) {
      const uint32_t first = a.valid != 0 ? __builtin_ctz(a.valid) : 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t tv = ((a.valid >> (4 * g + i)) & 1u) ? 4 * g + i : first;
        uint64_t row = a.row;
        uint32_t vo = c * (2 * kSlice);
        if constexpr (kFastPage) {
          vo += tv * tok_bytes;
        } else {
          bool ok;
          row = KeyRowSafe<D>(kv, p0, static_cast<int32_t>(a.g0 + tv), static_cast<int32_t>(t_end), kvh, &ok);
        }
        const char* vg = reinterpret_cast<const char*>(vbase + row);
#pragma unroll
        for (int h = 0; h < kVh; ++h) {
          vr[h][i] = __builtin_nontemporal_load(reinterpret_cast<const vword_t*>(vg + (vo + h * 32 * kSlice)));
        }
      }
    };
    auto scores = [&](const u32x4_t* kr) {
      f32x4_t s = {0.0f, 0.0f, 0.0f, 0.0f};
      int again = 0;
      if constexpr (kQLds) asm volatile("" : "+v"(again));  // keeps the reads in the loop
#pragma unroll
      for (int kc = 0; kc < kKc; ++kc) {
        u32x4_t qv;
        if constexpr (kQLds) qv = q_lds[64 * kc + again]; else qv = qb[kc];
        s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, kr[kc]),
                                                    __builtin_bit_cast(bf16x8_t, qv), s, 0, 0, 0);
      }
      return s;
    };
    auto fold = [&](f32x4_t s, const vword_t (*vr)[4], uint32_t valid) {
      float mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float y = s[j] * scale_log2;
        if (cap.capl != 0.0f) y = Capped(y, cap);
        s[j] = ((valid >> (4 * g + j)) & 1u) ? y : -INFINITY;
        mx = fmaxf(mx, s[j]);
      }
      mx = fmaxf(mx, ShflXor(mx, 16));
      mx = MaxXor32(mx);
      if (__any(mx > m_run)) {
        const float m_new = fmaxf(m_run, mx);
        const float corr = m_run == -INFINITY ? 0.0f : exp2f(m_run - m_new);
        l_lane *= corr;
        m_run = m_new;
        float cj[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) cj[j] = __shfl(corr, 4 * g + j, 64);  // lane h holds head h
#pragma unroll
        for (int e = 0; e < D / 16; ++e)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[e][j] *= cj[j];
      }
      const float m_use = m_run == -INFINITY ? 0.0f : m_run;  // a head with no visible key yet keeps p = 0
      float p[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) p[j] = __builtin_amdgcn_exp2f(s[j] - m_use);
      l_lane += (p[0] + p[1]) + (p[2] + p[3]);
      const i16x4v_t pa = __builtin_bit_cast(i16x4v_t, u32x2_t{PackRne(p[0], p[1]), PackRne(p[2], p[3])});
#pragma unroll
      for (int h = 0; h < kVh; ++h)
#pragma unroll
        for (int w = 0; w < kSlice / 2; ++w) {
          const u32x2_t b0{__builtin_amdgcn_perm(vr[h][1][w], vr[h][0][w], 0x05040100u),
                           __builtin_amdgcn_perm(vr[h][3][w], vr[h][2][w], 0x05040100u)};
          const u32x2_t b1{__builtin_amdgcn_perm(vr[h][1][w], vr[h][0][w], 0x07060302u),
                           __builtin_amdgcn_perm(vr[h][3][w], vr[h][2][w], 0x07060302u)};
          const int e = kSlice * h + 2 * w;
          acc[e] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pa, __builtin_bit_cast(i16x4v_t, b0), acc[e], 0, 0, 0);
          acc[e + 1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(pa, __builtin_bit_cast(i16x4v_t, b1), acc[e + 1], 0, 0, 0);
        }
    };

    if (nw > 0) {
      u32x4_t kr[kKc];
      vword_t vr[kVh][4];
      Place cur = place(0);
      load_k(cur, kr);
      load_v(cur, vr);
      for (uint32_t gi = 0; gi < nw; ++gi) {
        const Place nxt = place(gi + 1);
        const f32x4_t s = scores(kr);
        __builtin_amdgcn_sched_barrier(0);  // the next K rows are requested as soon as the scores have read these
        load_k(nxt, kr);
        if (cur.valid != 0) fold(s, vr, cur.valid);
        __builtin_amdgcn_sched_barrier(0);
        load_v(nxt, vr);
        cur = nxt;
      }
    }

    float lsum = l_lane + ShflXor(l_lane, 16);
    lsum = SumXor32(lsum);
    if (lane < NH) {
      m_lds[wave_id * NH + lane] = m_run;
      l_lds[wave_id * NH + lane] = lsum;
    }
    if (4 * g < NH) {
#pragma unroll
      for (int h = 0; h < kVh; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int e = 0; e < kSlice; ++e)
            o_lds[(wave_id * NH + 4 * g + j) * D + 16 * kSlice * h + kSlice * c + e] = acc[kSlice * h + e][j];
    }
    LdsBarrier();

    // Workgroup: merge the wavefronts of each KV head, then write the final row or this piece's partial (four dims per
    // thread: a head's weights are formed once for the four).
    const int split = wk.slot;
    for (int idx = threadIdx.x; idx < (int)(heads_per_wg * NH * D / 4); idx += 64 * kWaves) {
      const int hk = idx / (NH * D / 4);
      const int h = (idx / (D / 4)) % NH;
      const int d = 4 * (idx % (D / 4));
      float M = -INFINITY;
      for (int w = hk; w < kWaves; w += heads_per_wg) M = fmaxf(M, m_lds[w * NH + h]);
      f32x4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
      float L = 0.0f;
      for (int w = hk; w < kWaves; w += heads_per_wg) {
        const float f = m_lds[w * NH + h] == -INFINITY ? 0.0f : exp2f(m_lds[w * NH + h] - M);
        o += *reinterpret_cast<const f32x4_t*>(&o_lds[(w * NH + h) * D + d]) * f;
        L += l_lds[w * NH + h] * f;
      }
      const uint32_t qh = ((block % hblocks) * heads_per_wg + hk) * NH + h;
      if (split < 0) {
        const uint64_t row = tok * q_heads + qh;
        const float inv = L > 0.0f ? 1.0f / L : 0.0f;  // four divisions: 2% of a call of one-group contexts
        const u32x2_t v{PackBf16(o[0] * inv, o[1] * inv), PackBf16(o[2] * inv, o[3] * inv)};
        *reinterpret_cast<u32x2_t*>(out + row * D + d) = GateOut2(kv.out_gate, row * D + d, v);
        if (lse != nullptr && d == 0) lse[row] = L > 0.0f ? M + log2f(L) : -INFINITY;
      } else {
        const uint64_t prow = static_cast<uint64_t>(split) * q_heads + qh;
        *reinterpret_cast<f32x4_t*>(part_o + prow * D + d) = o;
        if (d == 0) {
          part_ml[prow * 2] = M;
          part_ml[prow * 2 + 1] = L;
        }
      }
    }
    LdsBarrier();  // the next piece reuses the LDS merge buffers
  }
}

template <int D, int NH, bool kFastPage>
__global__ void __launch_bounds__(256, kDecodeWgsPerCu)
    DecodeMfmaKernel(const uint16_t* __restrict__ q, uint16_t* __restrict__ out, float* __restrict__ lse, KvView kv,
                     const int32_t* __restrict__ kv_indices, const DecodeWork* __restrict__ work,
                     const int32_t* __restrict__ range_ptr, float* __restrict__ part_o, float* __restrict__ part_ml,
                     const int32_t* __restrict__ q_rows, uint32_t q_heads, uint32_t heads_per_wg, float scale_log2,
                     int32_t window, uint32_t causal, SoftCap cap) {
  __shared__ float m_lds[4][NH];
  __shared__ float l_lds[4][NH];
  __shared__ __attribute__((aligned(16))) float o_lds[4][NH][D];
  DecodeMfmaBody<D, NH, kFastPage, 4>(q, out, lse, kv, kv_indices, work, range_ptr, part_o, part_ml, q_rows, q_heads,
                                      heads_per_wg, scale_log2, window, causal, cap, blockIdx.x, &m_lds[0][0],
                                      &l_lds[0][0], &o_lds[0][0][0]);
}

// Combines the pieces of each split sequence: one workgroup per (sequence, query head) of D threads, four slices of D / 4
// threads. Slice s sums pieces s, s + 4, ... (four dims per thread, several pieces' loads in flight), wavefront 0 forms the
// per-piece rescale factors meanwhile, and the slices are added in order through LDS: a fixed order, so deterministic.
// Latency bound: one element per thread and one dependent load per piece past the 16th took 9.8 us on 94 pieces
// (the call over one context of 1,500 16.2 -> 13.5 us, three around 2,500 24.2 -> 22.4).
struct DecodeMergeArgs {
  const DecodeMerge* merges;
  const float* part_o;
  const float* part_ml;
  const int32_t* q_rows;  // the call's q_indptr in a prefill call, NULL in a decode call
};

template <typename T, int D>
__device__ __forceinline__ void DecodeMergeBody(T* __restrict__ out, float* __restrict__ lse, const DecodeMergeArgs& m,
                                                uint32_t q_heads, const void* out_gate, uint32_t bx) {
  constexpr int kSlices = 4;
  __shared__ float f_lds[kMaxMergeSplits];
  __shared__ float inv_lds;
  __shared__ __attribute__((aligned(16))) float o_lds[kSlices][D];
  const float* __restrict__ part_o = m.part_o;
  const float* __restrict__ part_ml = m.part_ml;
  const int32_t* __restrict__ q_rows = m.q_rows;
  const DecodeMerge mg = m.merges[bx / q_heads];
  const uint64_t tok = q_rows != nullptr
                           ? static_cast<uint64_t>(max(q_rows[mg.seq], q_rows[mg.seq + 1] - 1 - mg.q_back))
                           : static_cast<uint64_t>(mg.seq);
  const uint32_t qh = bx % q_heads;
  const int n = min(mg.count, static_cast<int32_t>(kMaxMergeSplits));
  const uint64_t base = static_cast<uint64_t>(mg.first) * q_heads + qh;  // partial row of piece c: base + c * q_heads
  // The first kPre pieces of every slice are requested before the weights, which are formed while they arrive.
  constexpr int kPre = 4;
  const int slice = threadIdx.x / (D / 4), d4 = 4 * (threadIdx.x % (D / 4));
  const float* po = part_o + base * D + d4;
  const uint64_t step = static_cast<uint64_t>(q_heads) * D;
  auto piece = [&](int c) { return *reinterpret_cast<const f32x4_t*>(po + min(c, n - 1) * step); };
  const uint64_t e = (tok * q_heads + qh) * D + threadIdx.x;
  const T gv = GateFetch<T>(out_gate, e);  // requested with the partials, applied at the end
  f32x4_t pre[kPre];
#pragma unroll
  for (int c = 0; c < kPre; ++c) pre[c] = piece(slice + kSlices * c);
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    // Piece `lane` (and lane + 64, ... for longer splits): its max and sum, read once.
    const float m0 = lane < n ? part_ml[(base + static_cast<uint64_t>(lane) * q_heads) * 2] : -INFINITY;
    const float l0 = lane < n ? part_ml[(base + static_cast<uint64_t>(lane) * q_heads) * 2 + 1] : 0.0f;
    float M = m0;
    for (int c = lane + 64; c < n; c += 64) M = fmaxf(M, part_ml[(base + static_cast<uint64_t>(c) * q_heads) * 2]);
    for (int mk = 32; mk >= 1; mk >>= 1) M = fmaxf(M, __shfl_xor(M, mk, 64));
    float L = 0.0f;
    if (lane < n) {
      const float f = m0 == -INFINITY ? 0.0f : exp2f(m0 - M);
      f_lds[lane] = f;
      L = l0 * f;
    }
    for (int c = lane + 64; c < n; c += 64) {
      const uint64_t prow = base + static_cast<uint64_t>(c) * q_heads;
      const float mc = part_ml[prow * 2];
      const float f = mc == -INFINITY ? 0.0f : exp2f(mc - M);
      f_lds[c] = f;
      L += part_ml[prow * 2 + 1] * f;
    }
    for (int mk = 32; mk >= 1; mk >>= 1) L += __shfl_xor(L, mk, 64);
    if (lane == 0) {
      inv_lds = L > 0.0f ? 1.0f / L : 0.0f;
      if (lse != nullptr) lse[tok * q_heads + qh] = L > 0.0f ? M + log2f(L) : -INFINITY;
    }
  }
  __syncthreads();
  f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
  auto add = [&](f32x4_t x, int c) {
    if (c >= n) return;
    const float f = f_lds[c];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = fmaf(x[i], f, acc[i]);
  };
#pragma unroll
  for (int c = 0; c < kPre; ++c) add(pre[c], slice + kSlices * c);
  for (int c0 = slice + kSlices * kPre; c0 < n; c0 += kSlices * kPre) {
#pragma unroll
    for (int c = 0; c < kPre; ++c) pre[c] = piece(c0 + kSlices * c);
#pragma unroll
    for (int c = 0; c < kPre; ++c) add(pre[c], c0 + kSlices * c);
  }
  *reinterpret_cast<f32x4_t*>(&o_lds[slice][d4]) = acc;
  __syncthreads();
  const int d = threadIdx.x;
  const float o = (o_lds[0][d] + o_lds[1][d]) + (o_lds[2][d] + o_lds[3][d]);
  out[e] = GateApply<T>(out_gate, gv, Narrow<T>(o * inv_lds));
}

template <typename T, int D>
__global__ void __launch_bounds__(D) DecodeMergeKernel(T* __restrict__ out, float* __restrict__ lse, DecodeMergeArgs m,
                                                       uint32_t q_heads, const void* out_gate) {
  DecodeMergeBody<T, D>(out, lse, m, q_heads, out_gate, blockIdx.x);
}

// ---- Prefill kernel (bf16, head_dim 256, MFMA) -----------------------------------------------------------------------

constexpr int kPD = 256;                 // head_dim
constexpr int kKStride = kPD + 8;        // K tile row stride in LDS (elements): 528 bytes
constexpr int kVtStride = kPrefillTileK + 8;  // V^T tile row stride (elements): 144 bytes

__device__ __forceinline__ f32x16_t Mfma32(const u32x4_t& a, const u32x4_t& b, const f32x16_t& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                 0, 0);
}

__global__ void __launch_bounds__(256, 1)
    PrefillKernel(const uint16_t* __restrict__ q, uint16_t* __restrict__ out, float* __restrict__ lse, KvView kv,
                  const int32_t* __restrict__ q_indptr, const PrefillWork* __restrict__ work, uint32_t q_heads,
                  uint32_t causal, float scale_log2, int32_t window, SoftCap cap) {
  __shared__ __attribute__((aligned(16))) uint16_t k_lds[kPrefillTileK * kKStride];
  __shared__ __attribute__((aligned(16))) uint16_t vt_lds[kPD * kVtStride];

  const PrefillWork wk = work[blockIdx.x];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int hl = lane >> 5;   // half of the wave
  const int col = lane & 31;  // MFMA N index: this lane's query within the tile
  const uint32_t kvh = static_cast<uint32_t>(wk.kv_head);
  const uint32_t head = kvh * kGroup + wave;
  const uint16_t* kbase = static_cast<const uint16_t*>(kv.k);
  const uint16_t* vbase = static_cast<const uint16_t*>(kv.v);

  int32_t p0 = 0;
  const uint32_t kv_len = SeqKvLen(kv, wk.seq, &p0);
  const int32_t qbeg = q_indptr[wk.seq];
  const int32_t n = q_indptr[wk.seq + 1] - qbeg;
  const int32_t q0 = wk.q0;
  const int32_t rows = wk.rows;
  // Key position of this lane's query, and of the tile's first / last query.
  const int32_t base_pos = static_cast<int32_t>(kv_len) - n + q0;
  const int32_t my_pos = base_pos + col;
  int32_t key_end = static_cast<int32_t>(kv_len);
  if (causal) key_end = min(key_end, base_pos + rows);  // last query sees keys <= base_pos + rows - 1
  if (key_end < 0) key_end = 0;

  // Q^T operand: lane holds q[query col][ks*16 + hl*8 .. +8] for ks = 0..15.
  u32x4_t qreg[16];
  {
    const bool ok = col < rows;
    const uint16_t* qrow = q + (static_cast<uint64_t>(qbeg + q0 + (ok ? col : 0)) * q_heads + head) * kPD + hl * 8;
#pragma unroll
    for (int ks = 0; ks < 16; ++ks) {
      qreg[ks] = ok ? *reinterpret_cast<const u32x4_t*>(qrow + ks * 16) : u32x4_t{0, 0, 0, 0};
    }
  }

  f32x16_t o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[dt][v] = 0.0f;
  float m_run = -INFINITY;
  float l_run = 0.0f;

  // K/V of the next 64-key tile are fetched into registers while the current tile is computed (software pipeline).
  u32x4_t kpre[8];
  u32x4_t vpre[2][4];
  auto fetch = [&](int32_t kb) {
    const u32x4_t zero{0, 0, 0, 0};
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int vi = tid + 256 * it;
      bool ok;
      const uint64_t row = KeyRowSafe<kPD>(kv, p0, kb + (vi >> 5), key_end, kvh, &ok);
      const u32x4_t x = *reinterpret_cast<const u32x4_t*>(kbase + row + (vi & 31) * 8);
      kpre[it] = ok ? x : zero;
    }
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int vi = tid + 256 * it;  // 16 groups of 4 keys x 32 slices of 8 dims
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        bool ok;
        const uint64_t row = KeyRowSafe<kPD>(kv, p0, kb + (vi >> 5) * 4 + t, key_end, kvh, &ok);
        const u32x4_t x = *reinterpret_cast<const u32x4_t*>(vbase + row + (vi & 31) * 8);
        vpre[it][t] = ok ? x : zero;
      }
    }
  };
  // With a window the tile's first query (position base_pos) sees keys from base_pos - window on; keys before that
  // are never read.
  const int32_t key_beg = window < 0 ? 0 : min(max(0, base_pos - window), key_end);
  if (key_end > key_beg) fetch(key_beg);

  for (int32_t kb = key_beg; kb < key_end; kb += kPrefillTileK) {
    __syncthreads();  // every wavefront is done reading the previous tile
    // K row-major; V transposed: 4 keys x 8 dims become 8 rows (dims) of 4 keys.
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int vi = tid + 256 * it;
      *reinterpret_cast<u32x4_t*>(&k_lds[(vi >> 5) * kKStride + (vi & 31) * 8]) = kpre[it];
    }
#pragma unroll
    for (int it = 0; it < 2; ++it) {
      const int vi = tid + 256 * it;
      const int kg = vi >> 5;
      const int c = vi & 31;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int w = e >> 1;
        uint32_t k01, k23;
        if ((e & 1) == 0) {
          k01 = (vpre[it][0][w] & 0xFFFFu) | (vpre[it][1][w] << 16);
          k23 = (vpre[it][2][w] & 0xFFFFu) | (vpre[it][3][w] << 16);
        } else {
          k01 = (vpre[it][0][w] >> 16) | (vpre[it][1][w] & 0xFFFF0000u);
          k23 = (vpre[it][2][w] >> 16) | (vpre[it][3][w] & 0xFFFF0000u);
        }
        *reinterpret_cast<u32x2_t*>(&vt_lds[(c * 8 + e) * kVtStride + kg * 4]) = u32x2_t{k01, k23};
      }
    }
    __syncthreads();
    if (kb + static_cast<int32_t>(kPrefillTileK) < key_end) fetch(kb + kPrefillTileK);

    // S^T = K Q^T for two 32-key halves: lane holds keys 8i + 4hl + jj of half kt for query col.
    f32x16_t s[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int v = 0; v < 16; ++v) s[kt][v] = 0.0f;
#pragma unroll
      for (int ks = 0; ks < 16; ++ks) {
        const u32x4_t a = *reinterpret_cast<const u32x4_t*>(&k_lds[(kt * 32 + col) * kKStride + ks * 16 + hl * 8]);
        s[kt] = Mfma32(a, qreg[ks], s[kt]);
      }
    }
    // Scale, mask, online softmax for this lane's query.
    const bool need_mask = (kb + static_cast<int32_t>(kPrefillTileK) > key_end) ||
                           (causal && kb + static_cast<int32_t>(kPrefillTileK) - 1 > base_pos) ||
                           (window >= 0 && kb < base_pos + rows - 1 - window);
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int32_t key = kb + kt * 32 + (v >> 2) * 8 + hl * 4 + (v & 3);
        float x = s[kt][v] * scale_log2;
        if (cap.capl != 0.0f) x = Capped(x, cap);
        if (need_mask && (key >= key_end || (causal && key > my_pos) || (window >= 0 && key < my_pos - window))) {
          x = -INFINITY;
        }
        s[kt][v] = x;
        mx = fmaxf(mx, x);
      }
    mx = MaxXor32(mx);
    // Lazy rescaling: the running max only moves when a score exceeds it by more than 2^8, so P stays below 256 (safe
    // in fp32 and bf16) and the O accumulators are rescaled on a handful of tiles instead of every tile.
    const bool grow = mx > m_run + 8.0f;
    if (__any(grow)) {
      const float m_new = grow ? mx : m_run;
      const float corr = m_run == -INFINITY ? 0.0f : exp2f(m_run - m_new);
      l_run *= corr;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[dt][v] *= corr;
      m_run = m_new;
    }
    const float m_use = m_run == -INFINITY ? 0.0f : m_run;  // a query with no visible key yet keeps p = 0
    float psum = 0.0f;
    u32x4_t pb[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int kt = c >> 1;
      const int i0 = (c & 1) * 2;
      float pf[8];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        pf[t] = exp2f(s[kt][i0 * 4 + t] - m_use);
        pf[4 + t] = exp2f(s[kt][(i0 + 1) * 4 + t] - m_use);
      }
#pragma unroll
      for (int t = 0; t < 8; ++t) psum += pf[t];
      pb[c] = u32x4_t{PackBf16(pf[0], pf[1]), PackBf16(pf[2], pf[3]), PackBf16(pf[4], pf[5]), PackBf16(pf[6], pf[7])};
    }
    l_run += psum;
    // O^T += V^T P^T: A = V^T rows (dims) with the keys in the order the P^T operand holds them.
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint16_t* vrow = &vt_lds[(dt * 32 + col) * kVtStride + c * 16 + hl * 4];
        const u32x2_t lo = *reinterpret_cast<const u32x2_t*>(vrow);
        const u32x2_t hi = *reinterpret_cast<const u32x2_t*>(vrow + 8);
        o[dt] = Mfma32(u32x4_t{lo[0], lo[1], hi[0], hi[1]}, pb[c], o[dt]);
      }
    }
  }

  // Normalise and write: lane holds dims dt*32 + 8i + 4hl + jj of query col.
  const float l_tot = SumXor32(l_run);
  if (col < rows) {
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    const uint64_t orow = (static_cast<uint64_t>(qbeg + q0 + col) * q_heads + head) * kPD;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = dt * 32 + i * 8 + hl * 4;
        const u32x2_t w{PackBf16(o[dt][i * 4] * inv, o[dt][i * 4 + 1] * inv),
                        PackBf16(o[dt][i * 4 + 2] * inv, o[dt][i * 4 + 3] * inv)};
        *reinterpret_cast<u32x2_t*>(out + orow + d) = GateOut2(kv.out_gate, orow + d, w);
      }
    if (lse != nullptr && hl == 0) {
      lse[static_cast<uint64_t>(qbeg + q0 + col) * q_heads + head] = l_tot > 0.0f ? m_run + log2f(l_tot) : -INFINITY;
    }
  }
}

// ---- Prefill kernel for page sizes that are multiples of 16 (bf16, head_dim 64/128/256, MFMA, DMA-fed) --------------
//
// One workgroup = 64 query tokens x the 4 query heads of one KV head, 8 wavefronts (two per SIMD, so one wavefront's
// softmax runs under the other's MFMAs): wavefront w is query head 4 kvh + (w & 3) for tokens 32 (w >> 2) .. +31.
// Per 64-key tile each wavefront copies 8 K rows and a quarter of the V tile (16-aligned groups of rows never straddle
// a page when the page size is a multiple of 16) from the paged cache straight into LDS with global_load_lds,
// double-buffered, so the copy of tile t + 1 runs under the products of tile t. The tile is consumed in two 32-key
// halves:
//   S^T = K Q^T  (v_mfma_f32_32x32x16_bf16; K rows from LDS as the A operand, Q^T held in registers as B),
//   online softmax per query (lane pair l, l ^ 32 holds one query's 32 scores; lazy rescaling: the running max only
//   moves when a score exceeds it by more than 2^8, so P stays below 256),
//   O^T += V^T P^T (V^T operands read from the V tile with ds_read_b64_tr_b16, P^T from registers).
// ds_read_b64_tr_b16 works within groups of 16 lanes: output lane 4a + b, element e, is element b of the 8 bytes that
// lane 4e + a addressed. So when lane 4e + a of a group addresses keys k0 + e, dims d0 + 4a .. +3, output lane j of the
// group receives V[k0 + e][d0 + j], e = 0..3: a V^T operand row.
// K rows are 512 bytes in LDS with 16-byte pieces at swizzled positions: piece p of row r at p ^ (r & 15) (the A-operand
// reads of 16 consecutive rows hit 16 distinct bank groups). The V tile is stored in the order the transposed reads
// consume it: 1 KB block (c16, dt) holds keys 16 c16 .. +15 x dims 32 dt .. +31, each read instruction takes one
// contiguous 512-byte half of a block (conflict-free, and every read is one base register plus an immediate). Each
// copy instruction then fetches 16 rows x 64 bytes; storing K the same way (32 rows x 32 bytes per copy) was measured
// 8% slower overall, the copy's wider spread of cache lines costing more than the cheaper reads gain.

typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) unsigned char lds_byte_t;

__device__ __forceinline__ uint32_t LdsAddr(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((const lds_byte_t*)p));
}

// global -> LDS copy of 16 bytes per lane (lane l lands at lds + 16 l; lds wave-uniform), from inline assembly so that
// the compiler does not make every later LDS access wait on it; the kernel waits for it itself. M0 is restored.
__device__ __forceinline__ void Dma16(const void* g, uint32_t lds) {
  uint32_t save;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
               : "=&s"(save) : "v"(g), "s"(lds));
}

// The same with a wave-uniform 64-bit base in SGPRs and a 32-bit per-lane byte offset.
__device__ __forceinline__ void Dma16(const void* sbase, uint32_t voff, uint32_t lds) {
  uint32_t save;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
               : "=&s"(save) : "v"(voff), "s"(sbase), "s"(lds));
}

// Both copies again with an immediate byte offset kOff (below 4096) on the global address. The instruction adds its
// offset to the LDS address as well, so M0 is set to lds - kOff and the 16 bytes of lane l still land at lds + 16 l.
template <int kOff>
__device__ __forceinline__ void Dma16At(const void* sbase, uint32_t voff, uint32_t lds) {
  uint32_t save;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\tglobal_load_lds_dwordx4 %1, %2 offset:%4\n\ts_mov_b32 m0, %0"
               : "=&s"(save) : "v"(voff), "s"(sbase), "s"(lds - kOff), "i"(kOff));
}

template <int kN, typename F>
__device__ __forceinline__ void StaticFor(F&& f) {
  if constexpr (kN > 0) {
    StaticFor<kN - 1>(f);
    f(std::integral_constant<int, kN - 1>{});
  }
}

__device__ __forceinline__ void WaitVmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0) only

__device__ __forceinline__ u32x2_t LdsTr16(const unsigned char* base, uint32_t off) {
  auto* ptr = reinterpret_cast<__attribute__((address_space(3))) i16x4_t*>(
      const_cast<lds_byte_t*>((const lds_byte_t*)base + off));
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16(ptr));
}


// Head dims 256, 128 and 64: a row is 2 D bytes = D / 8 16-byte pieces (32, 16 or 8). K pieces are swizzled by the
// row index modulo min(16, D / 8), which keeps every swizzled piece inside its row and any 8 consecutive rows (the
// lanes one LDS read cycle serves) on distinct 16-byte bank groups; the V offsets (at most 12 pieces) stay inside a row.
// kCap: the call caps its logits; `cap` is then the cap in the kernel's unscaled score units (the log2-unit cap divided
// by scale_log2, its slope multiplied by it), so that a capped score stays unscaled like an uncapped one. A separate
// instantiation keeps the cap's registers out of the uncapped kernel, which otherwise spills at head dim 256.
template <int D>
constexpr int kPfTileBytes = kPrefillTileK * 2 * D;  // one 64-key K or V tile in LDS

// Row `prow` (counted over all slots of `rows` rows) of the fp32 partials, which follow the splits_bf16 slots of bf16 rows.
__device__ __forceinline__ float* PartRowF32(uint16_t* part_o, uint32_t splits_bf16, uint64_t prow, uint32_t rows, int d) {
  const uint64_t first = static_cast<uint64_t>(splits_bf16) * rows;
  return reinterpret_cast<float*>(part_o + first * d) + (prow - first) * d;
}

// The tile kernel's work for item `item`; `tiles` is the caller's LDS, [2 buffers][K, V][kPfTileBytes<D>].
template <int D, bool kCap, int kWaves>
__device__ __forceinline__ void PrefillTileBody(const uint16_t* __restrict__ q, uint16_t* __restrict__ out,
                                                float* __restrict__ lse, KvView kv,
                                                const int32_t* __restrict__ kv_indices,
                                                const int32_t* __restrict__ q_indptr,
                                                const PrefillWork* __restrict__ work, uint16_t* __restrict__ part_o,
                                                float* __restrict__ part_ml, uint32_t splits_bf16, uint32_t q_heads,
                                                uint32_t causal, uint32_t ps_shift, float scale_log2, int32_t window,
                                                SoftCap cap, uint32_t item, unsigned char (*tiles)[2][kPfTileBytes<D>]) {
  static_assert(D == 64 || D == 128 || D == 256, "the tile kernel is built for head dims 64, 128 and 256");
  constexpr int kRowB = 2 * D;                  // bytes of one K or V row in LDS
  constexpr int kPieces = D / 8;                // 16-byte pieces per row
  constexpr int kRowsPerDma = 1024 / kRowB;     // rows one 64-lane global_load_lds_dwordx4 fills
  constexpr int kKs = D / 16;                   // K = 16 steps of S^T = K Q^T
  constexpr int kDt = D / 32;                   // 32-dim blocks of O^T
  constexpr int kNv = kDt / 2;                  // V blocks each wavefront copies per tile (4 kDt blocks / 8)
  constexpr int kSw = (kPieces < 16 ? kPieces : 16) - 1;  // K swizzle mask
  constexpr uint32_t kRows = 32 * kWaves;       // query rows of an item (8 kWaves tokens x kGroup heads)

  const PrefillWork wk = work[item];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hq = w & 3;       // query head within the KV head's group
  const int qt = w >> 2;      // 32-token half of the item
  const int hl = lane >> 5;   // half of the wave: MFMA k-slot group
  const int col = lane & 31;  // MFMA N index: this lane's query within the wavefront's 32
  const uint32_t kvh = static_cast<uint32_t>(wk.kv_head);
  const uint32_t head = kvh * kGroup + hq;
  const uint16_t* kbase = static_cast<const uint16_t*>(kv.k);
  const uint16_t* vbase = static_cast<const uint16_t*>(kv.v);
  const uint32_t ps = kv.page_size;  // a power of two, 1 << ps_shift

  int32_t p0 = 0;
  const uint32_t kv_len = SeqKvLen(kv, wk.seq, &p0);
  const int32_t qbeg = q_indptr[wk.seq];
  const int32_t n = q_indptr[wk.seq + 1] - qbeg;
  const int32_t r = 32 * qt + col;  // this lane's query within the item
  const bool row_ok = r < wk.rows;
  const int32_t last_pos = static_cast<int32_t>(kv_len) - n + wk.q0 + 32 * qt + 31;  // the wavefront's last query
  // The item's key range by the device's lengths: keys up to its last query (causal) or all keys, from its first
  // query's window start rounded down to 16. The plan's cuts between pieces stay; the outer bounds follow the device.
  const int32_t dev_first = static_cast<int32_t>(kv_len) - n + wk.q0;  // the item's first query position
  const int32_t dev_end = max(0, causal ? min(static_cast<int32_t>(kv_len), dev_first + wk.rows)
                                        : static_cast<int32_t>(kv_len));
  const int32_t dev_beg = window < 0 ? 0 : (max(0, dev_first - window) & ~15);
  const int32_t kbeg = (wk.ends & kPieceFirst) ? dev_beg : wk.kbeg;
  const int32_t kend = (wk.ends & kPieceLast) ? dev_end : min(wk.kend, dev_end);
  const int ntiles = kend > kbeg ? (kend - kbeg + 63) / 64 : 0;

  // Q^T operands: qreg[ks] = q[query r][dims 16 ks + 8 hl .. +8].
  u32x4_t qreg[kKs];
  {
    const uint16_t* qrow = q + (static_cast<uint64_t>(qbeg + wk.q0 + (row_ok ? r : 0)) * q_heads + head) * D + hl * 8;
#pragma unroll
    for (int ks = 0; ks < kKs; ++ks) {
      const u32x4_t x = *reinterpret_cast<const u32x4_t*>(qrow + ks * 16);
      qreg[ks] = row_ok ? x : u32x4_t{0, 0, 0, 0};
    }
  }

  // Page ids of the four 16-row groups of tile t (rows clamped into the item's keys); loaded one tile before the
  // copy that needs them, so the scalar loads never stall the loop.
  // With 16-token pages, a tile wholly inside the key range takes its four ids as one 16-byte scalar load of
  // consecutive page-table entries (all of them exist: the sequence has a page for every key below kend).
  auto load_ids = [&](int t, int32_t (&ids)[4]) {
    const int32_t kb = kbeg + 64 * t;
    if (ps_shift == 4 && kb + 64 <= kend) {
      int4 v;
      __builtin_memcpy(&v, kv_indices + p0 + (kb >> 4), sizeof(v));
      ids[0] = v.x;
      ids[1] = v.y;
      ids[2] = v.z;
      ids[3] = v.w;
    } else {
#pragma unroll
      for (int g = 0; g < 4; ++g) ids[g] = kv_indices[p0 + (min(kb + 16 * g, kend - 1) >> ps_shift)];
    }
  };
  // id in [0, pool_pages) as one unsigned 32-bit compare (pool page counts above 2^31 - 1 are clamped: ids are int32).
  const uint32_t pool32 = static_cast<uint32_t>(min(kv.pool_pages, static_cast<uint64_t>(0x7FFFFFFF)));
  auto good_page = [&](int32_t id) { return static_cast<uint32_t>(id) < pool32; };
  // Element offsets inside a page: a row at in-page position `within` starts at row_mul * within + row_add.
  const uint32_t row_mul = kv.hnd ? D : kv.kv_heads * D;
  const uint32_t kvr = kvh >> kv.head_shift;  // the real KV head the item's query heads read
  const uint32_t row_add = kv.hnd ? kvr * ps * D : kvr * D;
  const uint64_t page_elems = static_cast<uint64_t>(ps) * kv.kv_heads * D;
  // This wavefront's share of the copy of tile t: K rows 8w .. 8w + 7 (kRowsPerDma rows per instruction) and kNv
  // blocks of V.
  auto issue = [&](int t, int buf, const int32_t (&ids)[4], int ln) {
    if (kWaves > 8 && w >= 8) return;  // the first 8 wavefronts copy
    const int32_t kb = kbeg + 64 * t;
    const int32_t pos0 = kb + 8 * w;  // this wavefront's first row; all 8 lie in one page
    const int32_t id = ids[w >> 1];
    const uint64_t pg = good_page(id) ? static_cast<uint64_t>(id) : 0;  // a bad page's rows are masked, not read
    const int32_t page_first = min(pos0, kend - 1) & ~((1 << ps_shift) - 1);
    const uint16_t* kpage = kbase + pg * page_elems + row_add;
    const uint32_t kdst = LdsAddr(tiles[buf][0]) + 8 * w * kRowB;
    const int c = ln % kPieces, hh = ln / kPieces;
#pragma unroll
    for (int i = 0; i < 8 / kRowsPerDma; ++i) {
      const int rr = kRowsPerDma * i + hh;  // row 8w + rr of the tile
      const uint32_t within = static_cast<uint32_t>(min(pos0 + rr, kend - 1) - page_first);
      const uint32_t off = 2 * row_mul * within;
      const uint32_t kp = 16 * static_cast<uint32_t>(c ^ ((8 * w + rr) & kSw));
      Dma16(kpage, off + kp, kdst + i * 1024);
    }
    {  // V blocks (c16, dt0 + i): lane ln fetches key 16 c16 + 8 hi + 4 ((mm >> 4) & 1) + ((mm & 7) >> 1),
       // dims 32 (dt0 + i) + 16 ((mm >> 3) & 1) + 8 (mm & 1); the block's 16 keys lie in one page
      const int mm = ln & 31, hi = ln >> 5;
      const int c16 = w >> 1, dt0 = (w & 1) * kNv;
      const int32_t vid = ids[c16];
      const uint16_t* vpage = vbase + (good_page(vid) ? static_cast<uint64_t>(vid) : 0) * page_elems + row_add;
      const int key = 16 * c16 + 8 * hi + 4 * ((mm >> 4) & 1) + ((mm & 7) >> 1);
      const uint32_t within = static_cast<uint32_t>(min(kb + key, kend - 1)) & ((1u << ps_shift) - 1);
      const uint32_t voff = 2 * (row_mul * within + 32 * dt0 + 16 * ((mm >> 3) & 1) + 8 * (mm & 1));
      const uint32_t dst = LdsAddr(tiles[buf][1]) + 1024 * (c16 * kDt + dt0);
      StaticFor<kNv>([&](auto i) { Dma16At<64 * i.value>(vpage, voff, dst + 1024 * i.value); });
    }
  };

  f32x16_t o[kDt];
#pragma unroll
  for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[dt][v] = 0.0f;
  float m_run = -INFINITY;
  float l_run = 0.0f;

  int32_t ids_cur[4] = {0, 0, 0, 0}, ids_nxt[4] = {0, 0, 0, 0};
  if (ntiles > 0) {
    load_ids(0, ids_cur);
    issue(0, 0, ids_cur, lane);
    load_ids(min(1, ntiles - 1), ids_nxt);
  }
  for (int t = 0; t < ntiles; ++t) {
    const int buf = t & 1;
    WaitVmem();       // this wavefront's copies of tile t have landed
    __syncthreads();  // ... and everyone's; everyone is also done reading the other buffer
    // Every lane-dependent value the loop needs is re-derived here from the thread index, so that only the index
    // stays live across the loop (the register budget at two wavefronts per SIMD holds nothing more).
    int tx = static_cast<int>(threadIdx.x);
    asm volatile("" : "+v"(tx));
    const int ln = tx & 63, lc = ln & 31, lh = ln >> 5;
    if (t + 1 < ntiles) issue(t + 1, buf ^ 1, ids_nxt, ln);
    uint32_t bad = 0;  // 16-key groups of this tile whose page id lies outside the pool
#pragma unroll
    for (int g = 0; g < 4; ++g) bad |= good_page(ids_cur[g]) ? 0u : (1u << g);
#pragma unroll
    for (int g = 0; g < 4; ++g) ids_cur[g] = ids_nxt[g];
    load_ids(min(t + 2, ntiles - 1), ids_nxt);
    const int32_t kb = kbeg + 64 * t;
    // K operand: row 32 half + lc, piece 2 ks + lh at position (2 ks + lh) ^ (lc & kSw) (32 half keeps row & kSw =
    // lc & kSw); in bytes 16 ((2 ks + lh) ^ (lc & kSw)) = 32 ks ^ 16 (lh ^ (lc & kSw)).
    const int krow = lc * kRowB, kx = 16 * (lh ^ (lc & kSw));
    // V^T operands, read transposed: in lane group g = ln / 16, lane j = ln % 16 addresses key +(j / 4) at dims
    // +4 (j % 4), keys based at 16 c16 + 4 (g >> 1) (+8 for the operand's second half), dims at 32 dt + 16 (g & 1);
    // block (c16, dt) of the V tile holds exactly those 8 bytes at 8 ln (and the second half's at 512 + 8 ln).
    const int32_t qpos = static_cast<int32_t>(kv_len) - n + wk.q0 + 32 * qt + lc;  // this lane's query position
    // Every term is wave-uniform; readfirstlane says so, so that the masking below is skipped by a scalar branch
    // instead of running under an empty exec mask on every tile.
    const bool need_mask = __builtin_amdgcn_readfirstlane(
        static_cast<int>((kb + 64 > kend) | (causal && kb + 63 > last_pos - 31) | (bad != 0) |
                         (window >= 0 && kb < last_pos - window))) != 0;
    const unsigned char* ktile = tiles[buf][0];
    const unsigned char* vtile = tiles[buf][1];
    const unsigned char* vl = vtile + 8 * ln;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      // Keys after every query of the wavefront (uniform): nothing to add. Only the second half is left out: a test of the
      // first as well costs every tile more than it saves (chunks of 512 on 8,000 cached tokens, us, none / both / second:
      // 16 heads over 4 x 64 132 / 138 / 130, 32 over 8 x 128 330 / 334 / 326; four fresh prompts of 1,500 and 3,900 at 64
      // 48.0 / 46.4 / 46.2 and 173 / 175 / 170, of 3,900 at 128 530 / 527 / 522). At head dim 256 the branch costs more
      // registers than it saves work (8 ragged chunks on prefixes: 357 -> 365 us).
      if (D <= 128 && half == 1 && causal && kb + 32 > last_pos) break;
      f32x16_t sc;
#pragma unroll
      for (int v = 0; v < 16; ++v) sc[v] = 0.0f;
      const unsigned char* krow_p = ktile + 32 * half * kRowB + krow;
      constexpr int kRing = 2;  // K operands in flight ahead of the multiply that uses them
      u32x4_t ka[kRing];
#pragma unroll
      for (int j = 0; j < kRing; ++j) ka[j] = *reinterpret_cast<const u32x4_t*>(krow_p + ((32 * j) ^ kx));
#pragma unroll
      for (int ks = 0; ks < kKs; ++ks) {
        const u32x4_t a = ka[ks % kRing];
        if (ks + kRing < kKs) ka[ks % kRing] = *reinterpret_cast<const u32x4_t*>(krow_p + ((32 * (ks + kRing)) ^ kx));
        sc = Mfma32(a, qreg[ks], sc);
      }
      // Keep kRing operand reads in flight (left alone, the compiler waits out every read before its multiply at this
      // register budget): the reads of the first kRing steps, then one multiply and one read in turn.
      __builtin_amdgcn_sched_group_barrier(0x100, kRing, 0);
#pragma unroll
      for (int ks = 0; ks < kKs - kRing; ++ks) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, kRing, 0);
      if constexpr (kCap) {
#pragma unroll
        for (int v = 0; v < 16; ++v) sc[v] = Capped(sc[v], cap);
      }
      if (need_mask) {  // one uniform branch around branch-free selects
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int kk = 32 * half + (v >> 2) * 8 + lh * 4 + (v & 3);  // key within the tile
          const int32_t key = kb + kk;
          // Bitwise ors: no short-circuit branches (each would be an exec-mask change per score).
          const bool off = (key >= kend) | ((causal != 0) & (key > qpos)) | (((bad >> (kk >> 4)) & 1u) != 0) |
                           ((window >= 0) & (key < qpos - window));
          sc[v] = off ? -INFINITY : sc[v];
        }
      }
      float mx = -INFINITY;
#pragma unroll
      for (int v = 0; v < 16; ++v) mx = fmaxf(mx, sc[v]);
      mx = MaxXor32(mx);
      mx *= scale_log2;  // scores stay unscaled until the exponent: the scale is positive, so this is the scaled max
      const bool grow = mx > m_run + 8.0f;
      if (__any(grow)) {
        const float m_new = grow ? mx : m_run;
        const float corr = m_run == -INFINITY ? 0.0f : exp2f(m_run - m_new);
        l_run *= corr;
#pragma unroll
        for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
          for (int v = 0; v < 16; ++v) o[dt][v] *= corr;
        m_run = m_new;
      }
      const float m_use = m_run == -INFINITY ? 0.0f : m_run;
      float psum = 0.0f;
      u32x4_t pb[2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        float pf[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          pf[e] = __builtin_amdgcn_exp2f(fmaf(sc[(2 * c) * 4 + e], scale_log2, -m_use));
          pf[4 + e] = __builtin_amdgcn_exp2f(fmaf(sc[(2 * c + 1) * 4 + e], scale_log2, -m_use));
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) psum += pf[e];
        pb[c] = u32x4_t{PackRne(pf[0], pf[1]), PackRne(pf[2], pf[3]), PackRne(pf[4], pf[5]), PackRne(pf[6], pf[7])};
      }
      l_run += psum;
      // O^T += V^T P^T over this half's two 16-key steps.
      // V^T operands of the 16 multiplies (c, dt) in order, read kVRing ahead of use.
      constexpr int kVRing = 2;
      auto vread = [&](int j) {
        const int c = j / kDt, dt = j % kDt;
        const uint32_t off = 1024 * ((2 * half + c) * kDt + dt);
        const u32x2_t lo = LdsTr16(vl, off);
        const u32x2_t hi = LdsTr16(vl, off + 512);
        return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
      };
      u32x4_t va[kVRing];
#pragma unroll
      for (int j = 0; j < kVRing; ++j) va[j] = vread(j);
#pragma unroll
      for (int j = 0; j < 2 * kDt; ++j) {
        const u32x4_t av = va[j % kVRing];
        if (j + kVRing < 2 * kDt) va[j % kVRing] = vread(j + kVRing);
        o[j % kDt] = Mfma32(av, pb[j / kDt], o[j % kDt]);
      }
    }
  }

  // Lane holds dims 32 dt + 8 i + 4 hl + jj of query r.
  const float l_tot = SumXor32(l_run);
  if (!row_ok) return;
  const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
  if (wk.slot >= 0) {  // a piece of a split item: its normalised output and its (max, sum)
    const uint64_t prow = static_cast<uint64_t>(wk.slot) * kRows + static_cast<uint64_t>(r) * kGroup + hq;
    if (static_cast<uint32_t>(wk.slot) < splits_bf16) {
      uint16_t* po = part_o + prow * D;
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int d = dt * 32 + i * 8 + hl * 4;
          const u32x2_t v{PackRne(o[dt][i * 4] * inv, o[dt][i * 4 + 1] * inv),
                          PackRne(o[dt][i * 4 + 2] * inv, o[dt][i * 4 + 3] * inv)};
          *reinterpret_cast<u32x2_t*>(po + d) = v;
        }
    } else {
      float* po = PartRowF32(part_o, splits_bf16, prow, kRows, D);
#pragma unroll
      for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4_t v{o[dt][i * 4] * inv, o[dt][i * 4 + 1] * inv, o[dt][i * 4 + 2] * inv, o[dt][i * 4 + 3] * inv};
          *reinterpret_cast<f32x4_t*>(po + dt * 32 + i * 8 + hl * 4) = v;
        }
    }
    if (hl == 0) {
      part_ml[2 * prow] = m_run;
      part_ml[2 * prow + 1] = l_tot;
    }
    return;
  }
  const uint64_t orow = (static_cast<uint64_t>(qbeg + wk.q0 + r) * q_heads + head) * D;
#pragma unroll
  for (int dt = 0; dt < kDt; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = dt * 32 + i * 8 + hl * 4;
      const u32x2_t v{PackRne(o[dt][i * 4] * inv, o[dt][i * 4 + 1] * inv),
                      PackRne(o[dt][i * 4 + 2] * inv, o[dt][i * 4 + 3] * inv)};
      *reinterpret_cast<u32x2_t*>(out + orow + d) = GateOut2(kv.out_gate, orow + d, v);
    }
  if (lse != nullptr && hl == 0) {
    lse[static_cast<uint64_t>(qbeg + wk.q0 + r) * q_heads + head] = l_tot > 0.0f ? m_run + log2f(l_tot) : -INFINITY;
  }
}


template <int D, bool kCap, int kWaves>
__global__ void __launch_bounds__(64 * kWaves, 1)
    PrefillTileKernel(const uint16_t* __restrict__ q, uint16_t* __restrict__ out, float* __restrict__ lse, KvView kv,
                      const int32_t* __restrict__ kv_indices, const int32_t* __restrict__ q_indptr,
                      const PrefillWork* __restrict__ work, uint16_t* __restrict__ part_o, float* __restrict__ part_ml,
                      uint32_t splits_bf16, uint32_t q_heads, uint32_t causal, uint32_t ps_shift, float scale_log2,
                      int32_t window, SoftCap cap) {
  __shared__ __attribute__((aligned(16))) unsigned char tiles[2][2][kPfTileBytes<D>];  // [buffer][K, V]
  PrefillTileBody<D, kCap, kWaves>(q, out, lse, kv, kv_indices, q_indptr, work, part_o, part_ml, splits_bf16, q_heads,
                                   causal, ps_shift, scale_log2, window, cap, blockIdx.x, tiles);
}

// A mixed step's attention in one launch: workgroups [0, items) run the tile pieces, the rest the decode ranges with 8
// wavefronts each (one range of one KV-head block per CU, 8 / heads_per_wg wavefronts per head). Tile workgroups come
// first in launch order, so they take their CUs before the decode ranges fill the others. Both kinds use the one LDS
// buffer in their own layout (a decode workgroup needs far less than a tile one, and neither shares its CU).
// NH: query heads of a decode wavefront (DecodeGroupOf); dec_vheads and dec_shift are the decode side's KvView fields.
template <int D, int NH>
constexpr int kMixedDecodeLds = 4 * (2 * kMixedDecodeWaves * NH + kMixedDecodeWaves * NH * D);

template <int D, bool kCap, int NH>
__global__ void __launch_bounds__(512, 1)
    MixedAttentionKernel(const uint16_t* __restrict__ q, uint16_t* __restrict__ out, float* __restrict__ lse,
                         KvView kv, const int32_t* __restrict__ kv_indices, const int32_t* __restrict__ q_indptr,
                         const PrefillWork* __restrict__ work, uint16_t* __restrict__ part_o,
                         float* __restrict__ part_ml, uint32_t splits_bf16, uint32_t q_heads, uint32_t causal,
                         uint32_t ps_shift, float scale_log2, int32_t window, SoftCap raw_cap, uint32_t items,
                         const DecodeWork* __restrict__ dec_work, const int32_t* __restrict__ dec_range_ptr,
                         float* __restrict__ dec_part_o, float* __restrict__ dec_part_ml, uint32_t heads_per_wg,
                         uint32_t dec_vheads, uint32_t dec_shift, SoftCap cap) {
  constexpr int kTileLds = 2 * 2 * kPfTileBytes<D>;
  constexpr int kLds = kTileLds > kMixedDecodeLds<D, NH> ? kTileLds : kMixedDecodeLds<D, NH>;
  __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];
  if (blockIdx.x < items) {
    PrefillTileBody<D, kCap, 8>(q, out, lse, kv, kv_indices, q_indptr, work, part_o, part_ml, splits_bf16, q_heads,
                                causal, ps_shift, scale_log2, window, raw_cap, blockIdx.x,
                                reinterpret_cast<unsigned char (*)[2][kPfTileBytes<D>]>(lds));
    return;
  }
  constexpr int W = kMixedDecodeWaves;
  kv.vheads = dec_vheads;
  kv.head_shift = dec_shift;
  float* m_lds = reinterpret_cast<float*>(lds);
  float* l_lds = m_lds + W * NH;
  float* o_lds = l_lds + W * NH;
  DecodeMfmaBody<D, NH, true, W>(q, out, lse, kv, kv_indices, dec_work, dec_range_ptr, dec_part_o, dec_part_ml, q_indptr,
                                 q_heads, heads_per_wg, scale_log2, window, causal, cap, blockIdx.x - items, m_lds,
                                 l_lds, o_lds);
}

// Combines the pieces of a split prefill item: block (merge, group of kRows tokens) of kGroup * D / 4 threads; thread t
// handles query head t / (D / 4), dims 4 (t % (D / 4)) .. +3 of each of the group's tokens. Pieces are combined in
// key order (deterministic). Merges of two pieces (the plan puts them first) run 8 tokens per block with every load
// issued before any is combined; the others one token per block.
constexpr int kPfMergeRows = 8;

template <int D>
__device__ __forceinline__ void MergeWrite(uint16_t* __restrict__ out, float* __restrict__ lse, const void* gate,
                                           u32x2_t g, uint64_t token, uint32_t q_heads, uint32_t head, int d,
                                           float4 acc, float l, float mx) {
  const float inv = l > 0.0f ? 1.0f / l : 0.0f;
  const u32x2_t v{PackBf16(acc.x * inv, acc.y * inv), PackBf16(acc.z * inv, acc.w * inv)};
  const uint64_t e = (token * q_heads + head) * D + d;
  *reinterpret_cast<u32x2_t*>(out + e) = GateApply2(gate, g, v);
  if (lse != nullptr && d == 0) lse[token * q_heads + head] = l > 0.0f ? mx + log2f(l) : -INFINITY;
}

// acc += o * f for one piece's output slice (already divided by the piece's own sum), bf16 or fp32.
__device__ __forceinline__ void MergeAdd(float4& acc, f32x4_t o, float f) {
  acc.x = fmaf(o[0], f, acc.x);
  acc.y = fmaf(o[1], f, acc.y);
  acc.z = fmaf(o[2], f, acc.z);
  acc.w = fmaf(o[3], f, acc.w);
}
__device__ __forceinline__ void MergeAdd(float4& acc, u32x2_t raw, float f) {
  acc.x = fmaf(__uint_as_float(raw[0] << 16), f, acc.x);
  acc.y = fmaf(__uint_as_float(raw[0] & 0xFFFF0000u), f, acc.y);
  acc.z = fmaf(__uint_as_float(raw[1] << 16), f, acc.z);
  acc.w = fmaf(__uint_as_float(raw[1] & 0xFFFF0000u), f, acc.w);
}

// T: the type of the item's partial rows; part_o holds row 0 of slot 0 as if every slot were of that type.
template <typename T, int D, int kTokens, int kRows>
__device__ __forceinline__ void PrefillMergeRows(uint16_t* __restrict__ out, float* __restrict__ lse,
                                                 const PrefillMerge& mg, int r0, const T* __restrict__ part_o,
                                                 const float* __restrict__ part_ml,
                                                 const int32_t* __restrict__ q_indptr, uint32_t q_heads,
                                                 const void* gate) {
  using Slice = std::conditional_t<sizeof(T) == 2, u32x2_t, f32x4_t>;  // four dims
  if (r0 >= mg.rows) return;
  const int hq = threadIdx.x / (D / 4);
  const int d = 4 * (threadIdx.x % (D / 4));
  const uint32_t head = mg.kv_head * kGroup + hq;
  const uint64_t tok0 = static_cast<uint64_t>(q_indptr[mg.seq] + mg.q0);
  // Partial row of piece i for token row r: ((first + i) * kTokens + r) * kGroup + hq.
  auto prow = [&](int i, int r) {
    return ((static_cast<uint64_t>(mg.first) + i) * kTokens + r) * kGroup + hq;
  };
  if constexpr (kRows > 1) {  // merges of exactly two pieces
    float2 ml[kRows][2];
    Slice o[kRows][2];
    u32x2_t gw[kRows];
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      const int r = min(r0 + j, mg.rows - 1);  // rows past the item's end re-read its last row and are not written
      gw[j] = GateFetch2(gate, ((tok0 + r) * q_heads + head) * D + d);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        ml[j][i] = *reinterpret_cast<const float2*>(part_ml + 2 * prow(i, r));
        o[j][i] = *reinterpret_cast<const Slice*>(part_o + prow(i, r) * D + d);
      }
    }
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
      if (r0 + j >= mg.rows) break;
      const float mx = fmaxf(ml[j][0].x, ml[j][1].x);
      float l = 0.0f;
      float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (mx != -INFINITY) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          // The piece's weight is its sum rescaled to the common max (mx is finite here, so a piece without keys,
          // max -inf, gets exp2(-inf) = 0).
          const float f = ml[j][i].y * exp2f(ml[j][i].x - mx);
          l += f;
          MergeAdd(acc, o[j][i], f);
        }
      }
      MergeWrite<D>(out, lse, gate, gw[j], tok0 + r0 + j, q_heads, head, d, acc, l, mx);
    }
  } else {  // any count, one token row per block; the piece loops are unrolled so several pieces' loads are in flight
    const u32x2_t gw = GateFetch2(gate, ((tok0 + r0) * q_heads + head) * D + d);
    float mx = -INFINITY;
#pragma unroll 8
    for (int i = 0; i < mg.count; ++i) mx = fmaxf(mx, part_ml[2 * prow(i, r0)]);
    float l = 0.0f;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (mx != -INFINITY) {
#pragma unroll 4
      for (int i = 0; i < mg.count; ++i) {
        const float2 m = *reinterpret_cast<const float2*>(part_ml + 2 * prow(i, r0));
        const float f = m.y * exp2f(m.x - mx);
        l += f;
        MergeAdd(acc, *reinterpret_cast<const Slice*>(part_o + prow(i, r0) * D + d), f);
      }
    }
    MergeWrite<D>(out, lse, gate, gw, tok0 + r0, q_heads, head, d, acc, l, mx);
  }
}

// One launch for both forms: the first `two` merges (exactly two pieces) as blocks of kPfMergeRows token rows, the
// rest one token row per block (two merge launches one after the other cost a second launch's latency).
struct PrefillMergeArgs {
  const PrefillMerge* merges;
  const uint16_t* part_o;
  const float* part_ml;
  const int32_t* q_indptr;
  uint32_t splits_bf16;
  uint32_t two;     // merges of exactly two pieces, listed first
  uint32_t blocks;  // blocks of the launch's prefill share
};

template <int D, int kTokens>
__device__ __forceinline__ void PrefillMergeBody(uint16_t* __restrict__ out, float* __restrict__ lse,
                                                 const PrefillMergeArgs& m, uint32_t q_heads, const void* gate,
                                                 uint32_t b) {
  constexpr uint32_t kTwoBlocks = kTokens / kPfMergeRows;  // blocks per two-piece merge
  const uint32_t two = m.two;
  const bool pair = b < two * kTwoBlocks;
  const uint32_t k = b - two * kTwoBlocks;
  const PrefillMerge mg = m.merges[pair ? b / kTwoBlocks : two + k / kTokens];
  const int r0 = pair ? static_cast<int>(b % kTwoBlocks) * kPfMergeRows : static_cast<int>(k % kTokens);
  auto rows = [&](auto n, const auto* part_o, int first) {
    using T = std::remove_cv_t<std::remove_pointer_t<decltype(part_o)>>;
    PrefillMergeRows<T, D, kTokens, decltype(n)::value>(out, lse, mg, first, part_o, m.part_ml, m.q_indptr, q_heads, gate);
  };
  if (static_cast<uint32_t>(mg.first) < m.splits_bf16) {
    pair ? rows(std::integral_constant<int, kPfMergeRows>{}, m.part_o, r0)
         : rows(std::integral_constant<int, 1>{}, m.part_o, r0);
  } else {  // fp32 rows: half as many at a time, for the same registers
    const float* part_f = reinterpret_cast<const float*>(m.part_o) -
                          static_cast<uint64_t>(m.splits_bf16) * kTokens * kGroup * (D / 2);
    if (!pair) rows(std::integral_constant<int, 1>{}, part_f, r0);
    for (int h = 0; pair && h < 2; ++h) rows(std::integral_constant<int, kPfMergeRows / 2>{}, part_f, r0 + h * kPfMergeRows / 2);
  }
}

template <int D, int kTokens>
__global__ void __launch_bounds__(256) PrefillMergeKernel(uint16_t* __restrict__ out, float* __restrict__ lse,
                                                          PrefillMergeArgs m, uint32_t q_heads, const void* gate) {
  PrefillMergeBody<D, kTokens>(out, lse, m, q_heads, gate, blockIdx.x);
}

// A mixed step's two merges in one launch (both take D threads per block): the tile pieces' merge blocks first, then
// the decode ranges'. One launch instead of two saves the second's latency.
template <int D>
__global__ void __launch_bounds__(D) MixedMergeKernel(uint16_t* __restrict__ out, float* __restrict__ lse,
                                                      PrefillMergeArgs pm, DecodeMergeArgs dm, uint32_t q_heads,
                                                      const void* gate) {
  static_assert(kGroup * D / 4 == D, "a prefill merge block has D threads");
  if (blockIdx.x < pm.blocks) {
    PrefillMergeBody<D, kPfTokens>(out, lse, pm, q_heads, gate, blockIdx.x);
  } else {
    DecodeMergeBody<uint16_t, D>(out, lse, dm, q_heads, gate, blockIdx.x - pm.blocks);
  }
}

// The decode pieces' partials: fp32 rows (dec_splits x q_heads x D), then their (max, sum) pairs.
DecodeMergeArgs DecodeMergeArgsOf(const RoostPagedAttentionParams& p, const PlanRecord& rec, unsigned char* dev,
                                  uint32_t d) {
  DecodeMergeArgs m{};
  m.merges = reinterpret_cast<const DecodeMerge*>(dev + rec.dec_merge_offset);
  m.part_o = reinterpret_cast<const float*>(dev + rec.dec_float_offset);
  m.part_ml = m.part_o + rec.dec_splits * p.q_heads * d;
  m.q_rows = p.mode == ROOST_ATTENTION_PREFILL ? static_cast<const int32_t*>(p.q_indptr.address) : nullptr;
  return m;
}

template <typename T, int D>
RoostStatus LaunchDecodeMerge(const RoostPagedAttentionParams& p, const PlanRecord& rec, unsigned char* dev,
                              const KvView& kv, hipStream_t stream) {
  if (rec.dec_merges == 0) return ROOST_STATUS_OK;
  hipLaunchKernelGGL((DecodeMergeKernel<T, D>), dim3(static_cast<uint32_t>(rec.dec_merges * p.q_heads)), dim3(D), 0,
                     stream, static_cast<T*>(p.output.address), static_cast<float*>(p.lse.address),
                     DecodeMergeArgsOf(p, rec, dev, D), p.q_heads, kv.out_gate);
  return roost::HipStatus(hipGetLastError(), "paged_attention", "decode merge launch");
}

// The view of the decode kernels, whose virtual heads are groups of DecodeGroupOf query heads.
KvView DecodeView(const RoostPagedAttentionParams& p, KvView kv) {
  kv.vheads = DecodeHeads(p);
  kv.head_shift = static_cast<uint32_t>(__builtin_ctz(kv.vheads / p.kv_heads));
  return kv;
}

template <typename T, int D>
RoostStatus LaunchDecode(const RoostPagedAttentionParams& p, const PlanRecord& rec, unsigned char* dev, const KvView& kv,
                         float scale_log2, hipStream_t stream) {
  if (rec.dec_ranges == 0) return ROOST_STATUS_OK;
  const auto* items = reinterpret_cast<const DecodeWork*>(dev + rec.dec_item_offset);
  const auto* range_ptr = reinterpret_cast<const int32_t*>(dev + rec.dec_range_offset);
  auto* part_o = reinterpret_cast<float*>(dev + rec.dec_float_offset);
  auto* part_ml = part_o + rec.dec_splits * p.q_heads * D;
  // In a prefill call the decode pieces are its single-token sequences, whose query rows are q_indptr[seq].
  const auto* q_rows =
      p.mode == ROOST_ATTENTION_PREFILL ? static_cast<const int32_t*>(p.q_indptr.address) : nullptr;
  auto* out = static_cast<T*>(p.output.address);
  auto* lse = static_cast<float*>(p.lse.address);
  const uint32_t heads = DecodeHeads(p), hpw = rec.dec_heads_per_wg;
  const KvView dkv = DecodeView(p, kv);
  const dim3 grid(static_cast<uint32_t>(rec.dec_ranges * (heads / hpw)));
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, static_cast<const T*>(p.q.address), out, lse, dkv,
                       kv.kv_indices, items, range_ptr, part_o, part_ml, q_rows, p.q_heads, hpw, scale_log2, WindowOf(p),
                       p.causal, CapOf(p));
  };
  const bool fast = p.page_size % 16 == 0;
  if constexpr (sizeof(T) == 2) {
    auto of_group = [&](auto nh) {
      constexpr int kNh = decltype(nh)::value;
      fast ? launch(DecodeMfmaKernel<D, kNh, true>) : launch(DecodeMfmaKernel<D, kNh, false>);
    };
    const uint32_t nh = DecodeGroupOf(p);
    nh == 16  ? of_group(std::integral_constant<int, 16>{})
    : nh == 8 ? of_group(std::integral_constant<int, 8>{})
              : of_group(std::integral_constant<int, 4>{});
  } else {
    fast ? launch(DecodeF32Kernel<D, true>) : launch(DecodeF32Kernel<D, false>);
  }
  ROOST_RETURN_IF_FAILED(roost::HipStatus(hipGetLastError(), "paged_attention", "decode launch"));
  return LaunchDecodeMerge<T, D>(p, rec, dev, kv, stream);
}

// Partials of the tile pieces: rows of the pieces' normalised outputs, first the bf16 slots, then the fp32 ones, then their
// fp32 (max, sum) pairs.
uint16_t* PrefillPartO(const RoostPagedAttentionParams& p, const PlanRecord& rec, unsigned char* dev) {
  return reinterpret_cast<uint16_t*>(dev + rec.float_offset);
}
float* PrefillPartMl(const RoostPagedAttentionParams& p, const PlanRecord& rec, unsigned char* dev) {
  return reinterpret_cast<float*>(PrefillPartO(p, rec, dev) +
                                  (2 * rec.splits - rec.splits_bf16) * rec.item_tokens * kGroup * p.head_dim);
}

PrefillMergeArgs PrefillMergeArgsOf(const RoostPagedAttentionParams& p, const PlanRecord& rec, unsigned char* dev) {
  PrefillMergeArgs m{};
  m.merges = reinterpret_cast<const PrefillMerge*>(dev + rec.merge_offset);
  m.part_o = PrefillPartO(p, rec, dev);
  m.part_ml = PrefillPartMl(p, rec, dev);
  m.q_indptr = static_cast<const int32_t*>(p.q_indptr.address);
  m.splits_bf16 = static_cast<uint32_t>(rec.splits_bf16);
  m.two = static_cast<uint32_t>(rec.merges_two);
  const auto tokens = static_cast<uint32_t>(rec.item_tokens);
  m.blocks = m.two * (tokens / kPfMergeRows) + (static_cast<uint32_t>(rec.merges) - m.two) * tokens;
  return m;
}

RoostStatus LaunchPrefillMerge(const RoostPagedAttentionParams& p, const PlanRecord& rec, unsigned char* dev,
                               const KvView& kv, hipStream_t stream) {
  if (rec.merges == 0) return ROOST_STATUS_OK;
  auto* outp = static_cast<uint16_t*>(p.output.address);
  auto* lsep = static_cast<float*>(p.lse.address);
  const PrefillMergeArgs m = PrefillMergeArgsOf(p, rec, dev);
  const dim3 block(kGroup * p.head_dim / 4), g(m.blocks);
  const bool wide = rec.item_tokens == kPfWideTokens;
  auto* kernel = p.head_dim == 64    ? PrefillMergeKernel<64, kPfTokens>
                 : p.head_dim == 128 ? (wide ? PrefillMergeKernel<128, kPfWideTokens> : PrefillMergeKernel<128, kPfTokens>)
                                     : PrefillMergeKernel<256, kPfTokens>;
  hipLaunchKernelGGL(kernel, g, block, 0, stream, outp, lsep, m, p.q_heads, kv.out_gate);
  return roost::HipStatus(hipGetLastError(), "paged_attention", "prefill merge launch");
}

// A mixed step the plan chose to run in one launch (PlanRecord::overlap): the tile pieces and decode ranges on
// MixedAttentionKernel, then both merges in one MixedMergeKernel launch, all on the caller's stream.
RoostStatus LaunchMixed(const RoostPagedAttentionParams& p, const PlanRecord& rec, unsigned char* dev, const KvView& kv,
                        float scale_log2, hipStream_t stream) {
  const auto* q16 = static_cast<const uint16_t*>(p.q.address);
  const auto* q_indptr = static_cast<const int32_t*>(p.q_indptr.address);
  auto* outp = static_cast<uint16_t*>(p.output.address);
  auto* lsep = static_cast<float*>(p.lse.address);
  const auto* items = reinterpret_cast<const PrefillWork*>(dev);
  const uint32_t ps_shift = static_cast<uint32_t>(__builtin_ctz(p.page_size));
  const SoftCap cap = CapOf(p);
  const SoftCap raw{cap.capl / scale_log2, cap.k * scale_log2};
  const bool capped = cap.capl != 0.0f;
  const KvView dkv = DecodeView(p, kv);
  const uint32_t hpw = rec.dec_heads_per_wg;
  const uint32_t n_items = static_cast<uint32_t>(rec.work_items);
  const dim3 grid(n_items + static_cast<uint32_t>(rec.dec_ranges * (dkv.vheads / hpw)));
  const auto* dec_items = reinterpret_cast<const DecodeWork*>(dev + rec.dec_item_offset);
  const auto* dec_ranges = reinterpret_cast<const int32_t*>(dev + rec.dec_range_offset);
  auto* dec_o = reinterpret_cast<float*>(dev + rec.dec_float_offset);
  auto* dec_ml = dec_o + rec.dec_splits * p.q_heads * p.head_dim;
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(512), 0, stream, q16, outp, lsep, kv, kv.kv_indices, q_indptr, items,
                       PrefillPartO(p, rec, dev), PrefillPartMl(p, rec, dev), static_cast<uint32_t>(rec.splits_bf16),
                       p.q_heads, p.causal, ps_shift, scale_log2, WindowOf(p), raw, n_items,
                       dec_items, dec_ranges, dec_o, dec_ml, hpw, dkv.vheads, dkv.head_shift, cap);
  };
  auto of_group = [&](auto d, auto capped_c) {
    constexpr int kD = decltype(d)::value;
    constexpr bool kC = decltype(capped_c)::value;
    const uint32_t nh = DecodeGroupOf(p);
    nh == 16  ? launch(MixedAttentionKernel<kD, kC, 16>)
    : nh == 8 ? launch(MixedAttentionKernel<kD, kC, 8>)
              : launch(MixedAttentionKernel<kD, kC, 4>);
  };
  auto of_dim = [&](auto d) { capped ? of_group(d, std::true_type{}) : of_group(d, std::false_type{}); };
  p.head_dim == 64    ? of_dim(std::integral_constant<int, 64>{})
  : p.head_dim == 128 ? of_dim(std::integral_constant<int, 128>{})
                      : of_dim(std::integral_constant<int, 256>{});
  ROOST_RETURN_IF_FAILED(roost::HipStatus(hipGetLastError(), "paged_attention", "mixed attention launch"));
  const PrefillMergeArgs pm = rec.merges != 0 ? PrefillMergeArgsOf(p, rec, dev) : PrefillMergeArgs{};
  const DecodeMergeArgs dm = DecodeMergeArgsOf(p, rec, dev, p.head_dim);
  const uint64_t blocks = uint64_t{pm.blocks} + rec.dec_merges * p.q_heads;
  if (blocks == 0) return ROOST_STATUS_OK;
  const dim3 g(static_cast<uint32_t>(blocks)), block(p.head_dim);
  auto* merge = p.head_dim == 64 ? MixedMergeKernel<64> : p.head_dim == 128 ? MixedMergeKernel<128> : MixedMergeKernel<256>;
  hipLaunchKernelGGL(merge, g, block, 0, stream, outp, lsep, pm, dm, p.q_heads, kv.out_gate);
  return roost::HipStatus(hipGetLastError(), "paged_attention", "mixed merge launch");
}

RoostStatus LaunchPrefill(const RoostPagedAttentionParams& p, const PlanRecord& rec, unsigned char* dev, const KvView& kv,
                          float scale_log2, hipStream_t stream) {
  if (rec.work_items == 0) return ROOST_STATUS_OK;
  const auto* items = reinterpret_cast<const PrefillWork*>(dev);
  const auto* q_indptr = static_cast<const int32_t*>(p.q_indptr.address);
  auto* outp = static_cast<uint16_t*>(p.output.address);
  auto* lsep = static_cast<float*>(p.lse.address);
  if (PrefillFastPath(p)) {
    uint16_t* part_o = PrefillPartO(p, rec, dev);
    float* part_ml = PrefillPartMl(p, rec, dev);
    const dim3 grid(static_cast<uint32_t>(rec.work_items));
    const auto* q16 = static_cast<const uint16_t*>(p.q.address);
    const uint32_t ps_shift = static_cast<uint32_t>(__builtin_ctz(p.page_size));
    // The cap in unscaled score units: Capped(s * scale_log2, cap) / scale_log2 == Capped(s, raw).
    const SoftCap cap = CapOf(p);
    const SoftCap raw{cap.capl / scale_log2, cap.k * scale_log2};
    const bool capped = cap.capl != 0.0f;
    auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(static_cast<uint32_t>(8 * rec.item_tokens)), 0, stream, q16, outp, lsep, kv,
                         kv.kv_indices, q_indptr, items, part_o, part_ml, static_cast<uint32_t>(rec.splits_bf16), p.q_heads,
                         p.causal, ps_shift, scale_log2, WindowOf(p), raw);
    };
    const bool wide = rec.item_tokens == kPfWideTokens;
    if (p.head_dim == 64) {
      capped ? launch(PrefillTileKernel<64, true, 8>) : launch(PrefillTileKernel<64, false, 8>);
    } else if (p.head_dim == 128) {
      wide ? (capped ? launch(PrefillTileKernel<128, true, 12>) : launch(PrefillTileKernel<128, false, 12>))
           : (capped ? launch(PrefillTileKernel<128, true, 8>) : launch(PrefillTileKernel<128, false, 8>));
    } else {
      capped ? launch(PrefillTileKernel<256, true, 8>) : launch(PrefillTileKernel<256, false, 8>);
    }
    ROOST_RETURN_IF_FAILED(roost::HipStatus(hipGetLastError(), "paged_attention", "prefill launch"));
    return LaunchPrefillMerge(p, rec, dev, kv, stream);
  }
  hipLaunchKernelGGL(PrefillKernel, dim3(static_cast<uint32_t>(rec.work_items)), dim3(256), 0, stream,
                     static_cast<const uint16_t*>(p.q.address), outp, lsep, kv, q_indptr, items, p.q_heads, p.causal,
                     scale_log2, WindowOf(p), CapOf(p));
  return roost::HipStatus(hipGetLastError(), "paged_attention", "prefill launch");
}


constexpr char kOp[] = "paged_attention";

const RoostPagedAttentionParams* Params(const void* params) {
  return static_cast<const RoostPagedAttentionParams*>(params);
}

// The element type a plan is made for. plan() reads no spans, so a caller may leave it out: the tables are then those of
// bf16, which in a decode call also serve f32 (the partials are f32 rows either way, and every workgroup's share of bf16
// head groups divides the f32 ones).
uint32_t PlanDtype(const RoostPagedAttentionParams& p) {
  return p.q.dtype == ROOST_DTYPE_F32 || p.q.dtype == ROOST_DTYPE_BF16 ? p.q.dtype : ROOST_DTYPE_UNDEFINED;
}

// The plan record plan() leaves for run(): the batch shape it was made for and where its tables sit.
PlanRecord MakeRecord(const RoostPagedAttentionParams& p, const Layout& l) {
  PlanRecord r{};
  r.magic = kPlanMagic;
  r.mode = p.mode;
  r.batch = p.batch;
  r.tokens = p.tokens;
  r.page_size = p.page_size;
  r.kv_layout = p.kv_layout;
  r.head_dim = p.head_dim;
  r.kv_heads = p.kv_heads;
  r.window = WindowOf(p);
  r.merges_two = static_cast<uint32_t>(l.merges_two);
  r.item_tokens = l.item_tokens;
  r.splits_bf16 = l.splits_bf16;
  r.q_heads = p.q_heads;
  r.dtype = PlanDtype(p);
  r.overlap = l.overlap;
  r.dec_heads_per_wg = l.dec_heads_per_wg;
  r.pages = static_cast<uint64_t>(p.kv_indptr_host[p.batch]);
  r.work_items = l.work_items;
  r.ranges = l.ranges;
  r.merges = l.merges;
  r.range_offset = l.range_offset;
  r.merge_offset = l.merge_offset;
  r.counter_offset = l.counter_offset;
  r.splits = l.splits;
  r.int_bytes = l.int_bytes;
  r.float_offset = l.float_offset;
  r.float_bytes = l.float_bytes;
  r.dec_items = l.dec_items;
  r.dec_ranges = l.dec_ranges;
  r.dec_merges = l.dec_merges;
  r.dec_splits = l.dec_splits;
  r.dec_item_offset = l.dec_item_offset;
  r.dec_range_offset = l.dec_range_offset;
  r.dec_merge_offset = l.dec_merge_offset;
  r.dec_float_offset = l.dec_float_offset;
  return r;
}

// The partials and, in a prefill, the items are laid out for the plan's query heads, and a prefill's tables for its element
// type: run with others, the kernels would write past the workspace or leave rows unwritten.
bool RecordFits(const PlanRecord& r, const RoostPagedAttentionParams& p) {
  const bool dtype = r.dtype == p.q.dtype || (r.dtype == ROOST_DTYPE_UNDEFINED &&
                                              (p.mode == ROOST_ATTENTION_DECODE || p.q.dtype == ROOST_DTYPE_BF16));
  return dtype && r.q_heads == p.q_heads && r.mode == p.mode && r.batch == p.batch && r.tokens == p.tokens &&
         r.page_size == p.page_size && r.kv_layout == p.kv_layout && r.head_dim == p.head_dim && r.kv_heads == p.kv_heads && r.window == WindowOf(p);
}

}  // namespace

extern "C" ROOST_API RoostStatus roost_paged_attention_workspace(RoostContext* ctx, const void* params,
                                                                 RoostWorkspaceSizes* sizes) {
  roost::Gate gate(kOp);
  gate.Header(params, sizeof(RoostPagedAttentionParams))
      .Expect(sizes != nullptr, ROOST_STATUS_INVALID_ARGUMENT, "the sizes out-pointer is NULL");
  ROOST_GATE_RETURN(gate);
  const auto& p = *Params(params);
  return roost::CatchAll(kOp, [&]() -> RoostStatus {
    ROOST_RETURN_IF_FAILED(Admit(p, false));
    const Layout l = PlanLayout(p, ComputeUnits(ctx), nullptr);
    *sizes = RoostWorkspaceSizes{};
    sizes->device_bytes = l.total;
    sizes->pinned_host_bytes = l.int_bytes;
    sizes->plan_bytes = sizeof(PlanRecord);
    sizes->device_alignment = kAlign;
    return ROOST_STATUS_OK;
  });
}

extern "C" ROOST_API RoostStatus roost_paged_attention_plan(RoostContext* ctx, const void* params, const RoostWorkspace* ws,
                                                            void* stream) {
  roost::Gate gate(kOp);
  ROOST_GATE_RETURN(gate.Header(params, sizeof(RoostPagedAttentionParams)));
  const auto& p = *Params(params);
  return roost::CatchAll(kOp, [&]() -> RoostStatus {
    ROOST_RETURN_IF_FAILED(Admit(p, false));
    gate.Expect(ws != nullptr && ws->plan != nullptr, ROOST_STATUS_INVALID_ARGUMENT,
                "plan() writes its record into ws->plan, which is missing");
    ROOST_GATE_RETURN(gate);
    const uint32_t cus = ComputeUnits(ctx);
    const Layout l = PlanLayout(p, cus, nullptr);
    const bool fits = ws->plan_bytes >= sizeof(PlanRecord) && ws->pinned_host_bytes >= l.int_bytes &&
                      (l.int_bytes == 0 || ws->pinned_host != nullptr) && roost::HasDeviceRegion(ws, l.total, kAlign);
    gate.Expect(fits, ROOST_STATUS_WORKSPACE_TOO_SMALL,
                "this batch needs %llu device bytes (%u-aligned), %llu pinned bytes and a %zu-byte plan record; the "
                "workspace has %llu, %llu and %llu", static_cast<unsigned long long>(l.total), kAlign,
                static_cast<unsigned long long>(l.int_bytes), sizeof(PlanRecord),
                static_cast<unsigned long long>(ws->device_bytes), static_cast<unsigned long long>(ws->pinned_host_bytes),
                static_cast<unsigned long long>(ws->plan_bytes));
    ROOST_GATE_RETURN(gate);
    if (l.int_bytes > 0) {
      auto* host = static_cast<unsigned char*>(ws->pinned_host);
      std::memset(host, 0, l.int_bytes);
      PlanLayout(p, cus, host);
      ROOST_RETURN_IF_FAILED(roost::HipStatus(
          hipMemcpyAsync(ws->device, host, l.int_bytes, hipMemcpyHostToDevice, roost::Stream(stream)), kOp,
          "copy of the work tables to the device"));
    }
    const PlanRecord rec = MakeRecord(p, l);
    std::memcpy(ws->plan, &rec, sizeof(rec));
    return ROOST_STATUS_OK;
  });
}

namespace {

// run() of an admitted-or-not call; out_gate (NULL for none) folds SigmoidMul into every kernel that writes an output
// row.
RoostStatus RunAttention(RoostContext* ctx, const void* params, const RoostWorkspace* ws, void* stream,
                         const void* out_gate) {
  using namespace roost;
  Gate gate(kOp);
  ROOST_GATE_RETURN(gate.Header(params, sizeof(RoostPagedAttentionParams)));
  const auto& p = *Params(params);
  return CatchAll(kOp, [&]() -> RoostStatus {
    ROOST_RETURN_IF_FAILED(Admit(p, true));
    // C1: run() before plan() in this workspace is NOT_PLANNED (the caller then plans and runs again).
    if (ws == nullptr || ws->plan == nullptr || ws->plan_bytes < sizeof(PlanRecord)) {
      return Report(ROOST_STATUS_NOT_PLANNED, kOp, "the workspace carries no plan record; call plan() first");
    }
    PlanRecord rec;
    std::memcpy(&rec, ws->plan, sizeof(rec));
    if (rec.magic != kPlanMagic) {
      return Report(ROOST_STATUS_NOT_PLANNED, kOp, "the plan record is blank; call plan() first");
    }
    gate.Expect(RecordFits(rec, p), ROOST_STATUS_INVALID_ARGUMENT,
                "the plan record describes batch %u / tokens %u / mode %u / window %d; this call is batch %u / tokens "
                "%u / mode %u / window %d (or its page size, layout, head shape or element type differ)", rec.batch, rec.tokens,
                rec.mode, rec.window, p.batch, p.tokens, p.mode, WindowOf(p))
        .Tensor("kv_indices", p.kv_indices, ROOST_DTYPE_I32, rec.pages)
        .Expect(HasDeviceRegion(ws, rec.float_offset + rec.float_bytes, kAlign), ROOST_STATUS_WORKSPACE_TOO_SMALL,
                "the plan placed %llu bytes in the device workspace, which holds %llu",
                static_cast<unsigned long long>(rec.float_offset + rec.float_bytes),
                static_cast<unsigned long long>(ws->device_bytes));
    ROOST_GATE_RETURN(gate);
    const float scale = p.sm_scale != 0.0f ? p.sm_scale : 1.0f / std::sqrt(static_cast<float>(p.head_dim));
    const float scale_log2 = scale * kLog2e;
    KvView kv{};
    kv.k = p.k_cache.address;
    kv.v = p.v_cache.address;
    kv.kv_indptr = static_cast<const int32_t*>(p.kv_indptr.address);
    kv.kv_indices = static_cast<const int32_t*>(p.kv_indices.address);
    kv.last_len = static_cast<const int32_t*>(p.kv_last_page_len.address);
    const uint64_t page_elems = static_cast<uint64_t>(p.page_size) * p.kv_heads * p.head_dim;
    kv.pool_pages = std::min(p.k_cache.length, p.v_cache.length) / page_elems;
    kv.page_size = p.page_size;
    kv.kv_heads = p.kv_heads;
    kv.head_shift = HeadShift(p);
    kv.vheads = VirtualHeads(p);
    kv.hnd = p.kv_layout == ROOST_LAYOUT_PAGED_HND ? 1u : 0u;
    kv.out_gate = out_gate;
    auto* dev = static_cast<unsigned char*>(ws->device);
    hipStream_t s = Stream(stream);
    if (p.mode == ROOST_ATTENTION_DECODE) {
      const bool bf16 = p.q.dtype == ROOST_DTYPE_BF16;
      switch (p.head_dim) {
        case 64: return bf16 ? LaunchDecode<uint16_t, 64>(p, rec, dev, kv, scale_log2, s)
                             : LaunchDecode<float, 64>(p, rec, dev, kv, scale_log2, s);
        case 128: return bf16 ? LaunchDecode<uint16_t, 128>(p, rec, dev, kv, scale_log2, s)
                              : LaunchDecode<float, 128>(p, rec, dev, kv, scale_log2, s);
        default: return bf16 ? LaunchDecode<uint16_t, 256>(p, rec, dev, kv, scale_log2, s)
                             : LaunchDecode<float, 256>(p, rec, dev, kv, scale_log2, s);
      }
    }
    // The multi-token sequences on the tile kernels, then the single-token ones on the decode kernels (bf16 in prefill
    // mode, at the call's head dim), or both in one launch when the plan chose that (ChooseOverlap).
    if (p.q.dtype == ROOST_DTYPE_F32) {  // every query token is a row of the f32 decode kernel
      switch (p.head_dim) {
        case 64: return LaunchDecode<float, 64>(p, rec, dev, kv, scale_log2, s);
        case 128: return LaunchDecode<float, 128>(p, rec, dev, kv, scale_log2, s);
        default: return LaunchDecode<float, 256>(p, rec, dev, kv, scale_log2, s);
      }
    }
    if (rec.overlap != 0) return LaunchMixed(p, rec, dev, kv, scale_log2, s);
    ROOST_RETURN_IF_FAILED(LaunchPrefill(p, rec, dev, kv, scale_log2, s));
    switch (p.head_dim) {
      case 64: return LaunchDecode<uint16_t, 64>(p, rec, dev, kv, scale_log2, s);
      case 128: return LaunchDecode<uint16_t, 128>(p, rec, dev, kv, scale_log2, s);
      default: return LaunchDecode<uint16_t, 256>(p, rec, dev, kv, scale_log2, s);
    }
  });
}

}  // namespace

extern "C" ROOST_API RoostStatus roost_paged_attention_run(RoostContext* ctx, const void* params,
                                                           const RoostWorkspace* ws, void* stream) {
  return RunAttention(ctx, params, ws, stream, nullptr);
}

// PagedAttention followed by SigmoidMul on its output, in one call: the gate multiplies each output element where the
// kernels write it (the tile, decode and merge kernels' epilogues), with SigmoidMul's arithmetic on the output already
// rounded to its type, so the result equals run() then roost_sigmoid_mul_run bit for bit and the output is written once.
extern "C" ROOST_API RoostStatus roost_amd_paged_attention_gated_run(RoostContext* ctx, const void* params,
                                                                     const void* gate_params, const RoostWorkspace* ws,
                                                                     void* stream) {
  using namespace roost;
  Gate gate(kOp);
  ROOST_GATE_RETURN(gate.Header(params, sizeof(RoostPagedAttentionParams)));
  gate.Expect(gate_params != nullptr, ROOST_STATUS_INVALID_ARGUMENT, "no SigmoidMul params struct was passed");
  ROOST_GATE_RETURN(gate);
  ROOST_GATE_RETURN(gate.Header(gate_params, sizeof(RoostSigmoidMulParams)));
  const auto& p = *Params(params);
  const auto& sm = *static_cast<const RoostSigmoidMulParams*>(gate_params);
  return CatchAll(kOp, [&]() -> RoostStatus {
    ROOST_RETURN_IF_FAILED(Admit(p, true));
    const uint32_t dt = p.output.dtype;
    const uint64_t dim = static_cast<uint64_t>(p.q_heads) * p.head_dim, n = dim * p.tokens;
    gate.Expect(sm.rows == p.tokens && sm.dim == dim, ROOST_STATUS_INVALID_ARGUMENT,
                "the gate covers %u rows x %u; the attention output is %u tokens x %llu", sm.rows, sm.dim, p.tokens,
                static_cast<unsigned long long>(dim))
        .Expect(sm.input.address == p.output.address && sm.output.address == p.output.address,
                ROOST_STATUS_INVALID_ARGUMENT,
                "the gate applies in place: its input and output must both be the attention output (%p), not %p and %p",
                p.output.address, sm.input.address, sm.output.address)
        .Tensor("gate input", sm.input, dt, n)
        .Tensor("gate output", sm.output, dt, n)
        .Tensor("gate", sm.gate, dt, n)
        .Aligned("gate", sm.gate.address, 8);
    ROOST_GATE_RETURN(gate);
    const auto g0 = reinterpret_cast<uintptr_t>(sm.gate.address), o0 = reinterpret_cast<uintptr_t>(p.output.address);
    const uint64_t bytes = n * ElementBytes(dt);
    gate.Expect(n == 0 || g0 + bytes <= o0 || o0 + bytes <= g0, ROOST_STATUS_INVALID_ARGUMENT,
                "the gate (%p) overlaps the output (%p, %llu bytes)", sm.gate.address, p.output.address,
                static_cast<unsigned long long>(bytes));
    ROOST_GATE_RETURN(gate);
    return RunAttention(ctx, params, ws, stream, sm.gate.address);
  });
}
