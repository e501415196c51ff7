// Host-side launch wrappers for the gfx950 kernels (internal interface of
// liborion_hip.so; the public C ABI lives in include/orion_hip.h).
#pragma once

#include <hip/hip_runtime.h>
#ifdef __HIPCC__
#include "common.hpp"
#endif
#include <cstddef>
#include <cstdint>
#include <vector>

namespace orion {

// Geometry of a paged KV arena [layer][block][k|v][slot][kv_head][head_dim].
struct KvGeom {
  int64_t num_layers, num_blocks, block_size, num_kv_heads, head_dim;
  bool dtype_bf16;
  bool head_major = false;  // block-internal order [kv_head][k|v][slot] instead of [k|v][slot][kv_head]
};

// Element strides of the arena (one layer = num_blocks blocks).  Reference
// layout (attention.rs:11-22): [block][k|v][slot][kv_head][dim].  Head-major
// layout: [block][kv_head][k|v][slot][dim], so one head's K (or V) of a block
// is one contiguous block_size x dim run.
struct ArenaStrides {
  int64_t blk, v_off, slot, head, layer;
};
inline ArenaStrides arena_strides(const KvGeom& kv) {
  ArenaStrides a;
  const int64_t bs = kv.block_size, hkv = kv.num_kv_heads, D = kv.head_dim;
  a.blk = 2 * bs * hkv * D;
  if (kv.head_major) {
    a.head = 2 * bs * D;
    a.v_off = bs * D;
    a.slot = D;
  } else {
    a.head = D;
    a.v_off = bs * hkv * D;
    a.slot = hkv * D;
  }
  a.layer = kv.num_blocks * a.blk;
  return a;
}

// ---- attention --------------------------------------------------------------
// One decode work item: KV head `item % Hkv` of query row `item / Hkv` over
// context tokens [start, end), the row's piece `split` of `nsplit`.  The block
// table slice of the piece starts at block_table_ids[tbl_off]; blk0 is its
// first entry, so the first step's loads can be issued before the slice
// arrives.
struct DecodeWork {
  // shared: 1 when the item reads a block that another planned row also
  // reads, 2 for a packed prefix item (DecodePlanHost::num_packed)
  int32_t item, start, end, nsplit, tbl_off, blk0, shared, split;
};
// Decode work plan: packed prefix items first, then the others longest first;
// built on the host from the
// query positions and block tables, shared by every layer of a forward.
struct DecodePlanHost {
  int chunk = 0;       // longest piece, in tokens
  int max_splits = 0;  // most pieces of any row
  bool balanced = false;  // per-row piece lengths (else fixed chunks)
  std::vector<DecodeWork> work;
  std::vector<int32_t> row_nsplit;  // pieces per row (0: row not planned)
  std::vector<int32_t> rows;  // rows covered when a skip mask was given (else all)
  // No block is attended by two planned rows: K/V are then read once and
  // streamed past the caches; shared (prefix) blocks keep cached loads.
  bool stream_kv = true;
  // Some blocks are shared but some work items read none of them: those
  // items stream, the others keep cached loads (DecodeWork::shared).
  bool mixed_kv = false;
  // Packed items (DecodeWork::shared == 2, num_packed of them): a piece of a
  // prefix that up to pack_r rows share (identical leading block ids),
  // attended for all of them at once -- their query heads fill the query
  // columns of one MFMA wave, so the prefix is read once per pack instead of
  // once per row.  Entry item = pack * hkv + kv_head; the pack's rows are
  // pack_rows[pack * pack_r .. + pack_r) (-1: unused).  Their prefix pieces
  // are splits 0 .. np-1 of each of those rows; the rows' remaining context
  // follows as ordinary items with splits np ...
  int num_packed = 0;
  int pack_r = 0;
  std::vector<int32_t> pack_rows;
  // Short contexts: group_waves items per (row, KV head), run and merged by one
  // workgroup instead of `work` and the merge launch (build_decode_groups; end
  // 0: no piece, nsplit: the row's pieces).
  int group_waves = 0;
  std::vector<DecodeWork> groups;
};
struct DecodePlanDev {
  const DecodeWork* work = nullptr;
  const int32_t* row_nsplit = nullptr;  // DecodePlanHost::row_nsplit on the device
  int num_work = 0;
  int chunk = 0;
  int max_splits = 0;
  float* ws = nullptr;  // split-K partials, decode_workspace_bytes()
  size_t ws_bytes = 0;
  const int32_t* rows = nullptr;  // rows to merge (nullptr: every row)
  int num_rows = 0;
  bool stream_kv = true;  // DecodePlanHost::stream_kv
  bool mixed_kv = false;  // DecodePlanHost::mixed_kv
  // packed prefix items (DecodePlanHost::num_packed, counted in num_work),
  // DecodePlanHost::pack_rows on the device, and rows per pack
  int num_packed = 0;
  const int32_t* pack_rows = nullptr;
  int pack_r = 0;
  // DecodePlanHost::groups on the device; num_groups workgroups of group_waves
  const DecodeWork* groups = nullptr;
  int num_groups = 0;
  int group_waves = 0;
};
// pack_r: rows per packed prefix item; 0 packs nothing.  The decode kernels
// take packed items only on bf16 arenas at head_dim 64/128 with
// pack_r = 16 / (query heads per KV head) >= 2 (decode_pack_rows).
void build_decode_plan(const uint32_t* positions, const int32_t* row_seq,
                       const int64_t* bt_offsets, const uint32_t* bt_ids, int64_t rows,
                       int64_t hkv, int64_t block_size, int64_t wave_slots,
                       const uint8_t* skip_rows, DecodePlanHost* plan, int pack_r = 0);
// Waves per workgroup of a grouped plan: 16 where a wave fits 128 registers
// (head_dim 64; f32 arenas up to 4 query heads per KV head), else 8; 0 where the
// group kernels do not apply (they lost on f32 arenas at head_dim 128).
constexpr int kGroupWaves[2] = {8, 16};
int decode_group_waves(const KvGeom& kv, int64_t hq);
// Fills plan->groups when the planned rows are few and short enough
// (group_waves of 0 leaves the plan as it is).
void build_decode_groups(const uint32_t* positions, const int32_t* row_seq,
                         const int64_t* bt_offsets, const uint32_t* bt_ids, int64_t rows,
                         int64_t hkv, int64_t block_size, int64_t cus, int group_waves,
                         const uint8_t* skip_rows, DecodePlanHost* plan);
size_t decode_workspace_bytes(int64_t rows, int64_t hq, int64_t D, int64_t max_splits);
// Rows per packed prefix item for this arena and grouping (0: no packing).
int decode_pack_rows(const KvGeom& kv, int64_t hq);
// Where a decode pass writes its rows: f32 rows [row][hq * d], or fragment
// order over mtiles row tiles (frag set; the MFMA wave's shapes only,
// decode_mfma).
struct AttnOut {
  float* rows = nullptr;
  uint16_t* frag = nullptr;
  int mtiles = 0;
};
// Which launches of a decode pass to issue (the merge only runs when the
// plan splits some row).
enum class DecodePhase { kBoth, kSplit, kMerge };
// Merges split partials held in plan.ws (the decode split layout over `rows`
// batch rows, plan.max_splits slots per (row, head)) of the rows plan.rows
// lists, plan.row_nsplit[row] parts each, into out (the chunked-prefill key
// parts use it too).
hipError_t launch_split_merge(hipStream_t st, int64_t D, int64_t rows, int64_t hq,
                              const DecodePlanDev& plan, float* out);
// Whether launch_paged_decode runs this shape on the MFMA wave (bf16 arenas at
// head_dim 64/128, up to 16 query heads per KV head).
inline bool decode_mfma(const KvGeom& kv, int64_t hq) {
  return kv.dtype_bf16 && (kv.head_dim == 64 || kv.head_dim == 128) &&
         hq / kv.num_kv_heads <= 16;
}
hipError_t launch_paged_decode(hipStream_t st, const KvGeom& kv, const void* arena, int64_t layer,
                               const float* q, int64_t rows, int64_t hq,
                               const uint32_t* positions, const int32_t* row_seq,
                               const int64_t* bt_off, const uint32_t* bt_ids,
                               const DecodePlanDev& plan, const AttnOut& out,
                               DecodePhase phase = DecodePhase::kBoth);

// Prefill work list: one entry per (sequence, tile of packed rows, part of
// its keys), longest first (by the key tiles it reads), so the longest
// workgroups are dispatched first.  A sequence whose tiles would read far
// more keys than an even share of the CUs is cut into nparts key ranges; each
// part writes unnormalised partial results (the decode split layout) that a
// merge combines.  Built on the host from the chunk lengths and first
// positions; the device copy is what launch_paged_prefill takes.
struct PrefillTile {
  int32_t seq, tile;
  int32_t kt0, kt1;      // key tiles [kt0, kt1) (64 keys each) this workgroup reads
  int32_t part, nparts;  // nparts > 1: partial results of part `part`
};
struct PrefillPlan {
  std::vector<PrefillTile> order;
  int max_parts = 1;
  // batch rows whose results come in parts, and parts per batch row (0 for
  // rows of unsplit sequences; sized to the batch's rows)
  std::vector<int32_t> split_rows, row_parts;
};
int prefill_waves();      // waves per prefill workgroup (8, or 4 with ORION_PREFILL_WAVES=4)
// 16-row MFMA tiles of packed rows per prefill wave: two, one at head_dim 256
// (its query operands and output accumulators take twice the registers).
constexpr int prefill_wave_row_tiles(int64_t head_dim) { return head_dim > 128 ? 1 : 2; }
int prefill_tile_rows(int64_t head_dim);  // packed rows per prefill workgroup
// Largest head_dim the attention and RoPE kernels take (any even value up to
// it; the reference accepts any even head_dim).
constexpr int kMaxHeadDim = 2048;
// Prefill operand precision bits (launch_paged_prefill `operands`): each set
// bit carries that operand as a hi + lo bf16 pair, each clear one rounds it
// to bf16.
constexpr int kPrefillQHiLo = 1, kPrefillPHiLo = 2;
// cus: compute units (one prefill workgroup each); hkv: KV heads (workgroups
// per work-list entry); cus = 0 never splits.
void build_prefill_order(const int32_t* row_start, const int32_t* row_count,
                         const uint32_t* first_pos, int64_t num_seqs, int64_t group, int64_t hkv,
                         int64_t cus, PrefillPlan* plan, int64_t head_dim = 128);
// Where split parts go: the decode split workspace layout over the batch's
// rows (slot = (row * hq + head) * max_parts + part).
struct PrefillSplitOut {
  float* ws_o = nullptr;
  float* ws_ml = nullptr;
  int max_parts = 1;
  // finished rows are written in the split operand layout of GemmFuse::x_hilo
  // (only when no row comes in parts)
  int out_hilo = 0;
};
hipError_t launch_paged_prefill(hipStream_t st, const KvGeom& kv, const void* arena,
                                int64_t layer, const float* q, int64_t hq,
                                const PrefillTile* order, int64_t num_tiles,
                                const int32_t* row_start, const int32_t* row_count,
                                const uint32_t* first_pos, const int64_t* bt_off,
                                const uint32_t* bt_ids, int operands, float* out,
                                const PrefillSplitOut& split = PrefillSplitOut{});
// Packed (row, query head) rows per prefill workgroup tile.

// ---- GEMM -------------------------------------------------------------------
enum class Epilogue : int {
  kStore = 0,       // out = x W^T (+ bias)
  kAccumulate = 1,  // out += x W^T
  kSwiGLU = 2,      // W rows interleaved in groups of 8 gate / 8 up rows;
                    // out[:, N/2] = silu(gate) * up
};
// Activations of a decode-shaped forward in fragment order: the layout in
// which gemm_rows_kernel's lanes read them.  For 16-row tile mt of mtiles,
// k-step s of 32 and half h (0: the value rounded to bf16, 1: the remainder
// rounded to bf16; split2_rne) one KiB, lane l's 16 bytes (row 16 mt + l % 16, k
// 32 s + 8 (l / 16) .. + 8) at 16 l.  Rows are padded to 16; the bytes are
// those of f32.  Used past kFragMinRows rows (below, f32 rows are fewer bytes
// than a padded tile).
constexpr int64_t kFragMinRows = 9;
__host__ __device__ constexpr int act_tiles(int64_t rows) { return (int)((rows + 15) / 16); }
inline size_t act_frag_bytes(int64_t rows, int64_t cols) {
  return (size_t)act_tiles(rows) * 16 * (size_t)((cols + 31) / 32 * 32) * 4;
}
#ifdef __HIPCC__
// Element (row, col) of half 0, in 2-byte units; half 1 is 512 further on.
__device__ inline int64_t frag_at(int mtiles, int row, int col) {
  return ((int64_t)(col >> 5) * mtiles + (row >> 4)) * 1024 +
         (((col >> 3) & 3) * 16 + (row & 15)) * 8 + (col & 7);
}
__device__ inline void store_frag(uint16_t* frag, int mtiles, int row, int col, float v) {
  uint32_t h, l;
  split2_rne(v, 0.f, h, l);
  const int64_t at = frag_at(mtiles, row, col);
  frag[at] = (uint16_t)h;
  frag[at + 512] = (uint16_t)l;
}
// Four consecutive columns, col a multiple of 4.
__device__ inline void store_frag4(uint16_t* frag, int mtiles, int row, int col, float4 v) {
  uint2 h, l;
  split2_rne(v.x, v.y, h.x, l.x);
  split2_rne(v.z, v.w, h.y, l.y);
  const int64_t at = frag_at(mtiles, row, col);
  *reinterpret_cast<uint2*>(frag + at) = h;
  *reinterpret_cast<uint2*>(frag + at + 512) = l;
}
#endif
// Column `col` of a packed QKV matrix in W's own order: within the Q and K
// heads (columns below pair_cols, pair_dim each) a 16-column tile holds 8
// columns of the head's first half and the 8 of its second half that RoPE
// rotates them with.  pair_dim 0: W's order.
__host__ __device__ inline int packed_column(int col, int64_t pair_dim, int64_t pair_cols) {
  if (!pair_dim || col >= pair_cols) return col;
  const int D = (int)pair_dim, head = col / D, q = col - head * D;
  const int e = q & 15, j = (q >> 4) * 8 + (e & 7);
  return head * D + (e < 8 ? j : (D >> 1) + j);
}
// Weights [N, K] in packed order, the layout every GEMM of a forward reads:
// per 16 columns and 32 k one KiB (an MFMA B fragment, lane l's 16 bytes at
// 16 l), the k-steps of a column tile consecutive.  0 bytes: K not a multiple
// of 32.
size_t packed_weight_bytes(int64_t N, int64_t K);
hipError_t launch_pack_weights(hipStream_t st, const uint16_t* w, int64_t N, int64_t K,
                               int64_t pair_dim, int64_t pair_cols, uint16_t* out);
hipError_t launch_unpack_weights(hipStream_t st, const uint16_t* packed, int64_t N, int64_t K,
                                 int64_t pair_dim, int64_t pair_cols, uint16_t* w);

// RoPE and the KV write of a QKV GEMM's rows (launch_rope_and_cache's work):
// q_out null when the GEMM stores its output instead.  kv is the layer's
// arena, strides in elements.
struct RopeOut {
  float* q_out = nullptr;  // [rows, hq * d]
  void* kv = nullptr;
  bool kv_bf16 = false;
  int hq = 0, hkv = 0, bs_log2 = 0;
  int64_t blk = 0, v_off = 0, slot = 0, head = 0;
  const uint32_t* positions = nullptr;
  const int32_t* row_seq = nullptr;
  const int64_t* bt_off = nullptr;
  const uint32_t* bt_ids = nullptr;
  const float* cos = nullptr;
  const float* sin = nullptr;
};
#ifdef __HIPCC__
// Where a row's new K/V vector goes, and its position.
struct RowSlot {
  int64_t kv;
  uint32_t pos;
};
__device__ inline RowSlot row_slot(const RopeOut& r, int row) {
  const uint32_t pos = r.positions[row];
  const uint32_t blk = r.bt_ids[r.bt_off[r.row_seq[row]] + (pos >> r.bs_log2)];
  return {(int64_t)blk * r.blk + (int64_t)(pos & ((1u << r.bs_log2) - 1)) * r.slot, pos};
}
__device__ inline void store_kv1(void* base, bool bf16, int64_t at, float v) {
  if (bf16)
    static_cast<uint16_t*>(base)[at] = f32_to_bf16(v);
  else
    static_cast<float*>(base)[at] = v;
}
#endif
// A projection of a decode-shaped forward (gemm_rows.hip) on packed weights.
struct RowsGemm {
  const float* x = nullptr;  // f32 rows, or fragment order (x_frag)
  bool x_frag = false;
  const uint16_t* w = nullptr;
  const float* bias = nullptr;  // kStore
  int64_t M = 0, N = 0, K = 0;
  Epilogue ep = Epilogue::kStore;
  float* out = nullptr;
  // RMSNorm of x: the row sums of squares a previous kernel left
  // ([row][norm_slots] f64), and for f32 rows the norm weight (fragments
  // carry it multiplied in)
  const double* norm_sumsq = nullptr;
  int norm_slots = 0;
  const float* norm_weight = nullptr;
  float norm_eps = 0.f;
  // kSwiGLU: the output in fragment order instead of `out`.  kAccumulate: the
  // updated row times next_weight in fragment order, beside `out`.
  uint16_t* out_frag = nullptr;
  const float* next_weight = nullptr;
  double* sumsq_out = nullptr;  // kAccumulate: rows_sumsq_slots(N) f64 per row
  // QKV: the packed order of its columns, and the fused RoPE + KV write
  int64_t pair_dim = 0, pair_cols = 0;
  RopeOut rope;
  float* partial = nullptr;  // set by launch_gemm_rows
};
constexpr int64_t kRowsMax = 64;  // most rows of a launch_gemm_rows call
inline int rows_sumsq_slots(int64_t N) { return (int)((N + 15) / 16); }
size_t rows_scratch_bytes(const RowsGemm& g);
hipError_t launch_gemm_rows(hipStream_t st, const RowsGemm& g, float* scratch,
                            size_t scratch_bytes);

// Scratch for split-K GEMMs: the K-slice partial tiles.
struct GemmScratch {
  float* ws = nullptr;
  size_t ws_bytes = 0;
};
// What a forward's prefill-shaped GEMMs add to a launch_gemm call (M > 64).
struct GemmFuse {
  // the weights in packed order (launch_pack_weights), read instead of w; for
  // QKV also the order of its columns
  const uint16_t* w_packed = nullptr;
  int64_t pair_dim = 0, pair_cols = 0;
  // x arrives already split into its bf16 hi/lo pair (the layout
  // launch_rmsnorm and the SwiGLU epilogue write with `hilo`: per row, K/8
  // groups of [8 hi bf16 | 8 lo bf16], the same bytes as f32), and a SwiGLU
  // output is written that way.
  bool x_hilo = false;
  bool out_hilo = false;
  // QKV: rotate and write the cache and rope->q_out instead of `out`
  // (gemm_takes_rope; x_hilo)
  const RopeOut* rope = nullptr;
  bool unsplit = false;  // one K split, as with rope
};
// Whether a QKV launch_gemm of this shape should take RoPE and the cache write
// into its epilogue: it runs unsplit, and a head is whole pairs of 16-column tiles.
bool gemm_takes_rope(int64_t M, int64_t N, int64_t K, int64_t head_dim);

// Scratch a launch_gemm call of this shape uses: the decode GEMMs' K-slice
// partials, or the LDS-tiled GEMM's K-split sums (launch_gemm leaves a tiled
// GEMM unsplit when the scratch it is given is smaller).
// preferred: include the optional long-K splits (callers that can grow
// their scratch); false: only what the call requires.
// packed: GemmFuse::w_packed is set.
void gemm_scratch_need(int64_t M, int64_t N, int64_t K, size_t* ws_bytes, bool packed,
                       bool preferred = true);
hipError_t launch_gemm(hipStream_t st, const float* x, const uint16_t* w, const float* bias,
                       int64_t M, int64_t N, int64_t K, Epilogue ep, float* out,
                       const GemmScratch* scratch = nullptr, const GemmFuse* fuse = nullptr);

// ---- sampling (runtime/src/sampling.rs DefaultSampler) ----------------------
// Per-row SamplingParams fields the sampler reads (orion-core/src/sampling.rs).
struct SampleParams {
  float temperature;
  int32_t top_k;
  float top_p;
  float repetition_penalty;
};
constexpr int64_t kSampleMaxVocab = 262144;
// logits [rows, vocab] are filtered in place; out gets one token per row.
hipError_t launch_sample(hipStream_t st, float* logits, int64_t rows, int64_t vocab,
                         const SampleParams* params, const int64_t* prev_off,
                         const uint32_t* prev_tok, const float* uniform, int32_t* out);

// ---- elementwise / normalisation -------------------------------------------
// sumsq: when set, also the row sums of squares, one f64 per 64 columns
// (embed_sumsq_slots(hidden) per row); frag: when set, also the rows times
// next_weight in fragment order.
inline int embed_sumsq_slots(int64_t hidden) { return (int)((hidden + 63) / 64); }
hipError_t launch_embed(hipStream_t st, const uint32_t* tokens, int64_t n, const uint16_t* table,
                        int64_t hidden, float* out, double* sumsq = nullptr,
                        uint16_t* frag = nullptr, const float* next_weight = nullptr);
// The input of a launch_gemm_rows call that applies an RMSNorm, from f32 rows
// (gathered by row_index when given): embed_sumsq_slots(cols) sums of squares
// per row and, when set, the rows times weight in fragment order or a copy of
// the rows.
hipError_t launch_norm_input(hipStream_t st, const float* x, const int32_t* row_index,
                             const float* weight, int64_t rows, int64_t cols, double* sumsq,
                             uint16_t* frag, float* out_rows);
// rows selected by `row_index` (nullptr = identity)
// hilo: out holds each row as cols/8 groups of [8 hi bf16 | 8 lo bf16] (hi =
// the f32 value truncated to bf16, lo = the remainder truncated), the input
// layout of GemmFuse::x_hilo; needs cols % 8 == 0.
hipError_t launch_rmsnorm(hipStream_t st, const float* x, const int32_t* row_index,
                          const float* weight, int64_t rows, int64_t cols, float eps, float* out,
                          bool hilo = false);
hipError_t launch_rope_and_cache(hipStream_t st, const KvGeom& kv, void* arena, int64_t layer,
                                 int64_t rows, int64_t hq, const float* q_in, int64_t q_stride,
                                 float* q_out, const float* k, int64_t k_stride, const float* v,
                                 int64_t v_stride, const uint32_t* positions,
                                 const int32_t* row_seq, const int64_t* bt_off,
                                 const uint32_t* bt_ids, const float* cos_t, const float* sin_t);
hipError_t launch_silu_mul(hipStream_t st, float* gate, const float* up, int64_t count);
hipError_t launch_argmax(hipStream_t st, const float* logits, int64_t rows, int64_t cols,
                         int64_t* out);
// Copies between pinned host memory and the device in 16-byte words (both ends
// 16-byte aligned and allocated to a multiple of 16 bytes), for transfers of up
// to kHostCopyMax bytes; larger ones are a copy command's.
constexpr size_t kHostCopyMax = size_t(1) << 20;
hipError_t launch_host_copy(hipStream_t st, void* dst, const void* src, size_t bytes);
hipError_t launch_f32_to_bf16(hipStream_t st, const float* in, uint16_t* out, int64_t count);
hipError_t launch_synthetic_bf16(hipStream_t st, uint16_t* out, int64_t count, uint64_t key,
                                 float mul);
hipError_t launch_synthetic_f32(hipStream_t st, float* out, int64_t count, uint64_t key,
                                float mul);
hipError_t launch_fill_f32(hipStream_t st, float* out, int64_t count, float value);

// Synthetic-weight generator shared by host and device: splitmix64 of a
// per-tensor key plus the element index; the sum of the hash's four 16-bit
// fields (Irwin-Hall, mean 131070, sd 65536/sqrt(3)) centred and scaled.
__host__ __device__ inline uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}
__host__ __device__ inline float synthetic_normal(uint64_t key, uint64_t index, float mul) {
  const uint64_t h = splitmix64(key + index);
  const int32_t s = (int32_t)(h & 0xffff) + (int32_t)((h >> 16) & 0xffff) +
                    (int32_t)((h >> 32) & 0xffff) + (int32_t)(h >> 48);
  return (float)(s - 131070) * mul;
}
inline uint64_t synthetic_key(uint64_t seed, int which, int layer) {
  return splitmix64(seed ^ ((uint64_t)(which + 1) << 48) ^ ((uint64_t)(layer + 1) << 24));
}
constexpr float kIrwinHallSd = 37837.2265625f;  // 65536 / sqrt(3), rounded to f32

}  // namespace orion
