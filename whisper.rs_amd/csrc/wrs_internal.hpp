// Internal declarations shared by the HIP kernels and the C-ABI runtime.
//
// Layout conventions (all strides in elements, not bytes):
//   activations  element (b, h, t, d) at base + b*bs + h*hs + t*rs + d
//                (token-major [T][n_heads*d_head] rows of the reference are
//                 hs = d_head, rs = d_model; BHSD is hs = T*d_head, rs = d_head)
//   KV cache     f16 (or f32), one [ctx][64] plane per (layer, slot, head) --
//                rows of one head are contiguous 128-byte (256-byte) lines.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wrs {

enum DType : int { kF32 = 0, kF16 = 1, kBF16 = 2 };

// Activation applied by a projection's epilogue, in f32 before the output
// rounding (the reference runs gelu_inplace on the f32 projection output).
enum Act : int { kActNone = 0, kActGelu = 1 };

// GELU, tanh form, in the reference's order of operations with contraction
// off (crates/tensor/src/ops/gelu.rs:6-23; constants gelu.rs:3-4).
__device__ inline float gelu_tanh(float x) {
#pragma clang fp contract(off)
  const float kA = 0.044715f, kS = 0.7978846f;
  const float inner = kS * x * (1.0f + kA * x * x);
  return 0.5f * x * (1.0f + tanhf(inner));
}

struct Layout {
  int64_t bs;  // batch (window) stride
  int64_t hs;  // head stride
  int64_t rs;  // row (token) stride
};

// Logical workgroup id with an XCD-aware remap: the hardware hands linear ids
// round-robin to the 8 XCDs, so consecutive logical ids (the query blocks of
// one (window, head), which read the same K/V) are gathered onto one XCD and
// share its L2.
__device__ inline int xcd_remap(int pid, int nwg) {
  const int xcd = pid & 7, k = pid >> 3;
  const int per = nwg >> 3, rem = nwg & 7;
  return xcd < rem ? xcd * (per + 1) + k : rem * (per + 1) + (xcd - rem) * per + k;
}

// Agent-scope (L2-coherent across the GPU's XCDs) store and load of one
// float, for partials that another workgroup of the launch merges.
__device__ inline void st_agent(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline float ld_agent(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// x op x[lane ^ 32] and x op x[lane ^ 16] with the gfx950 lane-swap VALU
// instructions (no LDS round trip). Issued as inline asm on two distinct
// registers: the swap writes both operands.
__device__ inline void swap32(float& a, float& b) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
__device__ inline void swap16(float& a, float& b) {
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
}
__device__ inline float max_x16_x32(float x) {
  float a = x, b = x;
  swap16(a, b);  // a, b: x of this row and of the row 16 lanes away
  x = fmaxf(a, b);
  a = x;
  b = x;
  swap32(a, b);
  return fmaxf(a, b);
}
__device__ inline float sum_x16_x32(float x) {
  float a = x, b = x;
  swap16(a, b);
  x = a + b;
  a = x;
  b = x;
  swap32(a, b);
  return a + b;
}

// Flash-attention prefill over full query/key sequences
// (crates/tensor/src/ops/attention.rs:68-243 semantics).
struct PrefillArgs {
  const void* q;
  const void* k;
  const void* v;
  float* o;
  Layout lq, lk, lv, lo;
  int batch, n_heads, t_q, t_kv, d_head;
  int causal;        // mask keys j > i + q_pos_offset
  int q_pos_offset;  // absolute position of query row 0 (decoder prompt: t_past)
  float scale;       // 1/sqrt(d_head), rounded to f32 like attention.rs:107
  // Schedule overrides from the context (wrs_attn_set_schedule): queries per
  // workgroup of the 16-bit kernel (0 = by grid size), and the f32 kernel's
  // key split (-1 = by grid size, 0 = 128-query blocks, 1 = four waves,
  // 2..4 = that many waves, 5 = four waves over several workgroups).
  int force_queries;
  int force_f32_split;
  // Context scratch for grids whose blocks split their keys over several
  // workgroups (null when none is available): partials and merge counters
  // (zero between launches), with their sizes.
  float* split_part;
  size_t split_part_floats;
  unsigned* split_counters;
  size_t split_counter_words;
};

// MFMA f16/bf16 kernel, d_head == 64, q/k/v of one 16-bit type, rows 16-byte
// aligned; prefill_mfma16_supports() states the remaining shape limits.
bool prefill_mfma16_supports(const PrefillArgs& a);
// Scratch the 16-bit kernel's schedule for `a` uses (floats of partials and
// words of counters), both 0 when it uses none.
void prefill_mfma16_scratch(const PrefillArgs& a, size_t* part_floats, size_t* counter_words);
// The sizes the context allocates at least: enough for every grid whose
// blocks the default schedule splits over workgroups.
size_t prefill_split_floats_min();
size_t prefill_split_words_min();
hipError_t launch_prefill_mfma16(const PrefillArgs& a, DType dt, hipStream_t s);
// f32-accumulate-check kernel on f32 MFMA: q f32, k/v f32|f16|bf16 widened
// exactly to f32, any d_head <= 128.
hipError_t launch_prefill_f32(const PrefillArgs& a, DType q_dt, DType kv_dt, hipStream_t s);
// Scratch its schedule for `a` uses (as prefill_mfma16_scratch).
void prefill_f32_scratch(const PrefillArgs& a, size_t* part_floats, size_t* counter_words);

// Exact reference decode semantics on f32 K/V (attention.rs:246-434
// single_token_mha_d64 and decoder.rs:835-892): full score row, softmax with
// reciprocal multiply, weights < 1e-7 skipped. Rows come in groups of
// rows_per_group that share one K/V base (goff[g] elements past k and v);
// row i of group g sees keys [0, glen[g] + i * limit_step). Host slices are
// one group of token-major rows (kv_rs = d_model, kv_hs = d_head); the f32
// arena passes [head][ctx][64] planes (kv_rs = 64, kv_hs = the plane).
constexpr int kMaxExactGroups = 64;
struct ExactArgs {
  const float* q;
  const float* k;
  const float* v;
  float* o;
  int64_t q_rs, o_rs;   // row strides of q and out (head h at h * d_head)
  int64_t kv_rs, kv_hs;  // K/V: key row and head strides
  int n_rows, n_heads, d_head;
  int rows_per_group, n_groups, limit_step;
  float scale;
  // Scratch, as decode_exact_scratch sizes it.
  float* scores;  // [n_rows][n_heads][scores_stride]
  int64_t scores_stride;
  int n_chunks;
  float* stats;        // [n_rows][n_heads][n_chunks] (max, sum)
  float* part;         // [n_rows][n_heads][n_chunks][64]
  unsigned* counters;  // zero between launches
  int64_t goff[kMaxExactGroups];
  int glen[kMaxExactGroups];
};
constexpr int kOneKeys = 512;  // d_head 64: keys a row that one workgroup takes, without scratch
struct ExactScratch {
  size_t scores, stats, part, counter_words;  // floats, floats, floats, words
  int chunks;
};
ExactScratch decode_exact_scratch(int n_rows, int n_heads, int d_head, int max_keys, int n_groups,
                                  int rows_per_group);
size_t exact_scratch_bytes(size_t scores);
size_t exact_counter_words(size_t bytes);
hipError_t launch_decode_exact_f32(const ExactArgs& a, hipStream_t s);

// Split-K decode over an f16 KV cache: one query row per (group, row),
// all rows of a group share one K/V plane set (cross-attention: the beams of
// one utterance; self-attention: one row per slot).
constexpr int kMaxDecodeGroups = 64;
constexpr int kMaxRowsPerGroup = 8;
struct DecodeArgs {
  const float* q;   // row (g*rows_per_group + r): q + row*q_rs + h*64
  float* o;         // same indexing with o_rs
  const _Float16* k;  // plane (g, h): k + goff[g] + h*kv_hs, key j at +j*64
  const _Float16* v;
  int64_t q_rs, o_rs, kv_hs;
  int64_t goff[kMaxDecodeGroups];  // per-group plane offset (elements)
  int len[kMaxDecodeGroups];       // keys visible to group g
  int n_groups, rows_per_group, n_heads;
  int n_rows;    // query rows: the last group may hold fewer than rows_per_group
  int chunk;     // keys per workgroup (kDecodeChunk or kDecodeChunkLong)
  int n_splits;  // workgroups per (group, head) = ceil(max len / chunk)
  float scale_log2;  // (1/8) * log2(e)
  float* part;        // scratch: [groups][heads][splits][rows][68]
  unsigned* counters;  // scratch: one per (group, head) every 32 words, zero between launches
  // Optional: row statistics (max, sum of exp2(s - max)) of output row
  // lse_row0 + g*rows_per_group + r for head h at lse[2 * (h * lse_rows + row)].
  float* lse;
  int lse_rows, lse_row0;
};
constexpr int kDecodeChunk = 128;
constexpr int kDecodeChunkLong = 256;  // one workgroup per (group, head) up to this length
hipError_t launch_decode_f16(const DecodeArgs& a, hipStream_t s);
size_t decode_part_floats(int n_groups, int n_heads, int n_splits, int rows);
size_t decode_counter_words(int n_groups, int n_heads);

// Prompt rows over the f16 cache: query row i, head h at q + i*q_rs + h*64 (any
// dword) against n_keys keys of plane k + h*kv_hs (key j at +j*64). With causal,
// row i sees keys j < pos0 + i + 1 (the cached self-attention: three-part
// operands); without, every key (two parts, like the split-K decode).
struct RowsArgs {
  const float* q;
  float* o;  // same indexing with o_rs
  const _Float16* k;
  const _Float16* v;
  int64_t q_rs, o_rs, kv_hs;
  int n_rows, n_heads, n_keys;
  int causal, pos0;
  float scale_log2;  // (1/8) * log2(e)
  float* lse;        // optional: (max, sum of exp2(s - max)) at lse[2 * (h * n_rows + row)]
};
hipError_t launch_attend_rows(const RowsArgs& a, hipStream_t s);
// One past the keys a launch takes (32-bit plane offsets).
constexpr size_t kRowsMaxKeys = (size_t{1} << 24) - 4095;

// Measurement: a streaming read of `bytes` (multiple of 16, 16-byte aligned)
// with the split-K decode's grid shape (512 threads x 64 bytes per
// workgroup); sink receives stream_read_blocks(bytes) floats.
hipError_t launch_stream_read(const void* src, int64_t bytes, float* sink, hipStream_t s);
int64_t stream_read_blocks(int64_t bytes);
// The same with `threads` per workgroup (256, 512, 1024) and `loads` 16-byte
// loads per lane (1, 2, 4, 8, 16, 24).
hipError_t launch_stream_read_shape(const void* src, int64_t bytes, int threads, int loads,
                                    float* sink, hipStream_t s);
int64_t stream_read_shape_blocks(int64_t bytes, int threads, int loads);

// Alignment-head capture over the f16 cross plane
// (decoder.rs:796-828 semantics): for query row i and pair p,
// softmax_j(dot(q_i[head_p], k_j[head_p]) * scale) into
// out[((row_offset + i) * n_selected + slot_p) * n_audio + j].
constexpr int kCaptureRows = 16;       // query rows per workgroup
constexpr int kCaptureChunk = 128;     // keys per workgroup
constexpr int kMaxCapturePairs = 32;   // (slot, head) pairs per launch
struct CaptureArgs {
  const float* q;     // row i, head h: q + i*q_rs + h*64
  const _Float16* k;  // plane of head h: k + h*kv_hs, key j at +j*64
  const float* k32;   // the same for f32 planes (capture_cross_f32)
  float scale;        // 1/sqrt(64), capture_cross_f32
  float* out;
  float* part;        // scratch: capture_part_floats(n_pairs, n_tokens, n_audio)
  int64_t q_rs, kv_hs;
  int n_tokens, n_audio, n_selected, row_offset, n_pairs;
  float scale_log2;  // log2(e)/sqrt(64): decoder.rs:810's scale in the exp2 domain
  // When set: per-row softmax statistics of the attention pass over the same q
  // and keys, (max, sum) in the exp2 domain at lse[2 * (head * n_tokens + row)];
  // the capture then runs as one pass.
  const float* lse;
  int slot[kMaxCapturePairs];
  int head[kMaxCapturePairs];
};
size_t capture_part_floats(int n_pairs, int n_tokens, int n_audio);
hipError_t launch_capture_cross_f16(const CaptureArgs& a, hipStream_t s);
// Over f32 planes (k32, scale; no part, no lse): one workgroup per (row, pair).
hipError_t launch_capture_cross_f32(const CaptureArgs& a, hipStream_t s);

// Projections with f16 weights (quant.rs:415-473 semantics):
// out(t, r) = row_scale[t] * (W[r] . x'[t]) + bias[r] with W [n_out][n_in] f16
// and x' [n_tokens][parts n_in] f16 (one part, or the kSplitParts parts of split
// f32 rows, whose products with the same weights add up). Element (t, r) is stored at
// out + t*out_rs + (r/64)*out_hs + r%64. Groups share x and differ in W, bias
// and out (all layers' cross K and V in one launch).
constexpr int kLinearK = 64;          // n_in must be a multiple of this
constexpr int kSplitParts = 2;        // f16 parts of a split f32 row: hi, lo
constexpr int kMaxLinearGroups = 64;
struct LinearArgs {
  const _Float16* x;
  int64_t x_rs;
  const float* row_scale;  // nullable: 1
  int n_tokens, n_in, n_out, parts, n_groups;
  int64_t out_rs, out_hs;
  int act;  // Act, applied after the bias
  // Scratch for tiles whose k is split over workgroups (null: no split):
  // partial sums and merge counters (zero between launches), with their sizes.
  float* part;
  size_t part_floats;
  unsigned* counters;
  size_t counter_words;
  const _Float16* w[kMaxLinearGroups];
  const float* bias[kMaxLinearGroups];  // nullable entries
  void* out[kMaxLinearGroups];
};
hipError_t launch_linear_f16w(const LinearArgs& a, DType out_dt, hipStream_t s);
// Whether the launch splits k when it is given scratch, and the scratch that
// serves every such launch.
bool linear_needs_split(const LinearArgs& a);
size_t linear_split_floats();
size_t linear_split_words();
// Decode-sized batches (n_tokens <= kGemvMaxRows) of the same product on the
// f16 weight stream; x is f32 or f16 with row stride x_rs, no split needed.
constexpr int kGemvMaxRows = 8;
// Weight groups that a launch's arguments have room for: the arguments are copied, and
// these launches are host-bound in a step that is not captured. Room for 64 groups cost
// 0.5 us of a 6.7 us call (5 rows 768 x 768), room for 8 is what a layer's projections
// need (3). More groups still run in one launch, of the same kernels on larger arguments.
constexpr int kFewGemvGroups = 8;
constexpr int kGemvLnMax = 1280;  // longer f32 rows do not fit the decode kernels' registers
constexpr int kGemvXFloats = 40960;  // n_tokens * n_in staged in LDS (160 KB)
template <int kGroups>
struct GemvArgs {
  const void* x;
  int64_t x_rs;
  int n_tokens, n_in, n_out, n_groups;
  int64_t out_rs, out_hs;
  // Optional LayerNorm of every x row before the product (norm.rs:116-143,
  // the layer_norm_rows arithmetic exactly; f32 x only): ln_g null = none.
  const float* ln_g;
  const float* ln_b;
  float ln_eps;
  int act;  // Act, applied after the bias
  const _Float16* w[kGroups];
  const float* bias[kGroups];
  void* out[kGroups];
};
// kGroups: kFewGemvGroups or kMaxLinearGroups.
template <int kGroups>
hipError_t launch_gemv_f16w(const GemvArgs<kGroups>& a, DType x_dt, DType out_dt, hipStream_t s);
// Whether a fused LayerNorm is better taken out of such a launch (any number of groups).
bool gemv_norms_apart(int n_tokens, int n_in, int n_out, int n_groups);
// f32 rows -> [hi | lo] f16 rows (kSplitParts n_in each) and per-row 2^-shift,
// normalized first when ln_g is set (n_in <= kSplitLnMax; gamma and beta
// 16-byte aligned).
constexpr int kSplitLnMax = 2048;
hipError_t launch_linear_split(const float* x, int64_t x_rs, int n_tokens, int n_in,
                               const float* ln_g, const float* ln_b, float ln_eps, _Float16* xs,
                               float* row_scale, hipStream_t s);

// LayerNorm over f32 rows (norm.rs:116-143), output f32/f16/bf16 rows of d;
// d % 4 == 0, rows 16-byte aligned.
hipError_t launch_layer_norm(const float* x, const float* gamma, const float* beta, float eps,
                             int n_tokens, int d, DType out_dt, void* out, hipStream_t s);
// GELU, tanh form, in place on f32 (gelu.rs:11-23); data 16-byte aligned.
hipError_t launch_gelu(float* data, int64_t n, hipStream_t s);

// Zero fills issued as kernels (never as memset nodes, so that a caller may
// capture them into a graph): f32 element (b, h, r, c) at
// base + b*bs + h*hs + r*rs + c for c < cols; and n 32-bit words.
hipError_t launch_fill_zero_rows(float* base, int64_t bs, int64_t hs, int64_t rs, int batch,
                                 int n_heads, int n_rows, int cols, hipStream_t s);
hipError_t launch_fill_zero_u32(unsigned* p, int64_t n, hipStream_t s);

// KV arena kernels.
// f32 rows [n][d_model] of K and of V (row stride src_rs) -> planes, f16 or f32:
// head h, row i at dst + h*dst_hs + (pos + i)*64.
struct KvRows {
  const float *k_src, *v_src;
  void *k_dst, *v_dst;
};
hipError_t launch_kv_write_rows(const KvRows& rows, bool f32, int64_t src_rs, int n, int n_heads,
                                int64_t dst_hs, int pos, hipStream_t s);
// K and V planes of one slot: plane (l, h) at base + l*layer_stride +
// h*plane_stride, in rows of 64 f16 (an f32 plane is passed as twice the rows
// and strides).
// Move rows [drop, len) of every plane down to [0, len - drop).
hipError_t launch_kv_slide(_Float16* k, _Float16* v, int64_t layer_stride, int64_t plane_stride,
                           int n_layers, int n_heads, int len, int drop, hipStream_t s);
// Copy rows [0, len) of every plane from src to dst (same plane geometry).
hipError_t launch_kv_copy_planes(const _Float16* k_src, _Float16* k_dst, const _Float16* v_src,
                                 _Float16* v_dst, int64_t layer_stride, int64_t plane_stride,
                                 int n_layers, int n_heads, int len, hipStream_t s);

}  // namespace wrs
