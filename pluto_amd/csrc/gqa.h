// Argument blocks and launchers of the Qwen grouped-query attention kernels.
#pragma once

#include "common.h"

namespace pluto_hip {

constexpr int kDecodeBatchMax = 64;  // sequences per decode launch

struct CacheView {
  void* keys = nullptr;
  void* values = nullptr;
  int dtype = PLUTO_HIP_BF16;
  long long token_stride = 0;
  long long head_stride = 0;
};

struct PrefillPrepareArgs {
  const void* qg = nullptr;  // bf16 [T, qh, 2, d]
  const void* k = nullptr;   // bf16 [T, kh, d]
  const void* v = nullptr;   // bf16 [T, kh, d]
  const float* q_norm = nullptr;
  const float* k_norm = nullptr;
  float* cosines = nullptr;  // scratch for the rotation's table [T, rotary/2]
  float* sines = nullptr;
  bool keep_table = false;   // the caller reads the table afterwards
  float theta = 10000.0f;
  void* q_out = nullptr;  // [T, qh, d], bf16 when rounding, else fp32
  int q_out_dtype = PLUTO_HIP_BF16;
  CacheView cache;
  // optional second copies for the backward pass, in one block with the table: the prepared queries
  // [T, qh, d] as q_out, keys and values [T, kh, d] in the cache's storage
  void* q_copy = nullptr;
  void* k_copy = nullptr;
  void* v_copy = nullptr;
  int length = 0, start_position = 0;
  int query_heads = 0, key_value_heads = 0, head_dim = 0, rotary_dim = 0;
  float epsilon = 1e-6f;
  bool round = true;
};

// Per-launch slice of a decode batch, passed by value as a kernel argument.
struct DecodeBatch {
  int count = 0;
  int sequence[kDecodeBatchMax];  // index of entry i in the full batch
  int positions[kDecodeBatchMax];
  void* keys[kDecodeBatchMax];
  void* values[kDecodeBatchMax];
  int block_start[kDecodeBatchMax + 1];  // prefix sum of split-K blocks
  uint16_t split[kDecodeBatchMax];       // cache rows a block
};

struct DecodePrepareArgs {
  const void* q_gate = nullptr;  // [batch, qh, 2, d]
  const void* k = nullptr;       // [batch, kh, d]
  const void* v = nullptr;
  int io_dtype = PLUTO_HIP_F32;
  const float* q_norm = nullptr;
  const float* k_norm = nullptr;
  void* q_out = nullptr;  // [batch, qh, d]
  int q_out_dtype = PLUTO_HIP_BF16;
  int cache_dtype = PLUTO_HIP_BF16;
  long long token_stride = 0, head_stride = 0;
  int query_heads = 0, key_value_heads = 0, head_dim = 0, rotary_dim = 0;
  float epsilon = 1e-6f, theta = 1e7f;
  bool round = true;
};

// Split-K block sizes of the decode step: a multiple of 64 up to 512 cache
// rows, or the size the fused kernel is specialised for at this head width.
// At head width 256 one workgroup occupies a compute unit alone, so nothing
// covers the time it spends starting up and handing over its partial results;
// blocks of 1024 rows halve that share (0.435 -> 0.412 ms at 32 sequences of
// 1024..32768 tokens, 24 / 4 heads).  At the narrower widths three workgroups
// share a compute unit and 512 rows measure best.
constexpr int decode_split_default(int head_dim) { return head_dim == 256 ? 1024 : 512; }
constexpr bool decode_split_valid(int head_dim, int split) {
  return split >= 64 && split % 64 == 0 &&
         (split <= 512 || split == decode_split_default(head_dim));
}
// The block size of a sequence of `rows` rows where the caller leaves it to the
// library.  It depends on nothing but the sequence itself, so that a sequence's result
// does not change with the batch it is decoded in.  A block's rows are read one after
// the other and a sequence's blocks are added up one after the other, so the best size
// for a sequence alone grows with the square root of its length (head width 256: 128
// rows at 777, 18 us against 35 in one block of 1024; 256 at 4096, 26 against 39), and
// a full chip wants larger blocks, of which it starts fewer (32 sequences of 777 rows:
// 45 us in blocks of 128, 42 of 192, 36 of 256).  8 sqrt(rows) at head width 256 and 10
// sqrt(rows) below, to the nearest 64, lie between: batches of 1 to 32 with lengths
// spread to 32768 take 3.5 % longer on average than with a size picked for the whole
// batch, between 9 % less and 14 % more.  The default sizes have loops of their own: at the narrower widths they are faster
// than anything from 320 up (64 sequences of 2048 rows at width 64: 27 us, 34 in blocks of
// 448), at 256 beyond 16384 rows for all but a sequence or two.
constexpr int decode_split_for(int head_dim, int rows) {
  const long long factor = head_dim == 256 ? 8 : 10;
  if (head_dim == 256 && rows > 16384) return decode_split_default(head_dim);
  long long split = 64;
  while (split < 512 && factor * factor * rows > (split + 32) * (split + 32)) split += 64;
  return head_dim != 256 && split > 256 ? decode_split_default(head_dim) : static_cast<int>(split);
}
// The blocks of such a sequence.
constexpr int decode_blocks_for(int head_dim, int rows) {
  const int split = decode_split_for(head_dim, rows);
  return static_cast<int>((static_cast<long long>(rows) + split - 1) / split);
}
// The most blocks a sequence of up to `rows` rows has: where the size steps up, the
// blocks become fewer.
constexpr int decode_blocks_up_to(int head_dim, int rows) {
  int most = decode_blocks_for(head_dim, rows);
  const int factor = head_dim == 256 ? 8 : 10;
  for (int split = 64; split < 512; split += 64) {
    const int last = (split + 32) * (split + 32) / (factor * factor);  // longest with this size
    if (last < rows) most = most > decode_blocks_for(head_dim, last) ? most : decode_blocks_for(head_dim, last);
  }
  if (head_dim == 256 && rows > 16384) most = most > 32 ? most : 32;
  return most;
}

// The fused decode step (preparation of the new token, split-K attention over
// the cache, combine and gate in the workgroup that finishes a (sequence, kv
// head) last).
struct DecodeArgs {
  const void* q_gate = nullptr;  // [batch, qh, 2, d]
  const void* k = nullptr;       // [batch, kh, d]
  const void* v = nullptr;
  int io_dtype = PLUTO_HIP_F32;  // storage of q_gate, k, v and out
  const float* q_norm = nullptr;
  const float* k_norm = nullptr;
  void* out = nullptr;  // [batch, qh, d]
  long long token_stride = 0, head_stride = 0;  // of the bf16 caches
  int query_heads = 0, key_value_heads = 0, head_dim = 0, rotary_dim = 0;
  float epsilon = 1e-6f;
  float scale = 1.0f;
  // partial results of split-K block i (global index block_start[b] + j,
  // kv head g): o [block, kh, group, d], m and l [block, kh, group]
  float* part_o = nullptr;
  float* part_m = nullptr;
  float* part_l = nullptr;
  // one counter per (sequence, kv head) of the whole batch: zero when the
  // kernel starts, and zero again when it ends
  unsigned* arrivals = nullptr;
  long long block_base = 0;  // global index of this launch's first block
  // theta^(-2 f / rotary) for f < rotary / 2, evaluated on the host in FP64
  double inverse_frequency[128];
};

int launch_prefill_prepare(hipStream_t stream, const PrefillPrepareArgs& args);
int launch_decode_prepare(hipStream_t stream, const DecodePrepareArgs& args,
                          const DecodeBatch& batch);
bool decode_fast_supported(int head_dim, int group);
int launch_decode_fast(hipStream_t stream, const DecodeArgs& args,
                       const DecodeBatch& batch);
// Zeroes `count` arrival counters (a launch of its own: the fused kernel needs
// them zero, and leaves them zero).
// `always`: also when the test-support kernel mask has switched auxiliary kernels off
int launch_decode_clear(hipStream_t stream, unsigned* arrivals, int count, bool always = false);
// Two-pass probability rows (any dtype, any shape): row r of `rows` sees the
// first `first_visible + r` cache rows; output fp32 [query_heads, rows,
// row_width], zero beyond the visible prefix
// (AttentionProbabilitiesKernel, cached_attention_ops.cc:131-178; the probs
// tensor of ForwardKernel, qwen_attention.cc:68-119).
int launch_attention_probabilities(hipStream_t stream, const void* q, int q_dtype,
                                   const CacheView& cache, int query_heads,
                                   int key_value_heads, int head_dim, int rows,
                                   int first_visible, int row_width, float scale,
                                   float* probabilities);

// Pieces of the whole-sequence backward (gqa_backward.hip).
int launch_pack_heads(hipStream_t stream, const float* q, const float* k, const float* v, int length,
                      int query_heads, int key_value_heads, int head_dim, float* packed);
int launch_gate_backward(hipStream_t stream, const void* qg, const float* core, const float* dy,
                         int length, int query_heads, int head_dim, bool round, float* dc, float* dqg);
// The same for the matrix-core backward (head widths 64 and 128).
int launch_gate_rows(hipStream_t stream, const void* qg, const void* core, const float* dy,
                     const float* maxima, const float* normalizers, int length, int query_heads,
                     int head_dim, float scale2, uint16_t* dc, float* dqg, float* deltas,
                     float* lse2);
// The attention gradients the norm backward starts from: one dQ, dK and dV per
// query head, heads d elements apart, rows as given.
struct NormBackwardGrads {
  const float* dq = nullptr;
  const float* dk = nullptr;
  const float* dv = nullptr;
  long long dq_row = 0, dkv_row = 0;
};
// Workgroups of the norm backward at most: `partial` holds a row of head_dim
// floats for each.  (1536 workgroups of four waves are six waves a SIMD.)
constexpr int kNormQueryBlocks = 1024, kNormKeyBlocks = 512;
int launch_norm_rope_backward(hipStream_t stream, const void* qg, const void* k,
                              const float* q_norm, const float* k_norm,
                              const NormBackwardGrads& grads, const float* cosines,
                              const float* sines, int length, int query_heads, int key_value_heads,
                              int head_dim, int rotary_dim, float epsilon, float* dqg, float* dk,
                              float* dv, float* dq_norm, float* dk_norm, float* partial);

}  // namespace pluto_hip
