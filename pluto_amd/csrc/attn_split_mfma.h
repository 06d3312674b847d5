// Attention forward and backward to FP32 accuracy for bf16 queries, keys and
// values of head width 256 (attn_split_mfma.hip).
#pragma once

#include "common.h"

namespace pluto_hip {

constexpr int kSplitHeadDim = 256;

// All heads are 256 elements apart within a row.
struct SplitArgs {
  const uint16_t* q = nullptr;  // [T, heads, 256]
  const uint16_t* k = nullptr;  // [T, heads / group, 256]
  const uint16_t* v = nullptr;
  int length = 0, heads = 0, group = 1;
  float scale = 1.0f;
  float* core = nullptr;      // [T, heads, 256] attention output
  float* maxima = nullptr;    // [heads, T] of the scaled scores
  float* inverses = nullptr;  // [heads, T] 1 / normalizer
  // forward, optional: out = bf16(bf16(core) * bf16(sigmoid(gate))), [T, heads, 256], gate
  // at [T, heads, 2, 256] + 256 of qg; lse [T, heads], maximum + log(normalizer)
  uint16_t* out = nullptr;
  const uint16_t* qg = nullptr;
  float* lse = nullptr;
  // backward: the gradient of core as three bf16 tensors [T, heads, 256] whose sum
  // it is, `piece` elements apart, and its row products with core
  uint16_t* d_core = nullptr;
  long long piece = 0;
  float* deltas = nullptr;  // [heads, T]
  float* dq = nullptr;      // [T, heads, 256], one gradient per query head
  float* dk = nullptr;
  float* dv = nullptr;
};

// Rows of one head that a workgroup of 256 threads takes of the gates' backward, `d / 8` lanes
// a row: 64 where that still makes several workgroups a compute unit, fewer for shorter
// sequences, down to what the workgroup holds at once. 24 heads, 64 rows and so: 64 tokens
// 8.1 and 4.1 us at width 128, 11.0 and 4.3 at 256; 300 tokens 9.0 and 5.5, 12.5 and 9.2;
// 1024 tokens 11.0 and 9.0, 30 and 25; 3000 tokens 26.3 and 25.7, 69 and 67.
inline int gate_group_rows(int length, int heads, int d) {
  const int least = 2048 / d;
  int rows = 64;
  while (rows > least && 1LL * (length + rows - 1) / rows * heads < 2048) rows /= 2;
  return rows;
}

bool split_attention_supported(int length, int heads, int head_dim);
int launch_split_forward(hipStream_t stream, const SplitArgs& args);
// dC = dy * Round(sigmoid(gate)) into args.d_core and args.deltas;
// d gate = dy * Round(core) * s (1 - s) into the gate half of dqg.
int launch_split_gate(hipStream_t stream, const SplitArgs& args, const void* qg, const float* dy,
                      float* dqg);
int launch_split_backward(hipStream_t stream, const SplitArgs& args);

}  // namespace pluto_hip
