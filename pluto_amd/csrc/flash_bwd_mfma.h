// Launcher of the bf16 MFMA flash-attention backward kernels.
#pragma once

#include "attn_generic.h"

namespace pluto_hip {

// Heads are D elements apart within a row, sequences context_length rows.
struct FlashBackwardArgs {
  const uint16_t* q = nullptr;  // rows q_row elements apart
  const uint16_t* k = nullptr;  // rows kv_row elements apart, num_heads / group heads
  const uint16_t* v = nullptr;
  long long q_row = 0, kv_row = 0;
  int group = 1;  // query heads per key/value head
  // Either the FP32 upstream gradient and the stored output [rows, E]: the
  // query-owned kernel then fills d_out_bf16, deltas and lse2; or d_out null:
  // the caller has filled them.
  const float* d_out = nullptr;
  const uint16_t* out = nullptr;
  const float* maxima = nullptr;
  const float* normalizers = nullptr;
  uint16_t* d_out_bf16 = nullptr;  // [rows, E]
  float* deltas = nullptr;         // [sequences * H, T]: -sum(dO * O)
  float* lse2 = nullptr;           // same shape: -(log2-sum-exp) / (scale log2 e)
  // one gradient per query head, also for keys and values
  float* dq = nullptr;
  float* dk = nullptr;
  float* dv = nullptr;
  long long dq_row = 0, dkv_row = 0;
  int sequences = 0, context_length = 0, num_heads = 0, head_dim = 0;
  float scale = 1.0f;
};

// The packed [rows, 3E] operands of the multi-head layer.
FlashBackwardArgs packed_flash_backward(const GenericBackwardArgs& args, float* lse2,
                                        uint16_t* d_out_bf16);
bool flash_backward_supported(const FlashBackwardArgs& args);
int launch_flash_backward(hipStream_t stream, const FlashBackwardArgs& args);
// The key-owned kernels with a hand-scheduled main loop, heads of 64 or 128 channels
// (flash_dkv_wide.hip); they read what the query-owned kernel left in lse2, deltas
// and d_out_bf16.
int launch_flash_dkv_wide(hipStream_t stream, const FlashBackwardArgs& args);
// The query-owned kernel for heads of 128 channels (flash_dq_wide.hip).
int launch_flash_dq_wide(hipStream_t stream, const FlashBackwardArgs& args);

}  // namespace pluto_hip
