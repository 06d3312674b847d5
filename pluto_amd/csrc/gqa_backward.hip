// Backward of the whole-sequence Qwen GQA layer
// (QwenAttentionLayer::SequenceBackward, src/llm/layers/qwen_attention.cc:
// 450-499 and its kernels :124-239), without the reference's two quadratic
// buffers (saved probabilities and score gradients).
//
// The attention core of the backward is the multi-head kernel pair of this
// library.  The matrix-core pair reads each kv head's K and V where they lie; the
// FP32 kernels run on a packed [T, 3 * qh * d] view in which every query head
// carries a copy of them.  Both leave one dK and dV per query head, which are
// summed per kv head in ascending head order.  Around it:
//   gate_backward_kernel, gate_rows_kernel   GateBackwardKernel  (:124-141)
//   pack_heads_kernel                        layout only
//   norm_rope_*_kernel                       NormBackwardKernel  (:201-228), fused
//                                            with the per-kv-head sums and the first
//                                            level of ReduceNormKernel (:230-239)
//   norm_weight_kernel                       its second level, fixed order
#include "attn_split_mfma.h"
#include "gqa.h"
#include "mfma_tile.h"

namespace pluto_hip {
namespace {

// [T, qh, d] prepared queries, [T, kh, d] prepared keys and values ->
// packed [T, 3E] (E = qh * d): Q | K of the head's kv head | V of it.  Moved in
// pieces of PIECE elements (16 bytes when the head width allows).
template <int PIECE>
__global__ void __launch_bounds__(256)
pack_heads_kernel(const float* q, const float* k, const float* v, int length, int qh, int kh, int d,
                  float* packed) {
  struct alignas(sizeof(float) * PIECE) Piece {
    float e[PIECE];
  };
  const int pieces_per_head = d / PIECE;
  const long long pieces_per_part = 1LL * qh * pieces_per_head;
  const long long total = 3LL * length * pieces_per_part;
  const int group = qh / kh;
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < total; i += 256LL * gridDim.x) {
    const long long t = i / (3 * pieces_per_part);
    const long long within = i % (3 * pieces_per_part);
    const int part = static_cast<int>(within / pieces_per_part);
    const int h = static_cast<int>((within % pieces_per_part) / pieces_per_head);
    const int c = static_cast<int>(within % pieces_per_head) * PIECE;
    const float* source = part == 0 ? q + (t * qh + h) * d + c
                                    : (part == 1 ? k : v) + (t * kh + h / group) * d + c;
    *reinterpret_cast<Piece*>(packed + i * PIECE) = *reinterpret_cast<const Piece*>(source);
  }
}

// dC = dy * Round(sigmoid(gate)); d gate = dy * Round(core) * s (1 - s).
__global__ void __launch_bounds__(256)
gate_backward_kernel(const uint16_t* qg, const float* core, const float* dy, long long elements,
                     int d, bool round, float* dc, float* dqg) {
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < elements; i += 256LL * gridDim.x) {
    const long long unit = i / d;  // (row, head)
    const int c = static_cast<int>(i % d);
    const float gate = bf16_bits_to_float(qg[(unit * 2 + 1) * d + c]);
    const float sigmoid = 1.0f / (1.0f + expf(-gate));
    const float grad = dy[i];
    float value = core[i];
    if (round) value = round_to_bf16(value);
    dc[i] = grad * (round ? round_to_bf16(sigmoid) : sigmoid);
    dqg[(unit * 2 + 1) * d + c] = grad * value * sigmoid * (1.0f - sigmoid);
  }
}

// The same for the matrix-core kernels, which take dC as bf16 together with two
// values of each row: -sum(dC * core) and the row's log2-sum-exp in the form
// FlashBackwardArgs states.  Sixteen bytes of bf16 a lane, D / 8 lanes a row; a
// workgroup walks `rows` rows of one head, whose statistics are then contiguous.
// 350 MB in and out at T = 8192, 24 heads of 128; written as an FP32 dC that
// the query-owned kernel read again in pieces of its own rows, the same work moved
// 550 MB (83 us for this pass alone).  WIDE: every tensor is 16-byte aligned.
template <int D, bool WIDE>
__global__ void __launch_bounds__(256)
gate_rows_kernel(const uint16_t* __restrict__ qg, const uint16_t* __restrict__ core,
                 const float* __restrict__ dy, const float* __restrict__ maxima,
                 const float* __restrict__ normalizers, int length, int rows, int heads, float scale2,
                 uint16_t* __restrict__ dc, float* __restrict__ dqg, float* __restrict__ deltas,
                 float* __restrict__ lse2) {
  constexpr int LANES = D / 8, ROWS = 256 / LANES;
  const int piece = threadIdx.x % LANES, head = blockIdx.y;
  for (int i = 0; i < rows; i += ROWS) {
    const int row = blockIdx.x * rows + i + threadIdx.x / LANES;
    const bool exists = row < length;
    const long long unit = 1LL * min(row, length - 1) * heads + head;
    float grad[8], gates[8], values[8];
    load8<WIDE>(dy + unit * D + 8 * piece, grad);
    load8<WIDE>(qg + (unit * 2 + 1) * D + 8 * piece, gates);
    load8<WIDE>(core + unit * D + 8 * piece, values);
    float scaled[8], gate_grad[8];
    float dot = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float sigmoid = 1.0f / (1.0f + expf(-gates[e]));
      scaled[e] = grad[e] * round_to_bf16(sigmoid);
      gate_grad[e] = grad[e] * values[e] * sigmoid * (1.0f - sigmoid);
      dot += scaled[e] * values[e];
    }
#pragma unroll
    for (int offset = LANES / 2; offset > 0; offset >>= 1) dot += __shfl_xor(dot, offset, 64);
    if (!exists) continue;
    *reinterpret_cast<uint4*>(dc + unit * D + 8 * piece) =
        make_uint4(pack_bf16(scaled[0], scaled[1]), pack_bf16(scaled[2], scaled[3]),
                   pack_bf16(scaled[4], scaled[5]), pack_bf16(scaled[6], scaled[7]));
    store8<WIDE>(dqg + (unit * 2 + 1) * D + 8 * piece, gate_grad);
    if (piece == 0) {
      const long long at = 1LL * head * length + row;
      const float normalizer = normalizers[at];
      deltas[at] = -dot;
      lse2[at] = -(maxima[at] * kLog2e + __log2f(normalizer > 0.0f ? normalizer : 1.0f)) / scale2;
    }
  }
}

// What one of the two halves (queries, keys) of the norm backward works on.
struct NormSide {
  const uint16_t* input = nullptr;  // raw bf16 rows, `input_stride` apart
  const float* weight = nullptr;    // zero-centred norm weight [d]
  float* dx = nullptr;              // rows `input_stride` apart
  float* partial = nullptr;         // optional [blocks, d]: sums of the weight's gradient
  float* weight_grad = nullptr;
  int heads = 0, input_stride = 0, blocks = 0;
};
struct NormBackwardArgs {
  NormSide queries, keys;
  NormBackwardGrads grads;
  const float* cosines = nullptr;  // [T, rotary/2]
  const float* sines = nullptr;
  float* dv = nullptr;  // [T, kh, d]
  int length = 0, d = 0, rotary = 0, group = 0;
  float epsilon = 1e-6f;
};

// Both kernels below: the first `queries.blocks` workgroups take the (row, head)
// units of the queries, whose gradient is the head's dQ, the others those of
// the keys, where the gradients of the kv head's `group` copies are summed in
// ascending head order, for dK (which continues through RoPE and the norm) and
// for dV (which is final).  A workgroup walks units blocks apart and keeps its
// share of the weight's gradient in registers, so nothing per row is stored for
// it (a stored row each cost 100 MB out and, summed by 128 workgroups, 620 us
// back in at T = 8192, 24 heads of 128).

// D / 8 lanes a unit, eight channels a lane; RoPE partners are whole pieces.
template <int D>
__global__ void __launch_bounds__(256)
norm_rope_rows_kernel(NormBackwardArgs a) {
  constexpr int LANES = D / 8, UNITS = 256 / LANES;
  __shared__ float sums[UNITS][D];
  const bool key_mode = static_cast<int>(blockIdx.x) >= a.queries.blocks;
  const NormSide side = key_mode ? a.keys : a.queries;
  const int block = blockIdx.x - (key_mode ? a.queries.blocks : 0);
  const int piece = threadIdx.x % LANES, slot = threadIdx.x / LANES, c = 8 * piece;
  const int half = a.rotary / 2;
  const bool rotated = c < a.rotary, lower = c < half;
  const int frequency = lower ? c : c - half;
  // the lane of the same unit that holds the RoPE partner's piece
  const int partner = threadIdx.x % 64 - piece + (rotated ? (lower ? c + half : c - half) / 8 : piece);
  float factor[8], weight_sum[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    factor[e] = 1.0f + side.weight[c + e];
    weight_sum[e] = 0.0f;
  }
  const long long units = 1LL * a.length * side.heads;
  for (long long first = 1LL * block * UNITS; first < units; first += 1LL * side.blocks * UNITS) {
    const bool exists = first + slot < units;
    const long long unit = exists ? first + slot : units - 1;
    const long long row = unit / side.heads;
    const int head = static_cast<int>(unit % side.heads);
    float x[8], g[8];
    load8<true>(side.input + unit * side.input_stride + c, x);
    if (!key_mode) {
      load8<true>(a.grads.dq + row * a.grads.dq_row + head * D + c, g);
    } else {
      const long long at = row * a.grads.dkv_row + 1LL * head * a.group * D + c;
      float value_sum[8], key[8], value[8];
      load8<true>(a.grads.dk + at, g);
      load8<true>(a.grads.dv + at, value_sum);
      for (int copy = 1; copy < a.group; ++copy) {
        load8<true>(a.grads.dk + at + copy * D, key);
        load8<true>(a.grads.dv + at + copy * D, value);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          g[e] += key[e];
          value_sum[e] += value[e];
        }
      }
      if (exists) store8<true>(a.dv + unit * D + c, value_sum);
    }
    float squares = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) squares += x[e] * x[e];
    float normalized[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) normalized[e] = g[e];
    float other[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) other[e] = __shfl(g[e], partner, 64);
    if (rotated) {
      float co[8], si[8];
      load8<true>(a.cosines + row * half + frequency, co);
      load8<true>(a.sines + row * half + frequency, si);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        normalized[e] = g[e] * co[e] + (lower ? other[e] * si[e] : -other[e] * si[e]);
    }
    float dot = 0.0f, weighted[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      weighted[e] = normalized[e] * factor[e];
      dot += weighted[e] * x[e];
    }
#pragma unroll
    for (int offset = LANES / 2; offset > 0; offset >>= 1) {
      squares += __shfl_xor(squares, offset, 64);
      dot += __shfl_xor(dot, offset, 64);
    }
    const float inv = rsqrtf(squares / static_cast<float>(D) + a.epsilon);
    const float cubic = inv * inv * inv / static_cast<float>(D) * dot;
    if (!exists) continue;
    float dx[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      dx[e] = inv * weighted[e] - x[e] * cubic;
      weight_sum[e] += normalized[e] * x[e] * inv;
    }
    store8<true>(side.dx + unit * side.input_stride + c, dx);
  }
  if (!side.partial) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) sums[slot][c + e] = weight_sum[e];
  __syncthreads();
  if (threadIdx.x < D) {
    float total = 0.0f;
    for (int u = 0; u < UNITS; ++u) total += sums[u][threadIdx.x];
    side.partial[1LL * block * D + threadIdx.x] = total;
  }
}

// Any head width up to 256: one wave a workgroup, one channel of four a lane.
__global__ void __launch_bounds__(64)
norm_rope_backward_kernel(NormBackwardArgs a) {
  __shared__ float grads[256];
  const bool key_mode = static_cast<int>(blockIdx.x) >= a.queries.blocks;
  const NormSide side = key_mode ? a.keys : a.queries;
  const int block = blockIdx.x - (key_mode ? a.queries.blocks : 0);
  const int lane = threadIdx.x, d = a.d, half = a.rotary / 2;
  float weight_sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  const long long units = 1LL * a.length * side.heads;
  for (long long unit = block; unit < units; unit += side.blocks) {
    const long long row = unit / side.heads;
    const int head = static_cast<int>(unit % side.heads);
    float x[4], g[4];
    float sum_squares = 0.0f;
    __syncthreads();  // the unit before has read its partners
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = lane + 64 * j;
      x[j] = 0.0f;
      g[j] = 0.0f;
      if (c < d) {
        x[j] = bf16_bits_to_float(side.input[unit * side.input_stride + c]);
        if (!key_mode) {
          g[j] = a.grads.dq[row * a.grads.dq_row + head * d + c];
        } else {
          float key_sum = 0.0f, value_sum = 0.0f;
          for (int copy = 0; copy < a.group; ++copy) {
            const long long at = row * a.grads.dkv_row + 1LL * (head * a.group + copy) * d + c;
            key_sum += a.grads.dk[at];
            value_sum += a.grads.dv[at];
          }
          g[j] = key_sum;
          a.dv[unit * d + c] = value_sum;
        }
        grads[c] = g[j];
      }
      sum_squares += x[j] * x[j];
    }
    __syncthreads();
    sum_squares = wave_sum(sum_squares);
    const float inv = rsqrtf(sum_squares / static_cast<float>(d) + a.epsilon);
    float normalized[4], weighted[4];
    float dot = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = lane + 64 * j;
      normalized[j] = 0.0f;
      weighted[j] = 0.0f;
      if (c < d) {
        float ng = g[j];
        if (c < a.rotary) {
          const int frequency = c < half ? c : c - half;
          const float co = a.cosines[row * half + frequency];
          const float si = a.sines[row * half + frequency];
          const float partner = grads[c < half ? c + half : c - half];
          ng = g[j] * co + (c < half ? partner * si : -partner * si);
        }
        normalized[j] = ng;
        weighted[j] = ng * (1.0f + side.weight[c]);
        dot += weighted[j] * x[j];
      }
    }
    dot = wave_sum(dot);
    const float cubic = inv * inv * inv / static_cast<float>(d);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = lane + 64 * j;
      if (c < d) {
        side.dx[unit * side.input_stride + c] = inv * weighted[j] - x[j] * cubic * dot;
        weight_sum[j] += normalized[j] * x[j] * inv;
      }
    }
  }
  if (!side.partial) return;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (lane + 64 * j < d) side.partial[1LL * block * d + lane + 64 * j] = weight_sum[j];
}

// dw[c] += sum over the workgroups of partial[block, c], in a fixed order: row 0 of
// the grid the queries' weight, row 1 the keys'.  A workgroup takes eight
// channels, 128 threads each (one workgroup for all channels took 34 us over the
// same half megabyte).
__global__ void __launch_bounds__(1024)
norm_weight_kernel(NormBackwardArgs a) {
  __shared__ float sums[128][8], quarter[16][8];
  const NormSide side = blockIdx.y == 0 ? a.queries : a.keys;
  if (!side.partial) return;
  const int k = threadIdx.x % 8, g = threadIdx.x / 8, c = blockIdx.x * 8 + k;
  float sum = 0.0f;
  if (c < a.d)
    for (int block = g; block < side.blocks; block += 128) sum += side.partial[1LL * block * a.d + c];
  sums[g][k] = sum;
  __syncthreads();
  if (g < 16) {
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) total += sums[8 * g + i][k];
    quarter[g][k] = total;
  }
  __syncthreads();
  if (g != 0 || c >= a.d) return;
  float total = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) total += quarter[i][k];
  side.weight_grad[c] += total;
}

int grid_for(long long elements) {
  const long long blocks = (elements + 255) / 256;
  return static_cast<int>(blocks < 65536 ? blocks : 65536);
}

}  // namespace

int launch_pack_heads(hipStream_t stream, const float* q, const float* k, const float* v, int length,
                      int qh, int kh, int d, float* packed) {
  const long long elements = 3LL * length * qh * d;
  if (d % 4 == 0)
    pack_heads_kernel<4><<<grid_for(elements / 4), 256, 0, stream>>>(q, k, v, length, qh, kh, d, packed);
  else
    pack_heads_kernel<1><<<grid_for(elements), 256, 0, stream>>>(q, k, v, length, qh, kh, d, packed);
  return launch_status();
}

int launch_gate_backward(hipStream_t stream, const void* qg, const float* core, const float* dy,
                         int length, int qh, int d, bool round, float* dc, float* dqg) {
  const long long elements = 1LL * length * qh * d;
  gate_backward_kernel<<<grid_for(elements), 256, 0, stream>>>(static_cast<const uint16_t*>(qg), core, dy,
                                                              elements, d, round, dc, dqg);
  return launch_status();
}

int launch_gate_rows(hipStream_t stream, const void* qg, const void* core, const float* dy,
                     const float* maxima, const float* normalizers, int length, int qh, int d,
                     float scale2, uint16_t* dc, float* dqg, float* deltas, float* lse2) {
  const int rows = gate_group_rows(length, qh, d);
  const dim3 grid((length + rows - 1) / rows, qh);
  const auto* gates = static_cast<const uint16_t*>(qg);
  const auto* values = static_cast<const uint16_t*>(core);
  bool wide = true;
  for (const void* p : {qg, core, static_cast<const void*>(dy), static_cast<const void*>(dqg)})
    wide = wide && (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
  auto launch = [&](auto kernel) {
    kernel<<<grid, 256, 0, stream>>>(gates, values, dy, maxima, normalizers, length, rows, qh, scale2,
                                     dc, dqg, deltas, lse2);
  };
  if (d == 64)
    launch(wide ? gate_rows_kernel<64, true> : gate_rows_kernel<64, false>);
  else if (d == 128)
    launch(wide ? gate_rows_kernel<128, true> : gate_rows_kernel<128, false>);
  else
    return PLUTO_HIP_EUNSUPPORTED;
  return launch_status();
}

int launch_norm_rope_backward(hipStream_t stream, const void* qg, const void* k,
                              const float* q_norm, const float* k_norm,
                              const NormBackwardGrads& grads, const float* cosines,
                              const float* sines, int length, int qh, int kh, int d, int rotary,
                              float epsilon, float* dqg, float* dk, float* dv, float* dq_norm,
                              float* dk_norm, float* partial) {
  NormBackwardArgs a;
  a.queries = {static_cast<const uint16_t*>(qg), q_norm, dqg, nullptr, dq_norm, qh, 2 * d, 0};
  a.keys = {static_cast<const uint16_t*>(k), k_norm, dk, nullptr, dk_norm, kh, d, 0};
  a.grads = grads;
  a.cosines = cosines;
  a.sines = sines;
  a.dv = dv;
  a.length = length;
  a.d = d;
  a.rotary = rotary;
  a.group = qh / kh;
  a.epsilon = epsilon;
  bool rows = (d == 64 || d == 128 || d == 256) && rotary % 16 == 0 && grads.dq_row % 4 == 0 &&
              grads.dkv_row % 4 == 0;
  for (const void* p : {qg, k, static_cast<const void*>(dqg), static_cast<const void*>(dk),
                        static_cast<const void*>(dv), static_cast<const void*>(grads.dq),
                        static_cast<const void*>(grads.dk), static_cast<const void*>(grads.dv)})
    rows = rows && (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
  const long long per = rows ? 2048 / d : 1;  // units a workgroup works on at once
  auto blocks = [&](int heads, int most) {
    const long long wanted = (1LL * length * heads + per - 1) / per;
    return static_cast<int>(wanted < most ? wanted : most);
  };
  a.queries.blocks = blocks(qh, kNormQueryBlocks);
  a.keys.blocks = blocks(kh, kNormKeyBlocks);
  if (dq_norm) a.queries.partial = partial;
  if (dk_norm) a.keys.partial = partial + 1LL * kNormQueryBlocks * d;
  const int grid = a.queries.blocks + a.keys.blocks;
  if (!rows)
    norm_rope_backward_kernel<<<grid, 64, 0, stream>>>(a);
  else if (d == 64)
    norm_rope_rows_kernel<64><<<grid, 256, 0, stream>>>(a);
  else if (d == 128)
    norm_rope_rows_kernel<128><<<grid, 256, 0, stream>>>(a);
  else
    norm_rope_rows_kernel<256><<<grid, 256, 0, stream>>>(a);
  const int status = launch_status();
  if (status != 0 || (!dq_norm && !dk_norm)) return status;
  norm_weight_kernel<<<dim3((d + 7) / 8, 2), 1024, 0, stream>>>(a);
  return launch_status();
}

}  // namespace pluto_hip
