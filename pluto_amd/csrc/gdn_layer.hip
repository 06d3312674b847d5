// Layer-level pieces of the gated delta-net around the recurrence: causal
// depthwise convolution + SiLU, decay/beta gates, and the gated RMSNorm output.
// All are bandwidth-trivial elementwise kernels; every bf16 rounding point of
// the reference is kept (src/llm/layers/sequence_delta_net.cc:31-51,88-96,
// 104-121 and src/llm/layers/util/cached_attention_ops.cc:180-203,253-272).
#include "gdn.h"
#include "gdn_activation.h"
#include "mfma_tile.h"

namespace pluto_hip {
namespace {

__device__ inline float maybe_round(float x, bool round) {
  return round ? round_to_bf16(x) : x;
}

__global__ void __launch_bounds__(256)
conv_sequence_kernel(const void* input, int in_dtype, const float* __restrict__ weight,
                     int length, int channels, int kernel, bool round, void* post,
                     int post_dtype, long long total) {
  const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  const int c = static_cast<int>(i % channels);
  const long long row = i / channels;          // sequence * length + t
  const int t = static_cast<int>(row % length);
  float sum = 0.0f;
  for (int tap = 0; tap < kernel; ++tap) {
    const int source = t + tap - kernel + 1;
    if (source >= 0)
      sum += load_element(input, (row - t + source) * channels + c, in_dtype) *
             weight[static_cast<long long>(c) * kernel + tap];
  }
  sum = maybe_round(sum, round);
  store_element(post, i, post_dtype, maybe_round(sum / (1.0f + expf(-sum)), round));
}

// Eight bf16 of a 16-byte piece as floats.
__device__ inline void unpack8(uint4 v, float* x) {
  const uint32_t words[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[2 * i] = __uint_as_float(words[i] << 16);
    x[2 * i + 1] = __uint_as_float(words[i] & 0xffff0000u);
  }
}

// The same convolution for four taps, bf16 in and out.  The kernel above loads
// two bytes a lane and every input four times, and divides twice per element:
// 522 us for 8191 x 10240, where the 336 MB in and out take 69 us at a copy's
// rate.  Here a thread owns eight channels (16 bytes) and walks TOKENS rows with
// the last three in registers, so a row is read 1 + 3 / TOKENS times.
template <int TOKENS>
__global__ void __launch_bounds__(256)
conv_rows_kernel(const uint16_t* __restrict__ input, const float* __restrict__ weight, int length,
                 int channels, int segments, uint16_t* __restrict__ post) {
  const int group = blockIdx.x * 256 + threadIdx.x;
  if (group * 8 >= channels) return;
  const int sequence = blockIdx.y / segments, t0 = blockIdx.y % segments * TOKENS;
  const long long at = (1LL * sequence * length + t0) * channels + 8 * group;
  const uint16_t* in = input + at;
  uint16_t* out = post + at;
  float w[8][4];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float4 v = *reinterpret_cast<const float4*>(weight + 4LL * (8 * group + e));
    w[e][0] = v.x; w[e][1] = v.y; w[e][2] = v.z; w[e][3] = v.w;
  }
  const uint4 zero = make_uint4(0, 0, 0, 0);
  float x[4][8];  // rows t - 3 .. t
#pragma unroll
  for (int j = 0; j < 3; ++j)
    unpack8(t0 + j >= 3 ? *reinterpret_cast<const uint4*>(in + (j - 3LL) * channels) : zero, x[j]);
  const int rows = min(TOKENS, length - t0);
#pragma unroll
  for (int base = 0; base < TOKENS; base += 4) {
    uint4 raw[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      raw[j] = *reinterpret_cast<const uint4*>(in + static_cast<long long>(min(base + j, rows - 1)) * channels);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      unpack8(raw[j], x[3]);
      uint32_t packed[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float taps[2][4];
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int tap = 0; tap < 4; ++tap) taps[k][tap] = x[tap][2 * i + k];
        packed[i] = convolved_pair(taps[0], w[2 * i], taps[1], w[2 * i + 1]);
      }
      if (base + j < rows)
        *reinterpret_cast<uint4*>(out + static_cast<long long>(base + j) * channels) =
            make_uint4(packed[0], packed[1], packed[2], packed[3]);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[0][e] = x[1][e];
        x[1][e] = x[2][e];
        x[2][e] = x[3][e];
      }
    }
  }
}

__global__ void __launch_bounds__(128)
conv_step_kernel(const void* __restrict__ input, int in_dtype, const float* __restrict__ weight,
                 int channels, int kernel, bool round, float* __restrict__ state,
                 float* __restrict__ output) {
  const int c = blockIdx.x * 128 + threadIdx.x;
  if (c >= channels) return;
  // blockIdx.y: the sequence, each with its own shift registers and row
  const long long sequence = blockIdx.y;
  output += sequence * channels;
  float* taps = state + (sequence * channels + c) * kernel;
  const float* w = weight + static_cast<long long>(c) * kernel;
  float sum = 0.0f;
  // each channel is owned by one thread; shifting in ascending order never
  // overwrites a source still to be read
  for (int tap = 0; tap < kernel - 1; ++tap) {
    const float previous = taps[tap + 1];
    sum += previous * w[tap];
    taps[tap] = previous;
  }
  const float current = maybe_round(load_element(input, sequence * channels + c, in_dtype), round);
  taps[kernel - 1] = current;
  sum = maybe_round(sum + current * w[kernel - 1], round);
  output[c] = maybe_round(sum / (1.0f + expf(-sum)), round);
}

// One channel of four taps, its registers in one access each way: the same arithmetic.
__device__ inline float conv_step4(float4 taps, float4 w, float input, bool round, float* state) {
  const float current = maybe_round(input, round);
  *reinterpret_cast<float4*>(state) = make_float4(taps.y, taps.z, taps.w, current);
  float sum = 0.0f;
  sum += taps.y * w.x;
  sum += taps.z * w.y;
  sum += taps.w * w.z;
  sum = maybe_round(sum + current * w.w, round);
  return maybe_round(sum / (1.0f + expf(-sum)), round);
}
__global__ void __launch_bounds__(256)
conv_step4_kernel(const void* input, int in_dtype, const float* weight, int channels, bool round, float* state,
                  float* output) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= channels) return;
  const size_t index = static_cast<size_t>(blockIdx.y) * channels + c;
  output[index] = conv_step4(*reinterpret_cast<const float4*>(state + 4 * index),
                             *reinterpret_cast<const float4*>(weight + 4 * static_cast<size_t>(c)),
                             load_element(input, index, in_dtype), round, state + 4 * index);
}

__global__ void __launch_bounds__(256)
gates_kernel(const void* a, const void* b, int in_dtype, const float* __restrict__ a_log,
             const float* __restrict__ dt_bias, long long rows, int heads, bool round,
             float* __restrict__ log_decay, float* __restrict__ beta) {
  const long long i = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= rows * heads) return;
  const int head = static_cast<int>(i % heads);
  log_decay[i] = log_decay_of(load_element(a, i, in_dtype) + dt_bias[head], a_log[head]);
  beta[i] = maybe_round(beta_of(load_element(b, i, in_dtype)), round);
}

// One wave per (token, head) row of value_dim <= 256 channels.
__global__ void __launch_bounds__(256)
output_kernel(const void* core, int core_dtype, const void* z, int z_dtype,
              const float* __restrict__ norm, long long rows, int value_dim, float epsilon,
              bool round, void* out, int out_dtype) {
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const long long row = static_cast<long long>(blockIdx.x) * 4 + wave;
  if (row >= rows) return;
  float x[4];
  float square = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = lane + 64 * i;
    x[i] = c < value_dim ? load_element(core, row * value_dim + c, core_dtype) : 0.0f;
    square += x[i] * x[i];
  }
  square = wave_sum(square);
  const float inverse = rsqrtf(square / static_cast<float>(value_dim) + epsilon);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = lane + 64 * i;
    if (c >= value_dim) continue;
    const float normalized = maybe_round(x[i] * inverse, round);
    const float affine = maybe_round(normalized * norm[c], round);
    const float gate = load_element(z, row * value_dim + c, z_dtype);
    const float value = affine * (gate / (1.0f + expf(-gate)));
    // the sequence layer stores bf16; the single-token step keeps fp32 and
    // rounds only when asked to (cached_attention_ops.cc:270-271)
    store_element(out, row * value_dim + c, out_dtype,
                  out_dtype == PLUTO_HIP_BF16 ? value : maybe_round(value, round));
  }
}

// The same for rows of 128 bf16 values, in and out rounded.  The kernel above
// moves two bytes a lane and keeps one row a wave in flight (164 us for 8191
// tokens of 48 heads); here sixteen lanes own a row, eight channels each, and a
// thread requests its piece of four rows before it uses the first.
constexpr int kOutputRows = 4;
__global__ void __launch_bounds__(256)
output_rows128_kernel(const uint16_t* __restrict__ core, const uint16_t* __restrict__ z,
                      const float* __restrict__ norm, long long rows, float epsilon,
                      uint16_t* __restrict__ out) {
  const int piece = threadIdx.x % 16;
  const long long first = static_cast<long long>(blockIdx.x) * (16 * kOutputRows) + threadIdx.x / 16;
  float weight[8];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float4 v = *reinterpret_cast<const float4*>(norm + 8 * piece + 4 * e);
    weight[4 * e] = v.x; weight[4 * e + 1] = v.y; weight[4 * e + 2] = v.z; weight[4 * e + 3] = v.w;
  }
  uint4 core_raw[kOutputRows], gate_raw[kOutputRows];
#pragma unroll
  for (int r = 0; r < kOutputRows; ++r) {
    const long long row = min(first + 16 * r, rows - 1);
    core_raw[r] = *reinterpret_cast<const uint4*>(core + row * 128 + 8 * piece);
    gate_raw[r] = *reinterpret_cast<const uint4*>(z + row * 128 + 8 * piece);
  }
#pragma unroll
  for (int r = 0; r < kOutputRows; ++r) {
    float x[8], gate[8];
    unpack8(core_raw[r], x);
    unpack8(gate_raw[r], gate);
    float square = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) square += x[e] * x[e];
#pragma unroll
    for (int offset = 8; offset > 0; offset >>= 1) square += __shfl_xor(square, offset, 64);
    const float inverse = rsqrtf(square / 128.0f + epsilon);
    uint32_t packed[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t normalized = pack_bf16(x[2 * i] * inverse, x[2 * i + 1] * inverse);
      const uint32_t affine = pack_bf16(__uint_as_float(normalized << 16) * weight[2 * i],
                                        __uint_as_float(normalized & 0xffff0000u) * weight[2 * i + 1]);
      packed[i] = pack_bf16(__uint_as_float(affine << 16) * silu(gate[2 * i]),
                            __uint_as_float(affine & 0xffff0000u) * silu(gate[2 * i + 1]));
    }
    if (first + 16 * r < rows)
      *reinterpret_cast<uint4*>(out + (first + 16 * r) * 128 + 8 * piece) =
          make_uint4(packed[0], packed[1], packed[2], packed[3]);
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// One token of the gated delta rule for one (sequence, value head) with the
// gates before it and RMSNorm x SiLU(z) after it: DeltaRecurrenceKernel and
// DeltaOutputKernel (cached_attention_ops.cc:205-272) with the gate
// arithmetic of sequence_delta_net.cc:88-96 in one launch.  The state is read
// and written exactly once, every load is issued before anything is waited
// for.
struct StepArgs {
  const float* convolved = nullptr;  // [batch, channels] q | k | v after conv + SiLU
  const void* qkv = nullptr;         // [batch, channels] before it, of z's type, and its shift
  float* conv_state = nullptr;       // registers [batch, channels, 4]: step128_kernel's CONV
  const float* conv_weight = nullptr;
  const void* z = nullptr;           // [batch, vh * vd], fp32 or bf16 (template argument)
  const void* a = nullptr;           // [batch, vh]
  const void* b = nullptr;
  const float* a_log = nullptr;
  const float* dt_bias = nullptr;
  const float* norm = nullptr;
  float* state = nullptr;            // [batch, vh, kd, vd]
  void* out = nullptr;               // [batch, vh * vd], same type as z
  int batch = 0, kh = 0, vh = 0, kd = 0, vd = 0;
  float epsilon = 1e-6f;
  bool round = true;
};

// Threads per workgroup of step_kernel: thread (part, column) = (tid / 128,
// tid % 128) owns rows 16 part .. 16 part + 15 of its column.  With 64 rows a
// thread the kernel needed 272 registers, which left a compute unit four waves
// that loaded, computed and stored in turn (60 us for 32 x 48 heads); sixteen
// waves of 97 registers take 49 us.
constexpr int kStepThreads = 1024;
constexpr int kStepParts = kStepThreads / 128, kStepRows = 128 / kStepParts;

template <int IO>
__global__ void __launch_bounds__(kStepThreads)
step_kernel(StepArgs a) {
  __shared__ float ks[128], qs[128];
  __shared__ float partial[kStepParts][128];
  __shared__ float squares[2];
  const int bh = blockIdx.x, seq = bh / a.vh, head = bh % a.vh;
  const int key_head = head / (a.vh / a.kh);
  const int kd = a.kd, vd = a.vd;
  const int tid = threadIdx.x, column = tid % 128, part = tid / 128;
  const int channels = 2 * a.kh * kd + a.vh * vd;
  const float* token = a.convolved + static_cast<size_t>(seq) * channels;
  float* state = a.state + static_cast<size_t>(bh) * kd * vd;
  const bool active = column < vd;
  const int column_read = active ? column : vd - 1;
  // the state slice: rows beyond the key width read the last row and count as zero
  float s[kStepRows];
#pragma unroll
  for (int r = 0; r < kStepRows; ++r) {
    const int row = kStepRows * part + r;
    const float value = state[min(row, kd - 1) * vd + column_read];
    s[r] = (row < kd && active) ? value : 0.0f;
  }
  if (tid < 128) {
    const int d = min(tid, kd - 1);
    const float kv = token[(a.kh + key_head) * kd + d], qv = token[key_head * kd + d];
    ks[tid] = tid < kd ? kv : 0.0f;
    qs[tid] = tid < kd ? qv : 0.0f;
  }
  const float value = token[2 * a.kh * kd + head * vd + column_read];
  const float gate =
      load_element(a.z, (static_cast<long long>(seq) * a.vh + head) * vd + column_read, IO);
  const float weight = a.norm[column_read];
  const size_t scalar = static_cast<size_t>(seq) * a.vh + head;
  const float alpha = load_element(a.a, scalar, IO) + a.dt_bias[head];
  // stable softplus: no overflow for strongly positive time steps
  const float softplus = fmaxf(alpha, 0.0f) + log1pf(expf(-fabsf(alpha)));
  const float decay = __expf(-expf(a.a_log[head]) * softplus);
  const float beta = maybe_round(1.0f / (1.0f + expf(-load_element(a.b, scalar, IO))), a.round);
  __syncthreads();
  // the normalised key and the normalised, scaled query replace the raw ones
  // in LDS (1e-6 inside the root: cached_attention_ops.cc:224-228)
  float k_scaled = 0.0f, q_scaled = 0.0f;
  if (tid < 128) {
    float kk = 1e-6f, qq = 1e-6f;
    for (int d = 0; d < 128; ++d) {
      kk += ks[d] * ks[d];
      qq += qs[d] * qs[d];
    }
    k_scaled = ks[tid] * rsqrtf(kk);
    q_scaled = qs[tid] * (rsqrtf(qq) / sqrtf(static_cast<float>(kd)));
  }
  __syncthreads();
  if (tid < 128) {
    ks[tid] = k_scaled;
    qs[tid] = q_scaled;
  }
  __syncthreads();
  float prediction = 0.0f;
#pragma unroll
  for (int r = 0; r < kStepRows; ++r) {
    s[r] *= decay;
    prediction += s[r] * ks[kStepRows * part + r];
  }
  partial[part][column] = prediction;
  __syncthreads();
  float predicted = partial[0][column];
#pragma unroll
  for (int i = 1; i < kStepParts; ++i) predicted += partial[i][column];
  const float delta = (value - predicted) * beta;
  __syncthreads();
  float output = 0.0f;
#pragma unroll
  for (int r = 0; r < kStepRows; ++r) {
    s[r] += ks[kStepRows * part + r] * delta;
    output += s[r] * qs[kStepRows * part + r];
  }
#pragma unroll
  for (int r = 0; r < kStepRows; ++r) {
    const int row = kStepRows * part + r;
    if (row < kd && active) state[row * vd + column] = s[r];
  }
  partial[part][column] = output;
  __syncthreads();
  // RMSNorm over the head's columns, then the SiLU(z) gate
  float core = 0.0f;
  if (part == 0 && active) {
    core = partial[0][column];
#pragma unroll
    for (int i = 1; i < kStepParts; ++i) core += partial[i][column];
    core = maybe_round(core, a.round);
  }
  const float square = wave_sum(core * core);
  if (part == 0 && tid % 64 == 0) squares[tid / 64] = square;
  __syncthreads();
  if (part != 0 || !active) return;
  const float inverse = rsqrtf((squares[0] + squares[1]) / static_cast<float>(vd) + a.epsilon);
  const float normalized = maybe_round(core * inverse, a.round);
  const float affine = maybe_round(normalized * weight, a.round);
  const float result = affine * (gate / (1.0f + expf(-gate)));
  // a bf16 result is rounded once, by the store: the FP32 step followed by the
  // layer's cast (delta_net.cc:97-101) gives the same bits with or without the flag
  store_element(a.out, (static_cast<long long>(seq) * a.vh + head) * vd + column, IO,
                IO == PLUTO_HIP_BF16 ? result : maybe_round(result, a.round));
}

// The same for heads of 128 x 128: four waves a head, wave w columns 32 w .. + 31, its lane (r,
// c) = (lane / 8, lane % 8) rows r, r + 8, ... of columns 4 c .. + 3.  Sums over rows stay
// within a wave; the workgroup meets for the rows of k and q and for the mean square only.
// Workgroups are persistent, two a compute unit, and request a head's state before they work
// on the one before it.  Sequences of 16/48 heads, with workgroups of 1024 threads a head and
// eight barriers, whose vector instructions were 45 % of it, and so: 6 sequences 14.7 -> 10.7 us,
// 21 33.1 -> 22.1, 40 (255 MB) 56.4 -> 41.5.
// CONV: the shift registers too; a workgroup then walks all value heads of a key head, which
// share the channels of q and k (what one of them shifts, another one must have read).  28
// sequences, with the convolution's launch and without: 44.0 + 4.9 -> 30.6, 64 96.3 + 11.1 -> 73.8.
constexpr int kStepSlots = 512;
struct HeadLoads {
  float4 state[16];
  float4 v, z;
  float a, b, a_log, dt_bias, row;  // row: of k (threads below 128) or q
  float4 taps, taps_weight;         // CONV: of v (threads below 128)
  float current;
};
struct Head {
  int sequence, head;
};

__device__ inline float4 load_four(const void* base, size_t index, int dtype) {
  if (dtype != PLUTO_HIP_BF16) return *reinterpret_cast<const float4*>(static_cast<const float*>(base) + index);
  const uint2 v = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(base) + index);
  return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                     __uint_as_float(v.y & 0xffff0000u));
}

template <int IO, bool CONV>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2, 2)))
step128_kernel(StepArgs a) {
  __shared__ __attribute__((aligned(16))) float rows[2][2][128];  // k and q, element r of row block i at 16 r + i
  __shared__ __attribute__((aligned(16))) float values[2][128];  // CONV: v
  __shared__ float parts[2][4];
  const int tid = threadIdx.x, lane = tid % 64, r = lane / 8;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int column = 32 * wave + 4 * (lane % 8);
  const int group = a.vh / a.kh, channels = (2 * a.kh + a.vh) * 128;
  const int units = a.batch * (CONV ? a.kh : a.vh);
  const float4 weight = *reinterpret_cast<const float4*>(a.norm + column);
  // the heads of this workgroup in order
  auto head_of = [&](int unit, int member) {
    return CONV ? Head{unit / a.kh, unit % a.kh * group + member} : Head{unit / a.vh, unit % a.vh};
  };
  auto request = [&](HeadLoads& l, Head at) {
    const size_t head = static_cast<size_t>(at.sequence) * a.vh + at.head;
    const float* state = a.state + head * (128 * 128) + r * 128 + column;
#pragma unroll
    for (int i = 0; i < 16; ++i) l.state[i] = *reinterpret_cast<const float4*>(state + 8 * 128 * i);
    l.z = load_four(a.z, head * 128 + column, IO);
    l.a = load_element(a.a, head, IO), l.b = load_element(a.b, head, IO);
    l.a_log = a.a_log[at.head], l.dt_bias = a.dt_bias[at.head];
    if constexpr (CONV) {
      if (tid < 128) {
        const int channel = (2 * a.kh + at.head) * 128 + tid;
        const size_t index = static_cast<size_t>(at.sequence) * channels + channel;
        l.taps = *reinterpret_cast<const float4*>(a.conv_state + 4 * index);
        l.taps_weight = *reinterpret_cast<const float4*>(a.conv_weight + 4 * channel);
        l.current = load_element(a.qkv, index, IO);
      }
    } else {
      const float* token = a.convolved + static_cast<size_t>(at.sequence) * channels;
      l.row = token[(tid < 128 ? a.kh + at.head / group : at.head / group) * 128 + tid % 128];
      l.v = *reinterpret_cast<const float4*>(token + (2 * a.kh + at.head) * 128 + column);
    }
  };
  const int row_place = tid % 8 * 16 + tid % 128 / 8;
  float k_scale = 0.0f, q_scale = 0.0f, k[16], q[16];
  int parity = 0;
  // one head; `next` is requested before it is worked on
  auto process = [&](HeadLoads& l, HeadLoads& following, Head at, bool first, bool more, Head next) {
    if constexpr (CONV) {
      if (first) {
        const int channel = ((tid < 128 ? a.kh : 0) + at.head / group) * 128 + tid % 128;
        const size_t index = static_cast<size_t>(at.sequence) * channels + channel;
        rows[parity][tid / 128][row_place] =
            conv_step4(*reinterpret_cast<const float4*>(a.conv_state + 4 * index),
                       *reinterpret_cast<const float4*>(a.conv_weight + 4 * channel),
                       load_element(a.qkv, index, IO), a.round, a.conv_state + 4 * index);
      }
      if (tid < 128) {
        const size_t index = static_cast<size_t>(at.sequence) * channels + (2 * a.kh + at.head) * 128 + tid;
        values[parity][tid] = conv_step4(l.taps, l.taps_weight, l.current, a.round, a.conv_state + 4 * index);
      }
    } else {
      rows[parity][tid / 128][row_place] = l.row;
    }
    if (more) request(following, next);
    // LDS alone: the requests stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (!CONV || first) {
      // 1e-6 inside the roots: cached_attention_ops.cc:224-228
      const float k0 = rows[parity][0][lane], k1 = rows[parity][0][lane + 64];
      const float q0 = rows[parity][1][lane], q1 = rows[parity][1][lane + 64];
      k_scale = rsqrtf(wave_sum(k0 * k0 + k1 * k1) + 1e-6f);
      q_scale = rsqrtf(wave_sum(q0 * q0 + q1 * q1) + 1e-6f) / sqrtf(128.0f);
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        const float4 k4 = *reinterpret_cast<const float4*>(&rows[parity][0][16 * r + i]);
        const float4 q4 = *reinterpret_cast<const float4*>(&rows[parity][1][16 * r + i]);
        k[i] = k4.x * k_scale, k[i + 1] = k4.y * k_scale, k[i + 2] = k4.z * k_scale, k[i + 3] = k4.w * k_scale;
        q[i] = q4.x * q_scale, q[i + 1] = q4.y * q_scale, q[i + 2] = q4.z * q_scale, q[i + 3] = q4.w * q_scale;
      }
    }
    const float decay = __expf(log_decay_of(l.a + l.dt_bias, l.a_log));
    const float beta = maybe_round(beta_of(l.b), a.round);
    const float4 v = CONV ? *reinterpret_cast<const float4*>(&values[parity][column]) : l.v;
    // over the eight row lanes of a column
    auto across_rows = [&](float4 x) {
#pragma unroll
      for (int offset = 8; offset < 64; offset *= 2) {
        x.x += __shfl_xor(x.x, offset, 64), x.y += __shfl_xor(x.y, offset, 64);
        x.z += __shfl_xor(x.z, offset, 64), x.w += __shfl_xor(x.w, offset, 64);
      }
      return x;
    };
    float4 predicted = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float4& s = l.state[i];
      s.x *= decay, s.y *= decay, s.z *= decay, s.w *= decay;
      predicted.x += s.x * k[i], predicted.y += s.y * k[i], predicted.z += s.z * k[i], predicted.w += s.w * k[i];
    }
    predicted = across_rows(predicted);
    const float4 delta = make_float4((v.x - predicted.x) * beta, (v.y - predicted.y) * beta,
                                     (v.z - predicted.z) * beta, (v.w - predicted.w) * beta);
    float4 core = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const size_t head = static_cast<size_t>(at.sequence) * a.vh + at.head;
    float* state = a.state + head * (128 * 128) + r * 128 + column;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float4& s = l.state[i];
      s.x += k[i] * delta.x, s.y += k[i] * delta.y, s.z += k[i] * delta.z, s.w += k[i] * delta.w;
      core.x += s.x * q[i], core.y += s.y * q[i], core.z += s.z * q[i], core.w += s.w * q[i];
      *reinterpret_cast<float4*>(state + 8 * 128 * i) = s;
    }
    core = across_rows(core);
    core = make_float4(maybe_round(core.x, a.round), maybe_round(core.y, a.round), maybe_round(core.z, a.round),
                       maybe_round(core.w, a.round));
    // RMSNorm over the head's columns, then the SiLU(z) gate
    float square = (core.x * core.x + core.y * core.y) + (core.z * core.z + core.w * core.w);
#pragma unroll
    for (int offset = 1; offset < 8; offset *= 2) square += __shfl_xor(square, offset, 64);
    if (lane == 0) parts[parity][wave] = square;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (r == 0) {
      const float total = (parts[parity][0] + parts[parity][1]) + (parts[parity][2] + parts[parity][3]);
      const float inverse = rsqrtf(total / 128.0f + a.epsilon);
      auto finish = [&](float x, float w, float gate) {
        const float affine = maybe_round(maybe_round(x * inverse, a.round) * w, a.round);
        const float result = affine * (gate / (1.0f + expf(-gate)));
        // a bf16 result is rounded once, by the store, as in step_kernel
        return IO == PLUTO_HIP_BF16 ? result : maybe_round(result, a.round);
      };
      const float4 out = make_float4(finish(core.x, weight.x, l.z.x), finish(core.y, weight.y, l.z.y),
                                     finish(core.z, weight.z, l.z.z), finish(core.w, weight.w, l.z.w));
      if (IO == PLUTO_HIP_BF16)
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + head * 128 + column) =
            make_uint2(pack_bf16(out.x, out.y), pack_bf16(out.z, out.w));
      else
        *reinterpret_cast<float4*>(static_cast<float*>(a.out) + head * 128 + column) = out;
    }
    parity ^= 1;
  };
  const int members = CONV ? group : 1;
  int unit = blockIdx.x, member = 0;
  HeadLoads loads[2];
  request(loads[0], head_of(unit, 0));
  while (true) {
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const Head at = head_of(unit, member);
      const bool first = member == 0;
      if (++member == members) member = 0, unit += gridDim.x;
      const bool more = unit < units;
      process(loads[side], loads[side ^ 1], at, first, more, more ? head_of(unit, member) : at);
      if (!more) return;
    }
  }
}

}  // namespace

bool gdn_step_fused_supported(int key_dim, int value_dim) {
  return key_dim <= 128 && value_dim <= 128;
}

// What step128_kernel reads and writes four at a time.
static bool step128_supported(const StepArgs& s, int io_dtype) {
  const uintptr_t io = io_dtype == PLUTO_HIP_BF16 ? 8 : 16;
  return s.kd == 128 && s.vd == 128 && aligned16(s.state) && aligned16(s.norm) && aligned16(s.convolved) &&
         reinterpret_cast<uintptr_t>(s.z) % io == 0 && reinterpret_cast<uintptr_t>(s.out) % io == 0;
}

int launch_gdn_step_fused(hipStream_t stream, const void* qkv, const void* z, const void* a, const void* b,
                          int io_dtype, const float* conv_weight, const float* a_log, const float* dt_bias,
                          const float* norm, int batch, int key_heads, int value_heads, int key_dim, int value_dim,
                          int taps, float epsilon, bool round, float* conv_state, float* state, void* out,
                          float* convolved) {
  StepArgs s;
  s.convolved = convolved;
  s.qkv = qkv;
  s.conv_state = conv_state;
  s.conv_weight = conv_weight;
  s.z = z;
  s.a = a;
  s.b = b;
  s.a_log = a_log;
  s.dt_bias = dt_bias;
  s.norm = norm;
  s.state = state;
  s.out = out;
  s.batch = batch;
  s.kh = key_heads;
  s.vh = value_heads;
  s.kd = key_dim;
  s.vd = value_dim;
  s.epsilon = epsilon;
  s.round = round;
  const bool wide = step128_supported(s, io_dtype), bf16 = io_dtype == PLUTO_HIP_BF16;
  // The convolution's launch is saved where walking all heads of a key head makes no
  // workgroup's list longer.
  auto turns = [](long long units) { return (units + kStepSlots - 1) / kStepSlots; };
  const long long heads = 1LL * batch * value_heads, key_units = 1LL * batch * key_heads;
  if (wide && taps == 4 && aligned16(conv_state) && aligned16(conv_weight) &&
      turns(key_units) * (value_heads / key_heads) <= turns(heads)) {
    const unsigned blocks = static_cast<unsigned>(key_units < kStepSlots ? key_units : kStepSlots);
    if (bf16)
      step128_kernel<PLUTO_HIP_BF16, true><<<blocks, 256, 0, stream>>>(s);
    else
      step128_kernel<PLUTO_HIP_F32, true><<<blocks, 256, 0, stream>>>(s);
    return launch_status();
  }
  const int channels = 2 * key_heads * key_dim + value_heads * value_dim;
  const int status =
      launch_gdn_conv_step(stream, qkv, io_dtype, conv_weight, batch, channels, taps, round, conv_state, convolved);
  if (status != 0) return status;
  const unsigned blocks = static_cast<unsigned>(heads < kStepSlots ? heads : kStepSlots);
  if (wide && bf16)
    step128_kernel<PLUTO_HIP_BF16, false><<<blocks, 256, 0, stream>>>(s);
  else if (wide)
    step128_kernel<PLUTO_HIP_F32, false><<<blocks, 256, 0, stream>>>(s);
  else if (bf16)
    step_kernel<PLUTO_HIP_BF16><<<batch * value_heads, kStepThreads, 0, stream>>>(s);
  else
    step_kernel<PLUTO_HIP_F32><<<batch * value_heads, kStepThreads, 0, stream>>>(s);
  return launch_status();
}

int launch_gdn_conv_sequence(hipStream_t stream, const void* input, int in_dtype,
                             const float* weight, int batch, int length, int channels,
                             int kernel, bool round, void* post, int post_dtype) {
  if (kernel == 4 && round && in_dtype == PLUTO_HIP_BF16 && post_dtype == PLUTO_HIP_BF16 &&
      channels % 8 == 0 && aligned16(input) && aligned16(weight) && aligned16(post)) {
    const unsigned groups = (channels / 8 + 255) / 256;
    // sixteen rows a thread where that still leaves a few waves a SIMD, else four
    const bool many = 1LL * batch * length * channels >= 1LL << 23;
    const int tokens = many ? 16 : 4, segments = (length + tokens - 1) / tokens;
    if (1LL * batch * segments <= 65535) {
      const dim3 grid(groups, static_cast<unsigned>(batch) * segments);
      auto* in = static_cast<const uint16_t*>(input);
      auto* out = static_cast<uint16_t*>(post);
      if (many)
        conv_rows_kernel<16><<<grid, 256, 0, stream>>>(in, weight, length, channels, segments, out);
      else
        conv_rows_kernel<4><<<grid, 256, 0, stream>>>(in, weight, length, channels, segments, out);
      return launch_status();
    }
  }
  const long long total = static_cast<long long>(batch) * length * channels;
  conv_sequence_kernel<<<static_cast<unsigned>((total + 255) / 256), 256, 0, stream>>>(
      input, in_dtype, weight, length, channels, kernel, round, post, post_dtype, total);
  return launch_status();
}

int launch_gdn_conv_step(hipStream_t stream, const void* input, int in_dtype, const float* weight,
                         int batch, int channels, int kernel, bool round, float* state,
                         float* output) {
  if (kernel == 4 && aligned16(weight) && aligned16(state))
    conv_step4_kernel<<<dim3((channels + 255) / 256, batch), 256, 0, stream>>>(input, in_dtype, weight, channels, round,
                                                                               state, output);
  else
    conv_step_kernel<<<dim3((channels + 127) / 128, batch), 128, 0, stream>>>(
        input, in_dtype, weight, channels, kernel, round, state, output);
  return launch_status();
}

int launch_gdn_gates(hipStream_t stream, const void* a, const void* b, int in_dtype,
                     const float* a_log, const float* dt_bias, long long rows, int heads,
                     bool round, float* log_decay, float* beta) {
  const long long total = rows * heads;
  gates_kernel<<<static_cast<unsigned>((total + 255) / 256), 256, 0, stream>>>(
      a, b, in_dtype, a_log, dt_bias, rows, heads, round, log_decay, beta);
  return launch_status();
}

int launch_gdn_output(hipStream_t stream, const void* core, int core_dtype, const void* z,
                      int z_dtype, const float* norm, long long rows, int value_dim,
                      float epsilon, bool round, void* out, int out_dtype) {
  if (value_dim == 128 && round && core_dtype == PLUTO_HIP_BF16 && z_dtype == PLUTO_HIP_BF16 &&
      out_dtype == PLUTO_HIP_BF16 && aligned16(core) && aligned16(z) && aligned16(norm) &&
      aligned16(out)) {
    const long long per = 16 * kOutputRows;
    output_rows128_kernel<<<static_cast<unsigned>((rows + per - 1) / per), 256, 0, stream>>>(
        static_cast<const uint16_t*>(core), static_cast<const uint16_t*>(z), norm, rows, epsilon,
        static_cast<uint16_t*>(out));
    return launch_status();
  }
  output_kernel<<<static_cast<unsigned>((rows + 3) / 4), 256, 0, stream>>>(
      core, core_dtype, z, z_dtype, norm, rows, value_dim, epsilon, round, out, out_dtype);
  return launch_status();
}

}  // namespace pluto_hip
