// Backward of the gated delta-net layer over a sequence
// (SequenceDeltaNetLayer::bwd_impl, src/llm/layers/sequence_delta_net.cc:
// 482-561) in FP32, token by token as the reference does it: the forward pass
// is repeated with every state S_t kept, then the recurrence is differentiated
// in reverse.  Kernels and the reference kernels they follow:
//   conv_train_kernel            ConvForward            (:31-51), keeps `pre`
//   recurrence_states_kernel     RecurrenceForward      (:55-102)
//   output_backward_kernel       OutputBackward         (:125-155)
//   recurrence_backward_kernel   RecurrenceBackward     (:171-253)
//   gather_qk_kernel             GatherQkGradient       (:255-276)
//   gather_scalar_kernel         GatherScalarGradient   (:278-305); finish_parameters_kernel
//                                with the chunked kernels
//   conv_silu_backward_kernel    ConvSiluBackward       (:307-318)
//   conv_input_backward_kernel   ConvInputBackward      (:320-336)
//   conv_weight_*_kernel         ConvWeightBackward     (:338-355), two levels
//   sum_rows_*_kernel            SumNormGradient        (:157-166), two levels
//
// The two recurrence kernels share one layout: a workgroup owns the
// [key_dim, 32] slice of one head's state (as the reference's programs do),
// thread (kg, c) = (tid / 32, tid % 32) holds rows 16 kg .. 16 kg + 15 of
// column c in registers.  Sums over rows go through LDS (8 partials a column),
// sums over columns through LDS as well (one padded row of products per state
// row, added up by one thread per row).  What a token reads from global memory
// is requested one token ahead.
#include "gdn.h"
#include "gdn_activation.h"
#include "mfma_tile.h"

namespace pluto_hip {
namespace {

constexpr int kRows = 16;        // state rows per thread
constexpr int kGroups = 8;       // row groups per workgroup
constexpr int kColumns = 32;     // state columns per workgroup
constexpr int kMaxKey = kRows * kGroups;  // 128
constexpr int kConvSlices = 64;  // token slices of the convolution weight gradient

__device__ inline float round_if(float x, bool round) { return round ? round_to_bf16(x) : x; }

// VEC consecutive elements of a row as one access (VEC is 1 or 4).
template <int VEC>
struct Pack {
  float e[VEC];
};
template <int VEC>
__device__ inline Pack<VEC> load_floats(const float* p) {
  Pack<VEC> r;
  if constexpr (VEC == 4) {
    const float4 v = *reinterpret_cast<const float4*>(p);
    r.e[0] = v.x; r.e[1] = v.y; r.e[2] = v.z; r.e[3] = v.w;
  } else {
    r.e[0] = p[0];
  }
  return r;
}
template <int VEC>
__device__ inline void store_floats(float* p, const Pack<VEC>& v) {
  if constexpr (VEC == 4)
    *reinterpret_cast<float4*>(p) = make_float4(v.e[0], v.e[1], v.e[2], v.e[3]);
  else
    p[0] = v.e[0];
}
template <int VEC>
__device__ inline Pack<VEC> load_bf16s(const uint16_t* p) {
  Pack<VEC> r;
  if constexpr (VEC == 4) {
    const uint2 bits = *reinterpret_cast<const uint2*>(p);
    r.e[0] = __uint_as_float(bits.x << 16);
    r.e[1] = __uint_as_float(bits.x & 0xffff0000u);
    r.e[2] = __uint_as_float(bits.y << 16);
    r.e[3] = __uint_as_float(bits.y & 0xffff0000u);
  } else {
    r.e[0] = bf16_bits_to_float(p[0]);
  }
  return r;
}

// One thread per VEC channels of a token (channels % VEC == 0).
// POST: float, or uint16_t for bf16 (then `round`).
template <int VEC, class POST>
__global__ void __launch_bounds__(256)
conv_train_kernel(const uint16_t* input, const float* __restrict__ weight, int length,
                  int channels, int kernel, bool round, float* pre, POST* post) {
  const int groups = channels / VEC;
  const long long i = blockIdx.x * 256LL + threadIdx.x;
  if (i >= 1LL * length * groups) return;
  const int c = static_cast<int>(i % groups) * VEC, t = static_cast<int>(i / groups);
  Pack<VEC> sum;
#pragma unroll
  for (int e = 0; e < VEC; ++e) sum.e[e] = 0.0f;
  for (int tap = 0; tap < kernel; ++tap) {
    const int source = t + tap - kernel + 1;
    if (source < 0) continue;
    const Pack<VEC> x = load_bf16s<VEC>(input + 1LL * source * channels + c);
#pragma unroll
    for (int e = 0; e < VEC; ++e) sum.e[e] += x.e[e] * weight[1LL * (c + e) * kernel + tap];
  }
  Pack<VEC> activated;
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    sum.e[e] = round_if(sum.e[e], round);
    activated.e[e] = round_if(sum.e[e] / (1.0f + expf(-sum.e[e])), round);
  }
  store_floats<VEC>(pre + 1LL * t * channels + c, sum);
  if constexpr (sizeof(POST) == 4) {
    store_floats<VEC>(post + 1LL * t * channels + c, activated);
  } else {
    static_assert(VEC == 1);
    post[1LL * t * channels + c] = float_to_bf16_bits(activated.e[0]);
  }
}

// ---- four taps ---------------------------------------------------------------
// The convolution and its backward with the taps' rows in registers: a thread owns
// VEC channels and walks a run of tokens.  ALIGNED: rows and weights may be
// accessed VEC elements at once.
template <int VEC, bool ALIGNED>
__device__ inline void read_bf16(const uint16_t* p, float (&x)[VEC]) {
  static_assert(VEC == 2 || VEC == 4);
  if constexpr (ALIGNED) {
    uint32_t words[VEC / 2];
    if constexpr (VEC == 4) {
      const uint2 v = *reinterpret_cast<const uint2*>(p);
      words[0] = v.x, words[1] = v.y;
    } else {
      words[0] = *reinterpret_cast<const uint32_t*>(p);
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e)
      x[e] = __uint_as_float(e % 2 ? words[e / 2] & 0xffff0000u : words[e / 2] << 16);
  } else {
#pragma unroll
    for (int e = 0; e < VEC; ++e) x[e] = bf16_bits_to_float(p[e]);
  }
}
template <int VEC, bool ALIGNED>
__device__ inline void read_taps(const float* weight, int c, float (&w)[VEC][4]) {
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    const float* p = weight + 4LL * (c + e);
    if constexpr (ALIGNED) {
      const float4 v = *reinterpret_cast<const float4*>(p);
      w[e][0] = v.x, w[e][1] = v.y, w[e][2] = v.z, w[e][3] = v.w;
    } else {
#pragma unroll
      for (int tap = 0; tap < 4; ++tap) w[e][tap] = p[tap];
    }
  }
}

// post = SiLU(conv(input)) as FP32, both rounded to bf16 on request, or as bf16.  (One
// channel and one token a thread, four loads each, took 108 us at 2048 tokens of 10240
// channels.  Now 28.4 us as FP32, 126 MB in and out, 18.7 as bf16, 84 MB.)
constexpr int kConvRun = 8;
template <bool ALIGNED, class POST>
__global__ void __launch_bounds__(256)
conv_train4_kernel(const uint16_t* __restrict__ input, const float* __restrict__ weight, int length,
                   int channels, bool round, POST* __restrict__ post) {
  constexpr int VEC = 4;
  const int c = (blockIdx.x * 256 + threadIdx.x) * VEC, t0 = blockIdx.y * kConvRun;
  if (c >= channels) return;
  float w[VEC][4], x[4][VEC];
  read_taps<VEC, ALIGNED>(weight, c, w);
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    read_bf16<VEC, ALIGNED>(input + 1LL * max(t0 - 3 + j, 0) * channels + c, x[j]);
#pragma unroll
    for (int e = 0; e < VEC; ++e) x[j][e] = t0 - 3 + j >= 0 ? x[j][e] : 0.0f;
  }
  float rows[kConvRun][VEC];
#pragma unroll
  for (int r = 0; r < kConvRun; ++r)
    read_bf16<VEC, ALIGNED>(input + 1LL * min(t0 + r, length - 1) * channels + c, rows[r]);
#pragma unroll
  for (int r = 0; r < kConvRun; ++r) {
    float out[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      x[3][e] = rows[r][e];
      float sum = 0.0f;
#pragma unroll
      for (int tap = 0; tap < 4; ++tap) sum += x[tap][e] * w[e][tap];
      if constexpr (sizeof(POST) == 4) {
        sum = round_if(sum, round);
        out[e] = round_if(sum / (1.0f + expf(-sum)), round);
      } else {
        out[e] = silu_of_bf16(round_to_bf16(sum));
      }
      x[0][e] = x[1][e], x[1][e] = x[2][e], x[2][e] = x[3][e];
    }
    if (t0 + r >= length) continue;
    POST* to = post + 1LL * (t0 + r) * channels + c;
    if constexpr (sizeof(POST) == 4)
      *reinterpret_cast<float4*>(to) = make_float4(out[0], out[1], out[2], out[3]);
    else
      *reinterpret_cast<uint2*>(to) = make_uint2(pack_bf16(out[0], out[1]), pack_bf16(out[2], out[3]));
  }
}

// Everything behind the gradient of `post` in one pass: back through SiLU (with
// the convolution repeated instead of stored), the input's gradient, and this run's
// share of the weights' gradient.  The q and k channels' gradient is the sum of
// their value heads' partials, in ascending order.  (As five kernels that stored
// the convolution, the gathered and the inner gradient: 258 us at 2048 tokens of
// 10240 channels; what it cannot do without is 290 MB.)
struct ConvBackwardArgs {
  const uint16_t* input = nullptr;
  const float* weight = nullptr;
  const float* qk_partials = nullptr;  // [T, vh, tiles, 2, kd]
  const float* dpost = nullptr;        // [T, channels]: the value channels
  float* dx = nullptr;
  float* partial = nullptr;  // optional [runs, channels, 4]
  int length = 0, channels = 0, kh = 0, vh = 0, kd = 0, tiles = 0, run = 0;
  bool round = true;
};
// PARTS: partials a token's gradient is the sum of, 0 for any number.  Bound by memory:
// what it waited for most was the sum of three partials inside the request for a token two
// ahead; each partial has registers of its own and is added when the token's turn comes,
// in the same order, four tokens later: 80 -> 54 us at 2048 tokens of 10240 channels, three
// value heads a key head (276 MB), 23 -> 11 us at 85 tokens.
template <bool ALIGNED, int PARTS>
__device__ inline void conv_backward4_channels(const ConvBackwardArgs& a, int c) {
  constexpr int VEC = 2, kAhead = 4, kHeld = PARTS > 0 ? PARTS : 1;
  const int t0 = blockIdx.y * a.run, t1 = min(t0 + a.run, a.length);
  const int keys = a.kh * a.kd, group = a.vh / a.kh;
  const bool gathered = c < 2 * keys;
  // where a token's partials of these channels start, and how they continue
  const int key_head = c % keys / a.kd, channel = c % a.kd;
  const float* gather = a.qk_partials + (1LL * key_head * group * a.tiles * 2 + (c >= keys ? 1 : 0)) * a.kd + channel;
  const long long gather_token = 2LL * a.vh * a.tiles * a.kd;
  float w[VEC][4];
  read_taps<VEC, ALIGNED>(a.weight, c, w);
  float x[4][VEC], d[4][VEC], dw[VEC][4];  // rows t - 3 .. t of the input, of the inner gradient
#pragma unroll
  for (int e = 0; e < VEC; ++e)
#pragma unroll
    for (int j = 0; j < 4; ++j) d[j][e] = dw[e][j] = 0.0f;
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    read_bf16<VEC, ALIGNED>(a.input + 1LL * max(t0 - 3 + j, 0) * a.channels + c, x[j]);
#pragma unroll
    for (int e = 0; e < VEC; ++e) x[j][e] = t0 - 3 + j >= 0 ? x[j][e] : 0.0f;
  }
  // a token's gradient and input, requested kAhead tokens ahead
  auto fetch = [&](int t, float (&input)[VEC], float2 (&upstream)[kHeld]) {
    const int row = min(t, a.length - 1);
    read_bf16<VEC, ALIGNED>(a.input + 1LL * row * a.channels + c, input);
    const float* from = gathered ? gather + row * gather_token : a.dpost + 1LL * row * a.channels + c;
#pragma unroll
    for (int part = 0; part < kHeld; ++part)
      upstream[part] = *reinterpret_cast<const float2*>(from + 2LL * part * a.kd);
    if (PARTS == 0) {
      for (int part = 1; part < group * a.tiles; ++part) {
        const float2 v = *reinterpret_cast<const float2*>(from + 2LL * part * a.kd);
        upstream[0].x += v.x, upstream[0].y += v.y;
      }
    }
  };
  float next_x[kAhead][VEC];
  float2 next_g[kAhead][kHeld];
#pragma unroll
  for (int i = 0; i < kAhead; ++i) fetch(t0 + i, next_x[i], next_g[i]);
  // rows t1 .. t1 + 2 only complete the gradients of the rows before them
  auto token = [&](int t, float (&input)[VEC], float2 (&gradient)[kHeld]) {
    float upstream[VEC] = {gradient[0].x, gradient[0].y};
#pragma unroll
    for (int part = 1; part < kHeld; ++part) upstream[0] += gradient[part].x, upstream[1] += gradient[part].y;
#pragma unroll
    for (int e = 0; e < VEC; ++e) x[3][e] = input[e];
    fetch(t + kAhead, input, gradient);
    float out[VEC];
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      float pre = 0.0f;
#pragma unroll
      for (int tap = 0; tap < 4; ++tap) pre += x[tap][e] * w[e][tap];
      pre = round_if(pre, a.round);
      const float sigmoid = 1.0f / (1.0f + expf(-pre));
      d[3][e] = t < a.length ? upstream[e] * sigmoid * (1.0f + pre * (1.0f - sigmoid)) : 0.0f;
      out[e] = 0.0f;
#pragma unroll
      for (int tap = 0; tap < 4; ++tap) {
        out[e] += d[3 - tap][e] * w[e][tap];
        if (t < t1) dw[e][tap] += d[3][e] * x[tap][e];
      }
    }
    if (t - 3 >= t0) {
      float* p = a.dx + 1LL * (t - 3) * a.channels + c;
      if constexpr (ALIGNED) {
        *reinterpret_cast<float2*>(p) = make_float2(out[0], out[1]);
      } else {
        p[0] = out[0], p[1] = out[1];
      }
    }
#pragma unroll
    for (int e = 0; e < VEC; ++e)
#pragma unroll
      for (int j = 0; j < 3; ++j) x[j][e] = x[j + 1][e], d[j][e] = d[j + 1][e];
  };
  for (int t = t0; t < t1 + 3; t += kAhead) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (t + i >= t1 + 3) break;
      token(t + i, next_x[i], next_g[i]);
    }
  }
  if (!a.partial) return;
#pragma unroll
  for (int e = 0; e < VEC; ++e)
    *reinterpret_cast<float4*>(a.partial + (1LL * blockIdx.y * a.channels + c + e) * 4) =
        make_float4(dw[e][0], dw[e][1], dw[e][2], dw[e][3]);
}
template <bool ALIGNED>
__global__ void __launch_bounds__(256)
conv_backward4_kernel(ConvBackwardArgs a) {
  const int c = (blockIdx.x * 256 + threadIdx.x) * 2;
  if (c >= a.channels) return;
  const int parts = c < 2 * a.kh * a.kd ? a.vh / a.kh * a.tiles : 1;
  if (parts == 1)
    conv_backward4_channels<ALIGNED, 1>(a, c);
  else if (parts == 2)
    conv_backward4_channels<ALIGNED, 2>(a, c);
  else if (parts == 3)
    conv_backward4_channels<ALIGNED, 3>(a, c);
  else
    conv_backward4_channels<ALIGNED, 0>(a, c);
}

struct RecurrenceArgs {
  const float* post = nullptr;     // [T, channels]
  const uint16_t* a = nullptr;     // bf16 [T, vh]
  const uint16_t* b = nullptr;
  const float* a_log = nullptr;
  const float* dt_bias = nullptr;
  float* states = nullptr;         // [(T + 1), vh, kd, vd]
  float* core = nullptr;           // [T, vh, vd]
  const float* dcore = nullptr;    // [T, vh, vd]
  float* qk_partials = nullptr;    // [T, vh, tiles, 2, kd]
  float* scalar_partials = nullptr;  // [T, vh, tiles, 3]
  float* dpost = nullptr;          // [T, channels]; the value part is written here
  int length = 0, kh = 0, vh = 0, kd = 0, vd = 0;
  bool round = true;
};

struct TokenScalars {
  float alpha, softplus, rate, decay, sigmoid, beta;
};

// What a thread reads from global memory for one token.  It is requested one
// token ahead, so that the sequential chain never waits for these loads.
struct TokenInputs {
  float q[2], k[2];   // wave 0: raw q and k channels lane and lane + 64
  float a, b;         // the head's gate logits
  float v, dy;        // this thread's value column and (backward) its gradient
};

__device__ inline TokenInputs fetch_token(const RecurrenceArgs& a, int t, int head, int key_head,
                                          int column, bool column_ok, bool with_gradient) {
  TokenInputs in;
  const int channels = 2 * a.kh * a.kd + a.vh * a.vd;
  const int tid = threadIdx.x;
  in.q[0] = in.q[1] = in.k[0] = in.k[1] = 0.0f;
  if (tid < 64) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int d = tid + 64 * j;
      if (d < a.kd) {
        in.q[j] = a.post[1LL * t * channels + key_head * a.kd + d];
        in.k[j] = a.post[1LL * t * channels + (a.kh + key_head) * a.kd + d];
      }
    }
  }
  in.a = bf16_bits_to_float(a.a[1LL * t * a.vh + head]);
  in.b = bf16_bits_to_float(a.b[1LL * t * a.vh + head]);
  in.v = column_ok ? a.post[1LL * t * channels + 2 * a.kh * a.kd + head * a.vd + column] : 0.0f;
  in.dy = (with_gradient && column_ok) ? a.dcore[(1LL * t * a.vh + head) * a.vd + column] : 0.0f;
  return in;
}

__device__ inline TokenScalars token_scalars(const RecurrenceArgs& a, const TokenInputs& in,
                                             int head) {
  TokenScalars s;
  s.alpha = in.a + a.dt_bias[head];
  s.softplus = fmaxf(s.alpha, 0.0f) + logf(1.0f + expf(-fabsf(s.alpha)));
  s.rate = expf(a.a_log[head]);
  s.decay = expf(-s.rate * s.softplus);
  s.sigmoid = 1.0f / (1.0f + expf(-in.b));
  s.beta = round_if(s.sigmoid, a.round);
  return s;
}

// Raw q and k of the token into LDS together with 1/|q|, 1/|k| (1e-6 added to
// the sums of squares, sequence_delta_net.cc:84-85).
__device__ inline void publish_token_qk(const TokenInputs& in, float* raw_q, float* raw_k,
                                        float* inverses) {
  const int tid = threadIdx.x;
  if (tid < 64) {
    float qq = 0.0f, kk = 0.0f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      raw_q[tid + 64 * j] = in.q[j];
      raw_k[tid + 64 * j] = in.k[j];
      qq += in.q[j] * in.q[j];
      kk += in.k[j] * in.k[j];
    }
    qq = wave_sum(qq);
    kk = wave_sum(kk);
    if (tid == 0) {
      inverses[0] = rsqrtf(qq + 1e-6f);
      inverses[1] = rsqrtf(kk + 1e-6f);
    }
  }
}

// Sum over the kGroups row groups of a per-column partial.
__device__ inline float column_total(float partial, float (*scratch)[kColumns], int kg, int c) {
  scratch[kg][c] = partial;
  __syncthreads();
  float total = 0.0f;
#pragma unroll
  for (int g = 0; g < kGroups; ++g) total += scratch[g][c];
  __syncthreads();
  return total;
}

__global__ void __launch_bounds__(256)
recurrence_states_kernel(RecurrenceArgs a) {
  __shared__ float raw_q[kMaxKey], raw_k[kMaxKey], inverses[2];
  __shared__ float scratch[kGroups][kColumns];
  const int tiles = (a.vd + kColumns - 1) / kColumns;
  const int head = blockIdx.x / tiles, tile = blockIdx.x % tiles;
  const int key_head = head / (a.vh / a.kh);
  const int kg = threadIdx.x / kColumns, c = threadIdx.x % kColumns;
  const int column = tile * kColumns + c;
  const bool column_ok = column < a.vd;
  const int channels = 2 * a.kh * a.kd + a.vh * a.vd;
  const size_t stride = static_cast<size_t>(a.vh) * a.kd * a.vd;
  const float norm_scale = sqrtf(static_cast<float>(a.kd));
  float m[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    m[r] = 0.0f;
    const int row = kg * kRows + r;
    if (row < a.kd && column_ok) a.states[(static_cast<size_t>(head) * a.kd + row) * a.vd + column] = 0.0f;
  }
  TokenInputs next = fetch_token(a, 0, head, key_head, column, column_ok, false);
  for (int t = 0; t < a.length; ++t) {
    const TokenInputs in = next;
    if (t + 1 < a.length) next = fetch_token(a, t + 1, head, key_head, column, column_ok, false);
    publish_token_qk(in, raw_q, raw_k, inverses);
    __syncthreads();
    const TokenScalars s = token_scalars(a, in, head);
    const float iq = inverses[0], ik = inverses[1];
    float prediction = 0.0f;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      m[r] *= s.decay;
      prediction += m[r] * (raw_k[kg * kRows + r] * ik);
    }
    prediction = column_total(prediction, scratch, kg, c);
    const float delta = (in.v - prediction) * s.beta;
    float out = 0.0f;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int row = kg * kRows + r;
      m[r] += (raw_k[row] * ik) * delta;
      out += m[r] * (raw_q[row] * iq / norm_scale);
      if (row < a.kd && column_ok)
        a.states[(t + 1) * stride + (static_cast<size_t>(head) * a.kd + row) * a.vd + column] = m[r];
    }
    out = column_total(out, scratch, kg, c);
    if (kg == 0 && column_ok) a.core[(1LL * t * a.vh + head) * a.vd + column] = round_if(out, a.round);
  }
}

__global__ void __launch_bounds__(256)
recurrence_backward_kernel(RecurrenceArgs a) {
  __shared__ float raw_q[kMaxKey], raw_k[kMaxKey], inverses[2];
  __shared__ float scratch[kGroups][kColumns];
  __shared__ float dq_rows[kMaxKey], dk_rows[kMaxKey];
  __shared__ float block_sums[4][3];
  // per-element products whose sums over the 32 columns give dq and dk: one
  // padded row per state row, summed by one thread per row (a lane shuffle
  // tree per row costs a multiple of this)
  __shared__ float q_products[kMaxKey][kColumns + 1], k_products[kMaxKey][kColumns + 1];
  const int tiles = (a.vd + kColumns - 1) / kColumns;
  const int head = blockIdx.x / tiles, tile = blockIdx.x % tiles;
  const int key_head = head / (a.vh / a.kh);
  const int tid = threadIdx.x, wave = tid / 64;
  const int kg = tid / kColumns, c = tid % kColumns;
  const int column = tile * kColumns + c;
  const bool column_ok = column < a.vd;
  const int channels = 2 * a.kh * a.kd + a.vh * a.vd;
  const size_t stride = static_cast<size_t>(a.vh) * a.kd * a.vd;
  const float norm_scale = sqrtf(static_cast<float>(a.kd));
  float dm[kRows];
  // S_{t+1} of a token is S_t of the token processed just before it, and S_t is
  // requested one token ahead: no load of a state is waited for inside a token.
  float after[kRows], before[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    dm[r] = 0.0f;
    const int row = kg * kRows + r;
    const bool ok = row < a.kd && column_ok;
    const size_t at = (static_cast<size_t>(head) * a.kd + row) * a.vd + column;
    after[r] = ok ? a.states[a.length * stride + at] : 0.0f;
    before[r] = ok ? a.states[(a.length - 1) * stride + at] : 0.0f;
  }
  TokenInputs next = fetch_token(a, a.length - 1, head, key_head, column, column_ok, true);
  for (int t = a.length - 1; t >= 0; --t) {
    const TokenInputs in = next;
    if (t > 0) next = fetch_token(a, t - 1, head, key_head, column, column_ok, true);
    publish_token_qk(in, raw_q, raw_k, inverses);
    float ahead[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int row = kg * kRows + r;
      const bool ok = row < a.kd && column_ok && t > 0;
      ahead[r] = ok ? a.states[(t - 1) * stride + (static_cast<size_t>(head) * a.kd + row) * a.vd + column]
                    : 0.0f;
    }
    __syncthreads();
    const TokenScalars s = token_scalars(a, in, head);
    const float iq = inverses[0], ik = inverses[1];
    float previous[kRows], decayed[kRows], q[kRows], k[kRows];
    float prediction = 0.0f;
    const float dy = in.dy;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int row = kg * kRows + r;
      previous[r] = before[r];
      const float matrix = after[r];
      q[r] = raw_q[row] * iq / norm_scale;
      k[r] = raw_k[row] * ik;
      decayed[r] = previous[r] * s.decay;
      prediction += decayed[r] * k[r];
      // dq[row] = sum over columns of S_{t+1}[row, column] dy[column]
      q_products[row][c] = matrix * dy;
      dm[r] += q[r] * dy;
    }
    prediction = column_total(prediction, scratch, kg, c);
    if (tid < kMaxKey) {
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < kColumns; ++j) sum += q_products[tid][j];
      dq_rows[tid] = sum;
    }
    const float difference = in.v - prediction;
    const float delta = difference * s.beta;
    float ddelta = 0.0f;
#pragma unroll
    for (int r = 0; r < kRows; ++r) ddelta += dm[r] * k[r];
    ddelta = column_total(ddelta, scratch, kg, c);
    const float dv = ddelta * s.beta;
    if (kg == 0 && column_ok)
      a.dpost[1LL * t * channels + 2 * a.kh * a.kd + head * a.vd + column] = dv;
    float dg = 0.0f;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const int row = kg * kRows + r;
      k_products[row][c] = dm[r] * delta - decayed[r] * dv;
      const float ddecayed = dm[r] - k[r] * dv;
      dg += ddecayed * previous[r];
      dm[r] = ddecayed * s.decay;
      after[r] = before[r];
      before[r] = ahead[r];
    }
    // workgroup sums: dg over every element, d beta over the columns
    float db_partial = kg == 0 ? ddelta * difference : 0.0f;
    dg = wave_sum(dg);
    db_partial = wave_sum(db_partial);
    if (tid % 64 == 0) {
      block_sums[wave][0] = dg;
      block_sums[wave][1] = db_partial;
    }
    __syncthreads();
    if (tid < kMaxKey) {
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < kColumns; ++j) sum += k_products[tid][j];
      dk_rows[tid] = sum;
    }
    __syncthreads();
    const long long partial = (1LL * t * a.vh + head) * tiles + tile;
    if (tid < 64) {
      // the two row-space gradients back through the L2 normalisation
      float q_dot = 0.0f, k_dot = 0.0f;
      for (int d = tid; d < kMaxKey; d += 64) {
        q_dot += dq_rows[d] * raw_q[d];
        k_dot += dk_rows[d] * raw_k[d];
      }
      q_dot = wave_sum(q_dot);
      k_dot = wave_sum(k_dot);
      for (int d = tid; d < a.kd; d += 64) {
        a.qk_partials[partial * 2 * a.kd + d] =
            (dq_rows[d] * iq - raw_q[d] * iq * iq * iq * q_dot) / norm_scale;
        a.qk_partials[partial * 2 * a.kd + a.kd + d] =
            dk_rows[d] * ik - raw_k[d] * ik * ik * ik * k_dot;
      }
      if (tid == 0) {
        const float dg_total = (block_sums[0][0] + block_sums[1][0]) + (block_sums[2][0] + block_sums[3][0]);
        const float db_total = (block_sums[0][1] + block_sums[1][1]) + (block_sums[2][1] + block_sums[3][1]);
        a.scalar_partials[partial * 3 + 0] = -dg_total * s.decay * s.rate / (1.0f + expf(-s.alpha));
        a.scalar_partials[partial * 3 + 1] = db_total * s.sigmoid * (1.0f - s.sigmoid);
        a.scalar_partials[partial * 3 + 2] = -dg_total * s.decay * s.rate * s.softplus;
      }
    }
    __syncthreads();
  }
}

// One wave per (token, head) row of value_dim <= 256 channels.
__global__ void __launch_bounds__(64)
output_backward_kernel(const float* core, const uint16_t* z, const float* __restrict__ norm,
                       const float* dy, int vd, float epsilon, bool round, float* dcore,
                       float* dz, float* norm_partials) {
  const long long row = blockIdx.x;
  const int lane = threadIdx.x;
  float x[4], dn[4], gate[4], sigmoid[4], grad[4];
  float squares = 0.0f, dot = 0.0f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = lane + 64 * j;
    x[j] = dn[j] = gate[j] = sigmoid[j] = grad[j] = 0.0f;
    if (c < vd) {
      x[j] = core[row * vd + c];
      gate[j] = bf16_bits_to_float(z[row * vd + c]);
      sigmoid[j] = 1.0f / (1.0f + expf(-gate[j]));
      grad[j] = dy[row * vd + c];
      dn[j] = grad[j] * gate[j] * sigmoid[j] * norm[c];
    }
    squares += x[j] * x[j];
    dot += dn[j] * x[j];
  }
  squares = wave_sum(squares);
  dot = wave_sum(dot);
  const float inverse = rsqrtf(squares / static_cast<float>(vd) + epsilon);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = lane + 64 * j;
    if (c >= vd) continue;
    const float normalized = round_if(x[j] * inverse, round);
    const float affine = round_if(normalized * norm[c], round);
    dcore[row * vd + c] = inverse * dn[j] - x[j] * inverse * inverse * inverse / static_cast<float>(vd) * dot;
    dz[row * vd + c] = grad[j] * affine * sigmoid[j] * (1.0f + gate[j] * (1.0f - sigmoid[j]));
    if (norm_partials) norm_partials[row * vd + c] = grad[j] * gate[j] * sigmoid[j] * normalized;
  }
}

// The same for rows of 128: sixteen lanes a row, eight channels a lane; a workgroup
// walks rows `blocks` runs of sixteen apart and keeps its share of the norm weight's
// gradient in registers.  WIDE: the caller's tensors are 16-byte aligned.
constexpr int kOutputBlocks = 1024;
template <bool WIDE>
__global__ void __launch_bounds__(256)
output_backward128_kernel(const float* __restrict__ core, const uint16_t* __restrict__ z,
                          const float* __restrict__ norm, const float* __restrict__ dy,
                          long long rows, float epsilon, bool round, float* __restrict__ dcore,
                          float* __restrict__ dz, float* __restrict__ norm_partial) {
  __shared__ float sums[16][128];
  const int c = 8 * (threadIdx.x % 16), slot = threadIdx.x / 16;
  float weight[8], total[8];
  load8<WIDE>(norm + c, weight);
#pragma unroll
  for (int e = 0; e < 8; ++e) total[e] = 0.0f;
  for (long long first = 16LL * blockIdx.x; first < rows; first += 16LL * gridDim.x) {
    const bool exists = first + slot < rows;
    const long long at = (exists ? first + slot : rows - 1) * 128 + c;
    float x[8], gate[8], grad[8], sigmoid[8], dn[8];
    load8<true>(core + at, x);
    load8<WIDE>(z + at, gate);
    load8<WIDE>(dy + at, grad);
    float squares = 0.0f, dot = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      sigmoid[e] = 1.0f / (1.0f + expf(-gate[e]));
      dn[e] = grad[e] * gate[e] * sigmoid[e] * weight[e];
      squares += x[e] * x[e];
      dot += dn[e] * x[e];
    }
#pragma unroll
    for (int offset = 8; offset > 0; offset >>= 1) {
      squares += __shfl_xor(squares, offset, 64);
      dot += __shfl_xor(dot, offset, 64);
    }
    if (!exists) continue;
    const float inverse = rsqrtf(squares / 128.0f + epsilon);
    const float cubic = inverse * inverse * inverse / 128.0f * dot;
    float dx[8], dgate[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float normalized = round_if(x[e] * inverse, round);
      const float affine = round_if(normalized * weight[e], round);
      dx[e] = inverse * dn[e] - x[e] * cubic;
      dgate[e] = grad[e] * affine * sigmoid[e] * (1.0f + gate[e] * (1.0f - sigmoid[e]));
      total[e] += grad[e] * gate[e] * sigmoid[e] * normalized;
    }
    store8<true>(dcore + at, dx);
    store8<WIDE>(dz + at, dgate);
  }
  if (!norm_partial) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) sums[slot][c + e] = total[e];
  __syncthreads();
  if (threadIdx.x < 128) {
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) sum += sums[i][threadIdx.x];
    norm_partial[128LL * blockIdx.x + threadIdx.x] = sum;
  }
}

// gradient[c] += sum over rows of parts[row, c], eight columns a workgroup, 128
// threads a column, in a fixed order.
__global__ void __launch_bounds__(1024)
sum_columns_kernel(const float* parts, int rows, int width, float* gradient) {
  __shared__ float sums[128][8], groups[16][8];
  const int k = threadIdx.x % 8, g = threadIdx.x / 8, c = blockIdx.x * 8 + k;
  float sum = 0.0f;
  if (c < width)
    for (int row = g; row < rows; row += 128) sum += parts[1LL * row * width + c];
  sums[g][k] = sum;
  __syncthreads();
  if (g < 16) {
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) total += sums[8 * g + i][k];
    groups[g][k] = total;
  }
  __syncthreads();
  if (g != 0 || c >= width) return;
  float total = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) total += groups[i][k];
  gradient[c] += total;
}

// Heads of a key head and their column tiles add up, in ascending order.
__global__ void __launch_bounds__(128)
gather_qk_kernel(const float* partials, int kh, int vh, int kd, int tiles, int channels,
                 float* dpost) {
  const int key_head = blockIdx.x, t = blockIdx.y, d = threadIdx.x;
  if (d >= kd) return;
  const int group = vh / kh;
  float dq = 0.0f, dk = 0.0f;
  for (int h = key_head * group; h < (key_head + 1) * group; ++h)
    for (int tile = 0; tile < tiles; ++tile) {
      const long long at = ((1LL * t * vh + h) * tiles + tile) * 2 * kd;
      dq += partials[at + d];
      dk += partials[at + kd + d];
    }
  dpost[1LL * t * channels + key_head * kd + d] = dq;
  dpost[1LL * t * channels + (kh + key_head) * kd + d] = dk;
}

// da, db per token; the two per-head parameter gradients summed over the
// sequence by one workgroup per head in a fixed order.
__global__ void __launch_bounds__(256)
gather_scalar_kernel(const float* partials, int length, int vh, int tiles, float* da, float* db,
                     float* da_log, float* ddt_bias) {
  __shared__ float sums[256][2];
  const int head = blockIdx.x, tid = threadIdx.x;
  float log_sum = 0.0f, bias_sum = 0.0f;
  // eight tokens a thread are requested together (one at a time: 12.6 us at 2048 tokens,
  // 9.6 us so)
  for (int t0 = tid; t0 < length; t0 += 8 * 256) {
    float ga[8], gb[8], glog[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const long long at = (1LL * min(t0 + 256 * i, length - 1) * vh + head) * tiles * 3;
      ga[i] = partials[at], gb[i] = partials[at + 1], glog[i] = partials[at + 2];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int t = t0 + 256 * i;
      if (t >= length) break;
      for (int tile = 1; tile < tiles; ++tile) {
        const long long at = ((1LL * t * vh + head) * tiles + tile) * 3;
        ga[i] += partials[at];
        gb[i] += partials[at + 1];
        glog[i] += partials[at + 2];
      }
      da[1LL * t * vh + head] = ga[i];
      db[1LL * t * vh + head] = gb[i];
      log_sum += glog[i];
      bias_sum += ga[i];
    }
  }
  sums[tid][0] = log_sum;
  sums[tid][1] = bias_sum;
  __syncthreads();
  for (int width = 128; width > 0; width >>= 1) {
    if (tid < width) {
      sums[tid][0] += sums[tid + width][0];
      sums[tid][1] += sums[tid + width][1];
    }
    __syncthreads();
  }
  if (tid == 0) {
    if (da_log) da_log[head] += sums[0][0];
    if (ddt_bias) ddt_bias[head] += sums[0][1];
  }
}

template <int VEC>
__global__ void __launch_bounds__(256)
conv_silu_backward_kernel(const float* pre, const float* dpost, long long elements, float* dpre) {
  const long long i = (blockIdx.x * 256LL + threadIdx.x) * VEC;
  if (i >= elements) return;
  const Pack<VEC> x = load_floats<VEC>(pre + i), g = load_floats<VEC>(dpost + i);
  Pack<VEC> r;
#pragma unroll
  for (int e = 0; e < VEC; ++e) {
    const float sigmoid = 1.0f / (1.0f + expf(-x.e[e]));
    r.e[e] = g.e[e] * sigmoid * (1.0f + x.e[e] * (1.0f - sigmoid));
  }
  store_floats<VEC>(dpre + i, r);
}

template <int VEC>
__global__ void __launch_bounds__(256)
conv_input_backward_kernel(const float* dpre, const float* __restrict__ weight, int length,
                           int channels, int kernel, float* dx) {
  const int groups = channels / VEC;
  const long long i = blockIdx.x * 256LL + threadIdx.x;
  if (i >= 1LL * length * groups) return;
  const int c = static_cast<int>(i % groups) * VEC, t = static_cast<int>(i / groups);
  Pack<VEC> sum;
#pragma unroll
  for (int e = 0; e < VEC; ++e) sum.e[e] = 0.0f;
  for (int tap = 0; tap < kernel; ++tap) {
    const int future = t + kernel - 1 - tap;
    if (future >= length) continue;
    const Pack<VEC> g = load_floats<VEC>(dpre + 1LL * future * channels + c);
#pragma unroll
    for (int e = 0; e < VEC; ++e) sum.e[e] += g.e[e] * weight[1LL * (c + e) * kernel + tap];
  }
  store_floats<VEC>(dx + 1LL * t * channels + c, sum);
}

// dw[c, tap] += sum over t of dpre[t, c] x[t + tap - kernel + 1, c], in two
// levels with a fixed order: blockIdx.z sums one slice of the tokens.
__global__ void __launch_bounds__(256)
conv_weight_partial_kernel(const uint16_t* input, const float* dpre, int length, int channels,
                           int kernel, int slices, float* partial) {
  const int c = blockIdx.x * 256 + threadIdx.x, tap = blockIdx.y, slice = blockIdx.z;
  if (c >= channels) return;
  const int per = (length + slices - 1) / slices;
  const int first = max(slice * per, kernel - 1 - tap), last = min((slice + 1) * per, length);
  float sum = 0.0f;
  for (int t = first; t < last; ++t)
    sum += dpre[1LL * t * channels + c] *
           bf16_bits_to_float(input[1LL * (t + tap - kernel + 1) * channels + c]);
  partial[(1LL * slice * channels + c) * kernel + tap] = sum;
}

__global__ void __launch_bounds__(256)
conv_weight_final_kernel(const float* partial, long long elements, int slices, float* dw) {
  const long long i = blockIdx.x * 256LL + threadIdx.x;
  if (i >= elements) return;
  float sum = 0.0f;
#pragma unroll 16
  for (int slice = 0; slice < slices; ++slice) sum += partial[slice * elements + i];
  dw[i] += sum;
}

// The ends of the chunked backward's parameter gradients in one launch: the first blocks add
// up the norm's as sum_columns_kernel does, two columns each, the next the gates', 32 heads
// each, and the rest the convolution's.  (Three launches of 4.9, 9.5 and 4.7 us at 2048 tokens
// of 48 heads, most of it the arrival of code and arguments, now 5.6; da and db came the way of
// the gates' parameters then.)
struct FinishArgs {
  const float* norm_parts = nullptr;    // [norm_rows, norm_width]
  float* d_norm = nullptr;
  int norm_rows = 0, norm_width = 0, norm_blocks = 0;
  const float* scalar_parts = nullptr;  // [chunks, heads, 2]
  float *d_a_log = nullptr, *d_dt_bias = nullptr;
  int chunks = 0, heads = 0, head_blocks = 0;
  const float* conv_parts = nullptr;    // [slices, weights]
  float* d_conv = nullptr;
  long long weights = 0;
  int slices = 0;
};
__global__ void __launch_bounds__(256)
finish_parameters_kernel(FinishArgs a) {
  const int tid = threadIdx.x, block = blockIdx.x;
  if (block < a.norm_blocks) {
    __shared__ float sums[128][2], groups[16][2];
    const int k = tid % 2, g = tid / 2, c = 2 * block + k;
    float sum = 0.0f;
#pragma unroll 8
    for (int row = g; row < a.norm_rows; row += 128) sum += a.norm_parts[1LL * row * a.norm_width + c];
    sums[g][k] = sum;
    __syncthreads();
    if (g < 16) {
      float total = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) total += sums[8 * g + i][k];
      groups[g][k] = total;
    }
    __syncthreads();
    if (g != 0) return;
    float total = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) total += groups[i][k];
    a.d_norm[c] += total;
    return;
  }
  if (block < a.norm_blocks + a.head_blocks) {
    // a head's chunks in eight parts
    __shared__ float parts[8][32][2];
    const int head = 32 * (block - a.norm_blocks) + tid % 32, part = tid / 32;
    float log_sum = 0.0f, bias_sum = 0.0f;
    if (head < a.heads) {
#pragma unroll 4
      for (int chunk = part; chunk < a.chunks; chunk += 8) {
        const float2 v = *reinterpret_cast<const float2*>(a.scalar_parts + 2 * (1LL * chunk * a.heads + head));
        log_sum += v.x;
        bias_sum += v.y;
      }
    }
    parts[part][tid % 32][0] = log_sum;
    parts[part][tid % 32][1] = bias_sum;
    __syncthreads();
    if (part != 0 || head >= a.heads) return;
#pragma unroll
    for (int i = 1; i < 8; ++i) log_sum += parts[i][tid][0], bias_sum += parts[i][tid][1];
    if (a.d_a_log) a.d_a_log[head] += log_sum;
    if (a.d_dt_bias) a.d_dt_bias[head] += bias_sum;
    return;
  }
  const long long i = (block - a.norm_blocks - a.head_blocks) * 256LL + tid;
  if (i >= a.weights) return;
  float sum = 0.0f;
#pragma unroll 16
  for (int slice = 0; slice < a.slices; ++slice) sum += a.conv_parts[slice * a.weights + i];
  a.d_conv[i] += sum;
}

// gradient[c] += sum over rows of partials[row, c], two levels, fixed order.
// Sum of rows first..last-1 of a [rows, width] matrix (width <= 256), per
// column.  The 256 threads form up to 8 groups of `width`; group g takes rows
// first + g, first + g + groups, ...; the groups' sums are added in ascending
// order.  Returns the column's total in the threads of group 0.
__device__ inline float sum_block_rows(const float* parts, long long first, long long last,
                                       int width) {
  __shared__ float scratch[8][256];
  const int fit = 256 / width, groups = fit < 8 ? fit : 8;
  const int c = threadIdx.x % width, g = threadIdx.x / width;
  if (g < groups) {
    float sum = 0.0f;
#pragma unroll 8
    for (long long row = first + g; row < last; row += groups) sum += parts[row * width + c];
    scratch[g][c] = sum;
  }
  __syncthreads();
  float total = 0.0f;
  if (g == 0)
    for (int j = 0; j < groups; ++j) total += scratch[j][c];
  return total;
}

__global__ void __launch_bounds__(256)
sum_rows_partial_kernel(const float* parts, long long rows, int width, int chunks, float* partial) {
  const long long per = (rows + chunks - 1) / chunks;
  const long long first = blockIdx.x * per;
  const long long last = first + per < rows ? first + per : rows;
  const float total = sum_block_rows(parts, first, last, width);
  if (threadIdx.x < width) partial[1LL * blockIdx.x * width + threadIdx.x] = total;
}

__global__ void __launch_bounds__(256)
sum_rows_final_kernel(const float* partial, int chunks, int width, float* gradient) {
  const float total = sum_block_rows(partial, 0, chunks, width);
  if (threadIdx.x < width) gradient[threadIdx.x] += total;
}

unsigned blocks_for(long long elements) { return static_cast<unsigned>((elements + 255) / 256); }

}  // namespace

bool force_generic();  // mha_capi.hip

namespace {
bool use_chunks(const pluto_hip_delta_params* p) {
  return !force_generic() && gdn_backward_chunked_supported(p);
}
// Whether the kernels for four taps serve these widths.
bool four_taps(const pluto_hip_delta_params* p) {
  const int channels = 2 * p->key_heads * p->key_head_dim + p->value_heads * p->value_head_dim;
  return p->conv_kernel_dim == 4 && channels % 4 == 0 && p->key_head_dim % 2 == 0;
}
}  // namespace

size_t gdn_backward_workspace_bytes(const pluto_hip_delta_params* p, int length, bool norm_grad) {
  const size_t T = static_cast<size_t>(length);
  const size_t kh = p->key_heads, vh = p->value_heads, kd = p->key_head_dim, vd = p->value_head_dim;
  const size_t channels = 2 * kh * kd + vh * vd;
  const bool chunked = use_chunks(p);
  const size_t tiles = chunked ? 1 : (vd + kColumns - 1) / kColumns;
  size_t bytes = 0;
  // post, dpost, and what only the general convolution stores: pre, dpre
  bytes += (four_taps(p) ? 2 : 4) * align_up(T * channels * 4, 256);
  bytes += 2 * align_up(T * vh * vd * 4, 256);           // core, dcore
  bytes += chunked ? gdn_backward_chunked_bytes(p, length)
                   : align_up((T + 1) * vh * kd * vd * 4, 256);  // states
  bytes += align_up(T * vh * tiles * 2 * kd * 4, 256);   // q/k partials
  bytes += align_up(T * vh * tiles * 3 * 4, 256);        // scalar partials
  if (norm_grad && vd == 128)
    bytes += align_up(kOutputBlocks * vd * 4, 256);
  else if (norm_grad)
    bytes += align_up(T * vh * vd * 4, 256) + align_up(kGdnSumChunks * vd * 4, 256);
  bytes += align_up(kConvSlices * channels * p->conv_kernel_dim * 4, 256);  // conv weight partials
  return bytes;
}

int launch_gdn_backward(hipStream_t stream, const pluto_hip_delta_params* p, int length,
                        const void* qkv, const void* z, const void* a, const void* b,
                        const float* conv_weight, const float* a_log, const float* dt_bias,
                        const float* norm, const float* dy, float* dqkv, float* dz, float* da,
                        float* db, float* d_conv_weight, float* d_a_log, float* d_dt_bias,
                        float* d_norm, void* workspace) {
  note_path(use_chunks(p) ? PLUTO_HIP_PATH_CHUNKED : PLUTO_HIP_PATH_RECURRENCE);
  const size_t T = static_cast<size_t>(length);
  const int kh = p->key_heads, vh = p->value_heads, kd = p->key_head_dim, vd = p->value_head_dim;
  const int channels = 2 * kh * kd + vh * vd, kernel = p->conv_kernel_dim;
  const bool chunked = use_chunks(p);
  const int tiles = chunked ? 1 : (vd + kColumns - 1) / kColumns;
  const bool round = p->round_to_bfloat16 != 0;
  char* at = static_cast<char*>(workspace);
  auto take = [&](size_t bytes) {
    char* result = at;
    at += align_up(bytes, 256);
    return reinterpret_cast<float*>(result);
  };
  const bool taps4 = four_taps(p);
  float* pre = taps4 ? nullptr : take(T * channels * 4);
  float* post = take(T * channels * 4);
  float* dpost = take(T * channels * 4);
  float* dpre = taps4 ? nullptr : take(T * channels * 4);
  float* core = take(T * vh * vd * 4);
  float* dcore = take(T * vh * vd * 4);
  float* states = take(chunked ? gdn_backward_chunked_bytes(p, length) : (T + 1) * vh * kd * vd * 4);
  float* qk_partials = take(T * vh * tiles * 2 * kd * 4);
  float* scalar_partials = take(T * vh * tiles * 3 * 4);
  float* norm_partials =
      d_norm ? take((vd == 128 ? static_cast<size_t>(kOutputBlocks) : T * vh) * vd * 4) : nullptr;
  float* norm_chunks =
      d_norm && vd != 128 ? take(static_cast<size_t>(kGdnSumChunks) * vd * 4) : nullptr;
  float* conv_partials = take(static_cast<size_t>(kConvSlices) * channels * kernel * 4);

  const long long elements = 1LL * length * channels;
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  const bool rows_aligned = aligned(qkv) && aligned(conv_weight) && aligned(dqkv);
  auto convolve = [&](auto* to) {
    const auto* input = static_cast<const uint16_t*>(qkv);
    if (taps4) {
      const dim3 grid((channels / 4 + 255) / 256, (length + kConvRun - 1) / kConvRun);
      if (rows_aligned)
        conv_train4_kernel<true><<<grid, 256, 0, stream>>>(input, conv_weight, length, channels, round, to);
      else
        conv_train4_kernel<false><<<grid, 256, 0, stream>>>(input, conv_weight, length, channels, round, to);
    } else {
      // one channel a thread: four (one wide access instead of four) were slower in the
      // kernels for any number of taps that also read the weights
      conv_train_kernel<1><<<blocks_for(elements), 256, 0, stream>>>(input, conv_weight, length, channels, kernel,
                                                                     round, pre, to);
    }
  };
  // the chunked kernels take what is rounded to bf16 as such
  if (chunked && round)
    convolve(reinterpret_cast<uint16_t*>(post));
  else
    convolve(post);
  int status = launch_status();
  if (status != 0) return status;
  RecurrenceArgs r;
  r.post = post;
  r.a = static_cast<const uint16_t*>(a);
  r.b = static_cast<const uint16_t*>(b);
  r.a_log = a_log;
  r.dt_bias = dt_bias;
  r.states = states;
  r.core = core;
  r.dcore = dcore;
  r.qk_partials = qk_partials;
  r.scalar_partials = scalar_partials;
  r.dpost = dpost;
  r.length = length;
  r.kh = kh;
  r.vh = vh;
  r.kd = kd;
  r.vd = vd;
  r.round = round;
  GdnChunkedBackward c;
  c.post = post;
  c.a = r.a;
  c.b = r.b;
  c.a_log = a_log;
  c.dt_bias = dt_bias;
  c.dcore = dcore;
  c.core = core;
  c.dpost = dpost;
  c.qk_partials = qk_partials;
  c.da = da;
  c.db = db;
  c.scalar_partials = scalar_partials;
  c.records = states;
  c.length = length;
  c.key_heads = kh;
  c.value_heads = vh;
  c.round = round;
  if (chunked) {
    status = launch_gdn_backward_chunked_forward(stream, c);
  } else {
    recurrence_states_kernel<<<vh * tiles, 256, 0, stream>>>(r);
    status = launch_status();
  }
  if (status != 0) return status;
  int norm_rows = 0;  // of the partial sums for the norm's gradient
  if (vd == 128) {
    const long long rows = 1LL * length * vh, runs = (rows + 15) / 16;
    const int blocks = static_cast<int>(runs < kOutputBlocks ? runs : kOutputBlocks);
    const auto* gates = static_cast<const uint16_t*>(z);
    if (aligned(z) && aligned(norm) && aligned(dy) && aligned(dz))
      output_backward128_kernel<true><<<blocks, 256, 0, stream>>>(
          core, gates, norm, dy, rows, p->rms_norm_epsilon, round, dcore, dz, norm_partials);
    else
      output_backward128_kernel<false><<<blocks, 256, 0, stream>>>(
          core, gates, norm, dy, rows, p->rms_norm_epsilon, round, dcore, dz, norm_partials);
    norm_rows = blocks;
    if (d_norm && !chunked) sum_columns_kernel<<<16, 1024, 0, stream>>>(norm_partials, blocks, vd, d_norm);
  } else {
    output_backward_kernel<<<static_cast<unsigned>(length) * vh, 64, 0, stream>>>(
        core, static_cast<const uint16_t*>(z), norm, dy, vd, p->rms_norm_epsilon, round, dcore, dz,
        norm_partials);
  }
  status = launch_status();
  if (status != 0) return status;
  if (d_norm && vd != 128) {
    sum_rows_partial_kernel<<<kGdnSumChunks, 256, 0, stream>>>(norm_partials, 1LL * length * vh, vd,
                                                               kGdnSumChunks, norm_chunks);
    sum_rows_final_kernel<<<1, 256, 0, stream>>>(norm_chunks, kGdnSumChunks, vd, d_norm);
    status = launch_status();
    if (status != 0) return status;
  }
  if (chunked) {
    status = launch_gdn_backward_chunked_reverse(stream, c);
  } else {
    recurrence_backward_kernel<<<vh * tiles, 256, 0, stream>>>(r);
    status = launch_status();
  }
  if (status != 0) return status;
  if (!chunked)
    gather_scalar_kernel<<<vh, 256, 0, stream>>>(scalar_partials, length, vh, tiles, da, db, d_a_log,
                                                 d_dt_bias);
  const long long weights = 1LL * channels * kernel;
  auto finish_parameters = [&](int conv_slices) {
    if (!chunked) {
      if (d_conv_weight)
        conv_weight_final_kernel<<<blocks_for(weights), 256, 0, stream>>>(conv_partials, weights, conv_slices,
                                                                          d_conv_weight);
      return launch_status();
    }
    FinishArgs f;
    f.norm_parts = norm_partials;
    f.d_norm = d_norm;
    f.norm_rows = norm_rows;
    f.norm_width = vd;
    f.norm_blocks = d_norm ? vd / 2 : 0;
    f.scalar_parts = scalar_partials;
    f.d_a_log = d_a_log;
    f.d_dt_bias = d_dt_bias;
    f.chunks = (length + 63) / 64;
    f.heads = vh;
    f.head_blocks = d_a_log || d_dt_bias ? (vh + 31) / 32 : 0;
    f.conv_parts = conv_partials;
    f.d_conv = d_conv_weight;
    f.weights = d_conv_weight ? weights : 0;
    f.slices = conv_slices;
    const unsigned blocks = f.norm_blocks + f.head_blocks + static_cast<unsigned>((f.weights + 255) / 256);
    if (blocks > 0) finish_parameters_kernel<<<blocks, 256, 0, stream>>>(f);
    return launch_status();
  };
  if (taps4) {
    ConvBackwardArgs b;
    b.input = static_cast<const uint16_t*>(qkv);
    b.weight = conv_weight;
    b.qk_partials = qk_partials;
    b.dpost = dpost;
    b.dx = dqkv;
    b.partial = d_conv_weight ? conv_partials : nullptr;
    b.length = length;
    b.channels = channels;
    b.kh = kh;
    b.vh = vh;
    b.kd = kd;
    b.tiles = tiles;
    // a run repeats three rows of the next one: sixteen tokens at least, and no
    // more runs than there are slices of partial sums
    b.run = (length + kConvSlices - 1) / kConvSlices;
    if (b.run < 16) b.run = 16;
    b.round = round;
    const int runs = (length + b.run - 1) / b.run;
    const dim3 grid((channels / 2 + 255) / 256, runs);
    if (rows_aligned)
      conv_backward4_kernel<true><<<grid, 256, 0, stream>>>(b);
    else
      conv_backward4_kernel<false><<<grid, 256, 0, stream>>>(b);
    return finish_parameters(runs);
  }
  gather_qk_kernel<<<dim3(kh, length), 128, 0, stream>>>(qk_partials, kh, vh, kd, tiles, channels,
                                                         dpost);
  if (elements % 4 == 0)
    conv_silu_backward_kernel<4><<<blocks_for(elements / 4), 256, 0, stream>>>(pre, dpost, elements,
                                                                               dpre);
  else
    conv_silu_backward_kernel<1><<<blocks_for(elements), 256, 0, stream>>>(pre, dpost, elements,
                                                                           dpre);
  conv_input_backward_kernel<1><<<blocks_for(elements), 256, 0, stream>>>(
      dpre, conv_weight, length, channels, kernel, dqkv);
  if (d_conv_weight)
    conv_weight_partial_kernel<<<dim3((channels + 255) / 256, kernel, kConvSlices), 256, 0, stream>>>(
        static_cast<const uint16_t*>(qkv), dpre, length, channels, kernel, kConvSlices,
        conv_partials);
  return finish_parameters(kConvSlices);
}

}  // namespace pluto_hip
