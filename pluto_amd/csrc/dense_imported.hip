// FullyConnectedLayer, imported path (src/llm/layers/fully_connected.cc):
//   ImportedMatVecKernel          :40-68   y = bf16(W x), W output-major
//   QuantizeImportedInputKernel   :70-88   FP8 storage: x -> fp8(x / s) * s in
//                                          groups of 128, s = max|x| / 448
//   ImportedForward               :295-341 bf16 token -> fp32 -> (quantize) ->
//                                          mat-vec -> bf16
// One frozen checkpoint matrix [output_dim, input_dim] in bf16, fp32 or OCP
// FP8 E4M3 with FP32 scales [ceil(out/128), ceil(in/128)] times one bf16
// token.  Byte-bound: every weight is read once.  A wave owns four output
// rows and reads them in 16-byte pieces (whenever rows start 16-byte aligned),
// a single token is prepared by the workgroups themselves, several come from the
// FP32 copy a kernel of their own leaves in the workspace; all arithmetic is
// FP32, the 64 lane sums are added by a butterfly.
#include <algorithm>

#include "dense.h"

namespace pluto_hip {
namespace {

constexpr int kGroup = 128;  // quantization group and scale block edge

// Value of an OCP FP8 E4M3 code: 1-4-3 bits, bias 7, no infinities, S.1111.111
// is NaN, subnormals m * 2^-9.
__device__ inline float fp8_value(uint32_t bits) {
  const uint32_t exponent = (bits >> 3) & 15u, mantissa = bits & 7u;
  float magnitude;
  if (exponent == 0)
    magnitude = static_cast<float>(mantissa) * 0.001953125f;
  else if (exponent == 15 && mantissa == 7)
    magnitude = __builtin_nanf("");
  else
    magnitude = __uint_as_float(((exponent + 120u) << 23) | (mantissa << 20));
  return (bits & 0x80u) ? -magnitude : magnitude;
}

// FP8 quantization of a group of 128 token values (fully_connected.cc:70-88):
// scale = largest / 448, code = fp8(v / max(scale, 1e-12)), value = code * scale
// (only the divisor is floored).  The division is a multiplication by the
// group's reciprocal with one correction step, which rounds as the division
// does, and the rounding is the hardware conversion: six instructions a value
// where a divide and a rounding by parts took sixty, 9 us of a one-token
// projection whose workgroups each prepare the token.
struct GroupQuantizer {
  float scale, divisor, inverse;
  __device__ explicit GroupQuantizer(float largest) {
    scale = largest / 448.0f;
    divisor = fmaxf(scale, 1e-12f);
    inverse = 1.0f / divisor;
  }
  __device__ float quotient(float v) const {
    const float q = v * inverse;
    const float corrected = __builtin_fmaf(__builtin_fmaf(-q, divisor, v), inverse, q);
    return fminf(fmaxf(corrected, -448.0f), 448.0f);
  }
  // The FP8 values (unscaled) nearest to the two quotients, as floats.
  __device__ void round(float first, float second, float& a, float& b) const {
    const int codes = __builtin_amdgcn_cvt_pk_fp8_f32(quotient(first), quotient(second), 0, false);
    const auto values = __builtin_amdgcn_cvt_pk_f32_fp8(codes, false);
    a = values[0];
    b = values[1];
  }
};

// token[i] = float(x[i]), for FP8 storage quantized per group of 128.
template <bool FP8>
__global__ void __launch_bounds__(kGroup)
imported_token_kernel(const uint16_t* x, int n, float* token) {
  __shared__ float largest[2];
  x += static_cast<size_t>(blockIdx.y) * n;      // one token per grid row
  token += static_cast<size_t>(blockIdx.y) * n;
  const int i = blockIdx.x * kGroup + threadIdx.x;
  const float v = i < n ? bf16_bits_to_float(x[i]) : 0.0f;
  if constexpr (!FP8) {
    if (i < n) token[i] = v;
  } else {
    const float mine = wave_max(fabsf(v));
    if (threadIdx.x % 64 == 0) largest[threadIdx.x / 64] = mine;
    __syncthreads();
    const GroupQuantizer quantizer(fmaxf(largest[0], largest[1]));
    float value, unused;
    quantizer.round(v, 0.0f, value, unused);
    if (i < n) token[i] = value * quantizer.scale;
  }
}

// Several matrices applied to the same tokens in one launch: workgroup b works on
// matrix i with first_block[i] <= b < first_block[i + 1].
constexpr int kManyMax = 8;
struct MatVecArgs {
  const void* weights[kManyMax];
  const float* scales[kManyMax];  // FP8 only
  uint16_t* out[kManyMax];        // [tokens, rows]
  int rows[kManyMax];
  int first_block[kManyMax + 1];
  int matrices = 0;
  const uint16_t* input = nullptr;  // one bf16 token, when the kernel prepares it itself
  const float* token = nullptr;     // else [tokens, cols], prepared
  int cols = 0;
};

typedef float floatx2 __attribute__((ext_vector_type(2)));

// Four FP8 E4M3 codes of a word as floats, by the hardware conversion.
__device__ inline void fp8_word(uint32_t word, float* out) {
  const floatx2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(word), false);
  const floatx2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(word), true);
  out[0] = lo.x, out[1] = lo.y, out[2] = hi.x, out[3] = hi.y;
}

constexpr int kRowsPerWave = 4;

// The matrix a workgroup works on.
struct MatVecTarget {
  const unsigned char* weights;
  const float* scales;
  uint16_t* out;
  int rows, block;
};
__device__ inline MatVecTarget matvec_target(const MatVecArgs& a) {
  int which = 0;
  while (which + 1 < a.matrices && static_cast<int>(blockIdx.x) >= a.first_block[which + 1]) ++which;
  return {static_cast<const unsigned char*>(a.weights[which]), a.scales[which], a.out[which],
          a.rows[which], static_cast<int>(blockIdx.x) - a.first_block[which]};
}

// STORAGE: 0 bf16, 1 fp32, 2 FP8 E4M3.  A wave owns four consecutive output
// rows, a lane takes 16-byte pieces of them at the same columns: pieces lane,
// lane + 64, ...  BATCH pieces of all four rows are requested before the first is
// used: a workgroup's whole share of the weights is a few tens of KiB and the
// grid of a projection fits the chip at once, so what matters is how much of it
// travels together.  TOKENS tokens share one pass over the weights; each token's
// sum is formed in the order of the one-token kernel.  PREPARE (one token): the
// workgroup converts (FP8: quantizes) the token itself while its first weights
// travel, instead of reading what a launch of its own left in memory; in LDS the
// quarters of a piece lie apart, so that the lanes read consecutive 16 bytes.
// 5120 -> 12288 + 1024 + 1024 in FP8, one token: 41 us as a token and a mat-vec
// launch a matrix, 17 us as one launch.
template <int STORAGE, int TOKENS, int STEPS, bool PREPARE>
__global__ void __launch_bounds__(256, TOKENS > 1 ? 1 : PREPARE && STORAGE == 2 && STEPS < 8 ? 4 : 3)
imported_matvec_kernel(MatVecArgs a) {
  constexpr int kElementBytes = STORAGE == 0 ? 2 : (STORAGE == 1 ? 4 : 1);
  constexpr int kPiece = 16 / kElementBytes;  // elements per 16-byte load
  constexpr int kQuads = kPiece / 4;
  constexpr int R = kRowsPerWave, BATCH = STEPS < 4 ? STEPS : 4;
  extern __shared__ float4 token_lds[];  // PREPARE: [kQuads][pieces]
  const int lane = threadIdx.x % 64;
  const MatVecTarget m = matvec_target(a);
  const int row0 = (m.block * 4 + threadIdx.x / 64) * R;
  const int pieces = a.cols / kPiece;
  const unsigned char* row_start[R];
#pragma unroll
  for (int r = 0; r < R; ++r)  // rows past the end repeat the last one
    row_start[r] = m.weights + static_cast<size_t>(min(row0 + r, m.rows - 1)) * a.cols * kElementBytes;
  // the four rows lie in one 128-row block of scales
  const float* scale_row =
      STORAGE == 2 ? m.scales + static_cast<size_t>(min(row0, m.rows - 1) / kGroup) *
                                    ((a.cols + kGroup - 1) / kGroup)
                   : nullptr;
  uint4 raw[BATCH][R];
  float scale[BATCH];
  auto request = [&](int b, int first) {
    const int p = min(first + lane, pieces - 1);
#pragma unroll
    for (int r = 0; r < R; ++r)
      raw[b][r] = *reinterpret_cast<const uint4*>(row_start[r] + static_cast<size_t>(p) * 16);
    scale[b] = STORAGE == 2 ? scale_row[p * kPiece / kGroup] : 1.0f;
  };
#pragma unroll
  for (int b = 0; b < BATCH; ++b) request(b, 64 * b);
  if constexpr (PREPARE) {
    static_assert(TOKENS == 1);
    for (int c = threadIdx.x * 8; c < (a.cols + 127) / 128 * 128; c += 2048) {
      // sixteen lanes hold a group of 128
      uint4 bits = make_uint4(0, 0, 0, 0);
      if (c < a.cols) bits = *reinterpret_cast<const uint4*>(a.input + c);
      const uint32_t words[4] = {bits.x, bits.y, bits.z, bits.w};
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = __uint_as_float(e % 2 ? words[e / 2] & 0xffff0000u : words[e / 2] << 16);
      if constexpr (STORAGE == 2) {
        float largest = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) largest = fmaxf(largest, fabsf(v[e]));
#pragma unroll
        for (int offset = 8; offset > 0; offset >>= 1)
          largest = fmaxf(largest, __shfl_xor(largest, offset, 64));
        const GroupQuantizer quantizer(largest);
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
          quantizer.round(v[e], v[e + 1], v[e], v[e + 1]);
          v[e] *= quantizer.scale;
          v[e + 1] *= quantizer.scale;
        }
      }
      if (c < a.cols) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int quad = c / 4 + q;  // of the whole token
          token_lds[quad % kQuads * pieces + quad / kQuads] =
              make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
        }
      }
    }
    __syncthreads();
  }
  if (row0 >= m.rows) return;
  float sum[TOKENS][R];
#pragma unroll
  for (int t = 0; t < TOKENS; ++t)
#pragma unroll
    for (int r = 0; r < R; ++r) sum[t][r] = 0.0f;
  for (int first = 0; first < pieces; first += 64 * STEPS) {
    if (first > 0) {
#pragma unroll
      for (int b = 0; b < BATCH; ++b) request(b, first + 64 * b);
    }
#pragma unroll
    for (int step = 0; step < STEPS; ++step) {
      const int b = step % BATCH;
      // lanes past the end repeat the last piece and count it as nothing
      const bool exists = first + 64 * step + lane < pieces;
      const int p = exists ? first + 64 * step + lane : pieces - 1;
      auto decode = [&](int r, float (&w)[kPiece]) {
        const uint32_t words[4] = {raw[b][r].x, raw[b][r].y, raw[b][r].z, raw[b][r].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if constexpr (STORAGE == 0) {
            w[2 * k] = __uint_as_float(words[k] << 16);
            w[2 * k + 1] = __uint_as_float(words[k] & 0xffff0000u);
          } else if constexpr (STORAGE == 1) {
            w[k] = __uint_as_float(words[k]);
          } else {
            fp8_word(words[k], &w[4 * k]);
          }
        }
      };
      auto token_piece = [&](int t, float (&x)[kPiece]) {
#pragma unroll
        for (int q = 0; q < kQuads; ++q) {
          const float4 v = PREPARE ? token_lds[q * pieces + p]
                                   : *reinterpret_cast<const float4*>(
                                         a.token + static_cast<size_t>(t) * a.cols + p * kPiece + 4 * q);
          x[4 * q] = v.x, x[4 * q + 1] = v.y, x[4 * q + 2] = v.z, x[4 * q + 3] = v.w;
        }
      };
      auto add = [&](int t, int r, const float (&w)[kPiece], const float (&x)[kPiece]) {
        if constexpr (STORAGE == 2) {
          float part = 0.0f;
#pragma unroll
          for (int e = 0; e < kPiece; ++e) part += w[e] * x[e];
          const float total = sum[t][r] + part * scale[b];
          sum[t][r] = exists ? total : sum[t][r];
        } else {
          float total = sum[t][r];
#pragma unroll
          for (int e = 0; e < kPiece; ++e) total += w[e] * x[e];
          sum[t][r] = exists ? total : sum[t][r];
        }
      };
      if constexpr (TOKENS == 1) {
        float x[kPiece];
        token_piece(0, x);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          float w[kPiece];
          decode(r, w);
          add(0, r, w, x);
        }
      } else {
        // decoded once for all tokens
        float w[R][kPiece];
#pragma unroll
        for (int r = 0; r < R; ++r) decode(r, w[r]);
#pragma unroll
        for (int t = 0; t < TOKENS; ++t) {
          float x[kPiece];
          token_piece(t, x);
#pragma unroll
          for (int r = 0; r < R; ++r) add(t, r, w[r], x);
        }
      }
      if (step + BATCH < STEPS) request(b, first + 64 * (step + BATCH));
    }
  }
#pragma unroll
  for (int t = 0; t < TOKENS; ++t)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float total = wave_sum(sum[t][r]);
      if (lane == 0 && row0 + r < m.rows)
        m.out[static_cast<size_t>(t) * m.rows + row0 + r] = float_to_bf16_bits(total);
    }
}

// Rows that do not start 16-byte aligned: one element a lane.
template <int STORAGE, int TOKENS>
__global__ void __launch_bounds__(256) imported_matvec_ragged_kernel(MatVecArgs a) {
  constexpr int R = kRowsPerWave;
  const int lane = threadIdx.x % 64;
  const MatVecTarget m = matvec_target(a);
  const int row0 = (m.block * 4 + threadIdx.x / 64) * R;
  if (row0 >= m.rows) return;
  const int scale_cols = (a.cols + kGroup - 1) / kGroup;
  float sum[TOKENS][R];
#pragma unroll
  for (int t = 0; t < TOKENS; ++t)
#pragma unroll
    for (int r = 0; r < R; ++r) sum[t][r] = 0.0f;
  for (int c = lane; c < a.cols; c += 64) {
    float value[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int row = min(row0 + r, m.rows - 1);  // rows past the end repeat the last one
      const size_t i = static_cast<size_t>(row) * a.cols + c;
      if constexpr (STORAGE == 0)
        value[r] = bf16_bits_to_float(reinterpret_cast<const uint16_t*>(m.weights)[i]);
      else if constexpr (STORAGE == 1)
        value[r] = reinterpret_cast<const float*>(m.weights)[i];
      else
        value[r] = fp8_value(m.weights[i]) *
                   m.scales[static_cast<size_t>(row / kGroup) * scale_cols + c / kGroup];
    }
#pragma unroll
    for (int t = 0; t < TOKENS; ++t) {
      const float x = a.token[static_cast<size_t>(t) * a.cols + c];
#pragma unroll
      for (int r = 0; r < R; ++r) sum[t][r] += value[r] * x;
    }
  }
#pragma unroll
  for (int t = 0; t < TOKENS; ++t)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float total = wave_sum(sum[t][r]);
      if (lane == 0 && row0 + r < m.rows)
        m.out[static_cast<size_t>(t) * m.rows + row0 + r] = float_to_bf16_bits(total);
    }
}

// ---- more than eight tokens: the matrix cores --------------------------------
// out[t, r] = sum_k w[r, k] x[t, k] as a 32-row x 32-token tile per wave on
// v_mfma_f32_32x32x16_bf16.  bf16 weights and tokens are exact operands.  FP8
// codes are exact in bf16 too, so FP8 weights are multiplied unscaled with the
// FP8 values of the quantized tokens, and each block of 128 contraction
// elements is scaled once by (weight block scale) x (token group scale):
// the same products as (w s_w)(x s_x), summed in FP32 in a different order.
// Lane (n, h) covers elements [64 h, 64 h + 64) of a 128-element block, for
// weight row n (A operand) and for token n (B operand).  The eight waves of a
// workgroup share a tile and take every eighth block; their partial tiles are
// added in wave order through LDS.

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float floatx16;

// Tokens as FP8 values in bf16 and their group scales [tokens, n / 128].  The
// values are written in the order the matrix-core kernel reads them, so that
// each of its loads is one contiguous KiB: [pass of 32 tokens][block of 128
// columns][step j][lane = token % 32 + 32 h][8], the lane's elements being
// columns 128 block + 64 h + 8 j .. + 7.
__global__ void __launch_bounds__(kGroup)
imported_token_fp8_kernel(const uint16_t* x, int n, uint16_t* values, float* scales) {
  __shared__ float largest[2];
  const int token = blockIdx.y, block = blockIdx.x, c = threadIdx.x;
  x += static_cast<size_t>(token) * n;
  const int i = block * kGroup + c;
  const float v = i < n ? bf16_bits_to_float(x[i]) : 0.0f;
  const float mine = wave_max(fabsf(v));
  if (threadIdx.x % 64 == 0) largest[threadIdx.x / 64] = mine;
  __syncthreads();
  const GroupQuantizer quantizer(fmaxf(largest[0], largest[1]));
  float value, unused;
  quantizer.round(v, 0.0f, value, unused);
  const size_t pass = token / 32;
  const int lane = token % 32 + 32 * (c / 64), step = (c % 64) / 8;
  if (i < n)
    values[(((pass * gridDim.x + block) * 8 + step) * 64 + lane) * 8 + c % 8] =
        float_to_bf16_bits(value);
  if (threadIdx.x == 0) scales[static_cast<size_t>(token) * gridDim.x + block] = quantizer.scale;
}

struct TileArgs {
  const void* weights = nullptr;
  const float* weight_scales = nullptr;  // FP8 only
  const uint16_t* tokens = nullptr;      // bf16 [count, cols]; FP8: one pass in operand order
  const float* token_scales = nullptr;   // FP8 only: [count, cols / 128]
  uint16_t* out = nullptr;               // [count, rows]
  int cols = 0, rows = 0, count = 0;     // count <= 32
};

template <bool HIGH>
__device__ inline uint32_t fp8_pair_to_bf16(uint32_t word) {
  const floatx2 v = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(word), HIGH);
  return (__float_as_uint(v.y) & 0xffff0000u) | (__float_as_uint(v.x) >> 16);
}

constexpr int kTileWaves = 8;  // waves that split a tile's contraction

// Several matrices in one launch, numbered as in MatVecArgs.
struct TileManyArgs {
  const void* weights[kManyMax];
  const float* weight_scales[kManyMax];
  uint16_t* out[kManyMax];
  int rows[kManyMax];
  int first_block[kManyMax + 1];
  int matrices = 0;
  const uint16_t* tokens = nullptr;
  const float* token_scales = nullptr;
  int cols = 0, count = 0;
};

// One tile: 32 rows of the matrix times up to 32 tokens, the contraction split
// over the workgroup's waves.  AHEAD (FP8 only): blocks of a wave whose weight
// loads are issued together.
template <bool FP8, int AHEAD>
__device__ __forceinline__ void imported_tile(const TileArgs& a, int tile,
                                              float (*partial)[16][64]) {
  const int lane = threadIdx.x % 64, n = lane % 32, h = lane / 32;
  const int wave = threadIdx.x / 64;
  const int row_base = tile * 32;
  const int row = min(row_base + n, a.rows - 1);   // rows and tokens past the end repeat
  const int token = min(n, a.count - 1);           // the last one and are not stored
  const int groups = a.cols / kGroup;
  const unsigned char* w = static_cast<const unsigned char*>(a.weights) +
                           (static_cast<size_t>(row) * a.cols + 64 * h) * (FP8 ? 1 : 2);
  // FP8: operand order, 1 KiB a step; otherwise the token's own row
  const uint16_t* x = FP8 ? a.tokens + lane * 8 : a.tokens + static_cast<size_t>(token) * a.cols + 64 * h;
  const float* block_scale =
      FP8 ? a.weight_scales + static_cast<size_t>(row_base / kGroup) * groups : nullptr;
  const float* group_scale = FP8 ? a.token_scales + static_cast<size_t>(token) * groups : nullptr;
  floatx16 total;
#pragma unroll
  for (int i = 0; i < 16; ++i) total[i] = 0.0f;
  if constexpr (FP8) {
    // A wave's weight rows are few bytes (64 a lane and block): the loads of
    // AHEAD of its blocks (all of them for widths up to 8192) are issued before
    // anything is waited for, so that the latency of HBM is paid once a batch
    // and not once a block; the tokens (L2 hits) follow one block ahead of the
    // products.  Blocks past the end repeat the last one (loads without
    // branches) and are not added.
    constexpr int kAhead = AHEAD;
    for (int g0 = wave; g0 < groups; g0 += kTileWaves * kAhead) {
      uint4 raw[kAhead][4];
#pragma unroll
      for (int b = 0; b < kAhead; ++b) {
        const int g = min(g0 + b * kTileWaves, groups - 1);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          raw[b][j] = *reinterpret_cast<const uint4*>(w + static_cast<size_t>(g) * kGroup + 16 * j);
      }
      uint4 xs[2][8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        xs[0][j] = *reinterpret_cast<const uint4*>(x + (static_cast<size_t>(g0) * 8 + j) * 512);
#pragma unroll
      for (int b = 0; b < kAhead; ++b) {
        const int g = g0 + b * kTileWaves;
        if (b + 1 < kAhead) {
          const int next = min(g + kTileWaves, groups - 1);
#pragma unroll
          for (int j = 0; j < 8; ++j)
            xs[(b + 1) % 2][j] =
                *reinterpret_cast<const uint4*>(x + (static_cast<size_t>(next) * 8 + j) * 512);
        }
        floatx16 acc;
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t lo = j % 2 == 0 ? raw[b][j / 2].x : raw[b][j / 2].z;
          const uint32_t hi = j % 2 == 0 ? raw[b][j / 2].y : raw[b][j / 2].w;
          const uint4 bits = make_uint4(fp8_pair_to_bf16<false>(lo), fp8_pair_to_bf16<true>(lo),
                                        fp8_pair_to_bf16<false>(hi), fp8_pair_to_bf16<true>(hi));
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, bits),
                                                        __builtin_bit_cast(bf16x8, xs[b % 2][j]),
                                                        acc, 0, 0, 0);
        }
        // a block past the end contributes nothing (its scale is read in range)
        const int in_range = min(g, groups - 1);
        const float scale = g < groups ? block_scale[in_range] * group_scale[in_range] : 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) total[i] += acc[i] * scale;
      }
    }
  } else {
    for (int g = wave; g < groups; g += kTileWaves) {
      uint4 xs[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) xs[j] = *reinterpret_cast<const uint4*>(x + g * kGroup + 8 * j);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint4 bits =
            *reinterpret_cast<const uint4*>(w + (static_cast<size_t>(g) * kGroup + 8 * j) * 2);
        total = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, bits),
                                                        __builtin_bit_cast(bf16x8, xs[j]), total,
                                                        0, 0, 0);
      }
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int i = 0; i < 16; ++i) partial[wave - 1][i][lane] = total[i];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int i = 0; i < 16; ++i)
#pragma unroll
    for (int w = 0; w < kTileWaves - 1; ++w) total[i] += partial[w][i][lane];
  // accumulator element 4 q + i = (row 8 q + 4 h + i, token n)
  if (n >= a.count) return;
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = row_base + 8 * q + 4 * h + i;
      if (r < a.rows)
        a.out[static_cast<size_t>(n) * a.rows + r] = float_to_bf16_bits(total[4 * q + i]);
    }
}

template <bool FP8, int AHEAD = 1>
__global__ void __launch_bounds__(64 * kTileWaves) imported_tile_kernel(TileManyArgs m) {
  __shared__ float partial[kTileWaves - 1][16][64];
  int which = 0;
  while (which + 1 < m.matrices && static_cast<int>(blockIdx.x) >= m.first_block[which + 1])
    ++which;
  TileArgs a;
  a.weights = m.weights[which];
  a.weight_scales = m.weight_scales[which];
  a.tokens = m.tokens;
  a.token_scales = m.token_scales;
  a.out = m.out[which];
  a.cols = m.cols;
  a.rows = m.rows[which];
  a.count = m.count;
  imported_tile<FP8, AHEAD>(a, blockIdx.x - m.first_block[which], partial);
}

// Picks AHEAD = blocks a wave owns, up to eight.
void launch_fp8_tiles(hipStream_t s, const TileManyArgs& t, int blocks) {
  const int groups = t.cols / kGroup;
  auto launch = [&](auto kernel) { kernel<<<blocks, 64 * kTileWaves, 0, s>>>(t); };
  switch (std::min(8, (groups + kTileWaves - 1) / kTileWaves)) {
    case 1: return launch(imported_tile_kernel<true, 1>);
    case 2: return launch(imported_tile_kernel<true, 2>);
    case 3: return launch(imported_tile_kernel<true, 3>);
    case 4: return launch(imported_tile_kernel<true, 4>);
    case 5: return launch(imported_tile_kernel<true, 5>);
    case 6: return launch(imported_tile_kernel<true, 6>);
    case 7: return launch(imported_tile_kernel<true, 7>);
    default: return launch(imported_tile_kernel<true, 8>);
  }
}

// The matrix-core path takes bf16 and FP8 weights whose rows are whole
// 128-element blocks; fewer than nine tokens are cheaper on the vector path.
bool tile_path(int storage, int tokens, int input_dim) {
  return storage != PLUTO_HIP_MATRIX_F32 && tokens > 8 && input_dim % kGroup == 0;
}

template <int STORAGE, int TOKENS, bool PREPARE>
void launch_matvec_batches(hipStream_t s, const MatVecArgs& a, unsigned blocks) {
  constexpr int kPiece = STORAGE == 0 ? 8 : STORAGE == 1 ? 4 : 16;
  const size_t lds = PREPARE ? static_cast<size_t>(a.cols) * 4 : 0;
  auto launch = [&](auto kernel) { kernel<<<blocks, 256, lds, s>>>(a); };
  const int steps = (a.cols / kPiece + 63) / 64;  // pieces a lane takes
  switch ((steps + (steps + 7) / 8 - 1) / ((steps + 7) / 8)) {
    case 1: return launch(imported_matvec_kernel<STORAGE, TOKENS, 1, PREPARE>);
    case 2: return launch(imported_matvec_kernel<STORAGE, TOKENS, 2, PREPARE>);
    case 3: return launch(imported_matvec_kernel<STORAGE, TOKENS, 3, PREPARE>);
    case 4: return launch(imported_matvec_kernel<STORAGE, TOKENS, 4, PREPARE>);
    case 5: return launch(imported_matvec_kernel<STORAGE, TOKENS, 5, PREPARE>);
    case 6: return launch(imported_matvec_kernel<STORAGE, TOKENS, 6, PREPARE>);
    case 7: return launch(imported_matvec_kernel<STORAGE, TOKENS, 7, PREPARE>);
    default: return launch(imported_matvec_kernel<STORAGE, TOKENS, 8, PREPARE>);
  }
}

// The vector path: up to eight tokens share a pass over the weights.  `token`
// holds the prepared tokens unless a.input is set.
template <int STORAGE>
void launch_matvec(hipStream_t s, MatVecArgs a, int tokens) {
  constexpr int kElementBytes = STORAGE == 0 ? 2 : STORAGE == 1 ? 4 : 1;
  const unsigned blocks = static_cast<unsigned>(a.first_block[a.matrices]);
  const bool whole = static_cast<size_t>(a.cols) * kElementBytes % 16 == 0;
  while (tokens > 0) {
    const int now = tokens >= 8 ? 8 : (tokens >= 4 ? 4 : (tokens >= 2 ? 2 : 1));
    if (!whole) {
      if (now == 8)
        imported_matvec_ragged_kernel<STORAGE, 8><<<blocks, 256, 0, s>>>(a);
      else if (now == 4)
        imported_matvec_ragged_kernel<STORAGE, 4><<<blocks, 256, 0, s>>>(a);
      else if (now == 2)
        imported_matvec_ragged_kernel<STORAGE, 2><<<blocks, 256, 0, s>>>(a);
      else
        imported_matvec_ragged_kernel<STORAGE, 1><<<blocks, 256, 0, s>>>(a);
    } else if (a.input != nullptr) {
      launch_matvec_batches<STORAGE, 1, true>(s, a, blocks);
    } else if (now == 8) {
      launch_matvec_batches<STORAGE, 8, false>(s, a, blocks);
    } else if (now == 4) {
      launch_matvec_batches<STORAGE, 4, false>(s, a, blocks);
    } else if (now == 2) {
      launch_matvec_batches<STORAGE, 2, false>(s, a, blocks);
    } else {
      launch_matvec_batches<STORAGE, 1, false>(s, a, blocks);
    }
    a.token += static_cast<size_t>(now) * a.cols;
    for (int i = 0; i < a.matrices; ++i) a.out[i] += static_cast<size_t>(now) * a.rows[i];
    tokens -= now;
  }
}

// One token of up to 16384 columns (64 KiB as FP32 in LDS) is prepared by the
// workgroups that use it.
bool matvec_prepares(int storage, const void* input, int tokens, int input_dim) {
  const int element_bytes =
      storage == PLUTO_HIP_MATRIX_BF16 ? 2 : storage == PLUTO_HIP_MATRIX_F32 ? 4 : 1;
  return tokens == 1 && input_dim <= 16384 && input_dim % 8 == 0 &&
         static_cast<size_t>(input_dim) * element_bytes % 16 == 0 &&
         (reinterpret_cast<uintptr_t>(input) & 15u) == 0;
}

}  // namespace

namespace {
size_t tile_values_bytes(int tokens, int input_dim) {
  const size_t padded = (static_cast<size_t>(tokens) + 31) / 32 * 32;
  return align_up(padded * input_dim * 2, 256);
}
}  // namespace

size_t dense_imported_workspace_bytes(int tokens, int input_dim) {
  // FP32 tokens (vector path), or their FP8 values in bf16, in whole passes of
  // 32 tokens, and the group scales (matrix-core path)
  const size_t vector_path = align_up(static_cast<size_t>(tokens) * input_dim * sizeof(float), 256);
  const size_t groups = (static_cast<size_t>(input_dim) + kGroup - 1) / kGroup;
  const size_t tile_path = tile_values_bytes(tokens, input_dim) + align_up(tokens * groups * 4, 256);
  return std::max(vector_path, tile_path) + 256;
}

// Matrices of one storage kind and input width applied to the same tokens: the
// tokens are prepared once, and every pass (up to 8 tokens on the vector path,
// 32 on the matrix cores) is one launch over all matrices.
int launch_dense_imported_forward(hipStream_t s, int storage, int matrices,
                                  const void* const* weights, const float* const* scales,
                                  const int* output_dims, const void* input, int tokens,
                                  int input_dim, void* const* outputs, void* workspace) {
  const bool fp8 = storage == PLUTO_HIP_MATRIX_FP8_E4M3;
  const dim3 groups(static_cast<unsigned>((input_dim + kGroup - 1) / kGroup),
                    static_cast<unsigned>(tokens));
  auto fill = [&](auto& args, auto& scale_list, int rows_per_block) {
    args.matrices = matrices;
    args.cols = input_dim;
    args.first_block[0] = 0;
    for (int i = 0; i < kManyMax; ++i) {
      const bool used = i < matrices;
      args.weights[i] = used ? weights[i] : nullptr;
      scale_list[i] = used && fp8 ? scales[i] : nullptr;
      args.out[i] = used ? static_cast<uint16_t*>(outputs[i]) : nullptr;
      args.rows[i] = used ? output_dims[i] : 0;
      args.first_block[i + 1] =
          args.first_block[i] + (used ? (output_dims[i] + rows_per_block - 1) / rows_per_block : 0);
    }
  };
  if (!tile_path(storage, tokens, input_dim)) {
    MatVecArgs a;
    fill(a, a.scales, 4 * kRowsPerWave);
    if (matvec_prepares(storage, input, tokens, input_dim)) {
      a.input = static_cast<const uint16_t*>(input);
    } else {
      float* token = static_cast<float*>(workspace);
      if (fp8)
        imported_token_kernel<true><<<groups, kGroup, 0, s>>>(static_cast<const uint16_t*>(input),
                                                              input_dim, token);
      else
        imported_token_kernel<false><<<groups, kGroup, 0, s>>>(static_cast<const uint16_t*>(input),
                                                               input_dim, token);
      a.token = token;
    }
    if (storage == PLUTO_HIP_MATRIX_BF16)
      launch_matvec<0>(s, a, tokens);
    else if (storage == PLUTO_HIP_MATRIX_F32)
      launch_matvec<1>(s, a, tokens);
    else
      launch_matvec<2>(s, a, tokens);
    return launch_status();
  }
  TileManyArgs t;
  fill(t, t.weight_scales, 32);
  t.tokens = static_cast<const uint16_t*>(input);
  if (fp8) {
    uint16_t* values = static_cast<uint16_t*>(workspace);
    float* token_scales = reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                                   tile_values_bytes(tokens, input_dim));
    imported_token_fp8_kernel<<<groups, kGroup, 0, s>>>(static_cast<const uint16_t*>(input),
                                                        input_dim, values, token_scales);
    t.tokens = values;
    t.token_scales = token_scales;
  }
  const int blocks = t.first_block[matrices];
  for (int done = 0; done < tokens; done += 32) {
    t.count = tokens - done < 32 ? tokens - done : 32;
    if (fp8)
      launch_fp8_tiles(s, t, blocks);
    else
      imported_tile_kernel<false><<<blocks, 64 * kTileWaves, 0, s>>>(t);
    t.tokens += static_cast<size_t>(32) * input_dim;
    if (fp8) t.token_scales += static_cast<size_t>(32) * (input_dim / kGroup);
    for (int i = 0; i < matrices; ++i) t.out[i] += static_cast<size_t>(32) * output_dims[i];
  }
  return launch_status();
}

}  // namespace pluto_hip

using namespace pluto_hip;

extern "C" {

static int validate_imported(int storage, const float* scales, int tokens, int input_dim,
                             int output_dim) {
  if (storage != PLUTO_HIP_MATRIX_BF16 && storage != PLUTO_HIP_MATRIX_F32 &&
      storage != PLUTO_HIP_MATRIX_FP8_E4M3)
    return PLUTO_HIP_EINVAL;
  // fully_connected.cc:271-275: dimensions in [1, 1048576]
  if (input_dim <= 0 || input_dim > PLUTO_HIP_IMPORTED_MAX_DIM || output_dim <= 0 ||
      output_dim > PLUTO_HIP_IMPORTED_MAX_DIM)
    return PLUTO_HIP_EINVAL;
  if (tokens <= 0 || tokens > PLUTO_HIP_IMPORTED_MAX_TOKENS) return PLUTO_HIP_EINVAL;
  // :279-281: only FP8 weights have block scales
  if ((storage == PLUTO_HIP_MATRIX_FP8_E4M3) != (scales != nullptr)) return PLUTO_HIP_EINVAL;
  return 0;
}

size_t pluto_hip_dense_imported_workspace_bytes(int input_dim) {
  return pluto_hip_dense_imported_batch_workspace_bytes(1, input_dim);
}

size_t pluto_hip_dense_imported_batch_workspace_bytes(int tokens, int input_dim) {
  if (input_dim <= 0 || input_dim > PLUTO_HIP_IMPORTED_MAX_DIM || tokens <= 0 ||
      tokens > PLUTO_HIP_IMPORTED_MAX_TOKENS)
    return 0;
  return dense_imported_workspace_bytes(tokens, input_dim);
}

int pluto_hip_dense_imported_forward(void* stream, int storage, const void* weights,
                                     const float* scales, const void* input, int input_dim,
                                     int output_dim, void* output, void* workspace,
                                     size_t workspace_bytes) {
  return pluto_hip_dense_imported_forward_batch(stream, storage, weights, scales, input, 1,
                                                input_dim, output_dim, output, workspace,
                                                workspace_bytes);
}

int pluto_hip_dense_imported_forward_batch(void* stream, int storage, const void* weights,
                                           const float* scales, const void* input, int tokens,
                                           int input_dim, int output_dim, void* output,
                                           void* workspace, size_t workspace_bytes) {
  const int status = validate_imported(storage, scales, tokens, input_dim, output_dim);
  if (status != 0) return status;
  if (!weights || !input || !output) return PLUTO_HIP_EINVAL;
  if (!workspace || workspace_bytes < dense_imported_workspace_bytes(tokens, input_dim))
    return PLUTO_HIP_EWORKSPACE;
  return launch_dense_imported_forward(static_cast<hipStream_t>(stream), storage, 1, &weights,
                                       &scales, &output_dim, input, tokens, input_dim, &output,
                                       workspace);
}

int pluto_hip_dense_imported_forward_many(void* stream, int storage, int matrices,
                                          const void* const* weights,
                                          const float* const* scales, const int* output_dims,
                                          const void* input, int tokens, int input_dim,
                                          void* const* outputs, void* workspace,
                                          size_t workspace_bytes) {
  if (matrices <= 0 || matrices > PLUTO_HIP_IMPORTED_MAX_MATRICES || !weights || !output_dims ||
      !outputs || !input)
    return PLUTO_HIP_EINVAL;
  const bool fp8 = storage == PLUTO_HIP_MATRIX_FP8_E4M3;
  if (fp8 && !scales) return PLUTO_HIP_EINVAL;
  long long tiles = 0;
  for (int i = 0; i < matrices; ++i) {
    const int status = validate_imported(storage, fp8 ? scales[i] : nullptr, tokens, input_dim,
                                         output_dims[i]);
    if (status != 0) return status;
    if (!fp8 && scales && scales[i]) return PLUTO_HIP_EINVAL;
    if (!weights[i] || !outputs[i]) return PLUTO_HIP_EINVAL;
    tiles += (output_dims[i] + 31) / 32;
  }
  if (tiles > 0x7fffffffLL) return PLUTO_HIP_EINVAL;
  if (!workspace || workspace_bytes < dense_imported_workspace_bytes(tokens, input_dim))
    return PLUTO_HIP_EWORKSPACE;
  return launch_dense_imported_forward(static_cast<hipStream_t>(stream), storage, matrices, weights,
                                       scales, output_dims, input, tokens, input_dim, outputs,
                                       workspace);
}

}  // extern "C"
