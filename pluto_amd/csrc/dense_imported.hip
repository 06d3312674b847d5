// FullyConnectedLayer, imported path (src/llm/layers/fully_connected.cc):
//   ImportedMatVecKernel          :40-68   y = bf16(W x), W output-major
//   QuantizeImportedInputKernel   :70-88   FP8 storage: x -> fp8(x / s) * s in
//                                          groups of 128, s = max|x| / 448
//   ImportedForward               :295-341 bf16 token -> fp32 -> (quantize) ->
//                                          mat-vec -> bf16
// One frozen checkpoint matrix [output_dim, input_dim] in bf16, fp32 or OCP
// FP8 E4M3 with FP32 scales [ceil(out/128), ceil(in/128)] times bf16 tokens.
// Byte-bound for few tokens: every weight is read once.  Three families of kernels:
//   vector        any storage, width and alignment; up to eight tokens a pass over the
//                 weights, FP32 arithmetic
//   few tokens    bf16 and FP8 weights of whole 128-element blocks, up to eight tokens:
//                 4 x 4 blocks on the matrix cores, tokens prepared by the workgroups
//   tiles         the same weights, more tokens: 16 x 16 blocks, 32 tokens a pass
// All sums are FP32.
#include <algorithm>
#include <type_traits>

#include "dense.h"
#include "imported_offsets.h"

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
// projection whose workgroups each prepare the token.  The largest magnitude comes as
// the bits of its bf16 value, of which a maximum keeps a NaN where that of floats loses
// it.  A group with a NaN or an infinity makes every sum it enters NaN (fp8(NaN) is NaN
// and fp8(v / inf) * inf is 0 * inf or NaN); its scale says so for all of its values,
// and the quotients, which the clamp keeps finite, need not be looked at.
struct GroupQuantizer {
  float scale, divisor, inverse;
  __device__ explicit GroupQuantizer(uint32_t largest) {
    scale = largest < 0x7f80u ? __uint_as_float(largest << 16) / 448.0f : __builtin_nanf("");
    divisor = fmaxf(scale, 1e-12f);
    inverse = 1.0f / divisor;
  }
  __device__ float quotient(float v) const {
    const float q = v * inverse;
    const float corrected = __builtin_fmaf(__builtin_fmaf(-q, divisor, v), inverse, q);
    return fminf(fmaxf(corrected, -448.0f), 448.0f);
  }
  // The FP8 code of the value nearest to the quotient.
  __device__ int code(float v) const {
    return __builtin_amdgcn_cvt_pk_fp8_f32(quotient(v), 0.0f, 0, false) & 0xff;
  }
  // The FP8 values (unscaled) nearest to the two quotients, as floats.
  __device__ void round(float first, float second, float& a, float& b) const {
    const int codes = __builtin_amdgcn_cvt_pk_fp8_f32(quotient(first), quotient(second), 0, false);
    const auto values = __builtin_amdgcn_cvt_pk_f32_fp8(codes, false);
    a = values[0];
    b = values[1];
  }
};

// Largest of `lanes` neighbouring lanes' values.
__device__ inline uint32_t lanes_max(uint32_t v, int lanes) {
  for (int offset = lanes / 2; offset > 0; offset >>= 1)
    v = max(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), offset, 64)));
  return v;
}

// token[i] = float(x[i]), for FP8 storage quantized per group of 128.
template <bool FP8>
__global__ void __launch_bounds__(kGroup)
imported_token_kernel(const uint16_t* x, int n, float* token) {
  __shared__ uint32_t largest[2];
  x += static_cast<size_t>(blockIdx.y) * n;      // one token per grid row
  token += static_cast<size_t>(blockIdx.y) * n;
  const int i = blockIdx.x * kGroup + threadIdx.x;
  const uint16_t bits = i < n ? x[i] : 0;
  const float v = bf16_bits_to_float(bits);
  if constexpr (!FP8) {
    if (i < n) token[i] = v;
  } else {
    const uint32_t mine = lanes_max(bits & 0x7fffu, 64);
    if (threadIdx.x % 64 == 0) largest[threadIdx.x / 64] = mine;
    __syncthreads();
    const GroupQuantizer quantizer(max(largest[0], largest[1]));
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

// Largest of sixteen neighbouring lanes' values.
__device__ inline uint32_t row_max(uint32_t v) {
  auto step = [&](auto control) {
    v = max(v, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), decltype(control)::value, 0xf, 0xf, true)));
  };
  step(std::integral_constant<int, 0xB1>());   // quad_perm 1, 0, 3, 2
  step(std::integral_constant<int, 0x4E>());   // quad_perm 2, 3, 0, 1
  step(std::integral_constant<int, 0x141>());  // row_half_mirror
  step(std::integral_constant<int, 0x140>());  // row_mirror
  return v;
}

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
// (Rows of whole 128-element blocks have kernels of their own, see below.)
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
        uint32_t largest = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          largest = max(largest, max(words[i] & 0x7fffu, words[i] >> 16 & 0x7fffu));
        const GroupQuantizer quantizer(lanes_max(largest, 16));
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

// ---- up to eight tokens of whole 128-element blocks ---------------------------
// v_mfma_f32_4x4x4_16b_bf16 multiplies sixteen independent pairs of 4 x 4 blocks: lane i of
// a block gives four elements of row i and of column i and finds element (j, i) of the
// product in register j.  Two kernels use it, both with persistent waves that own four
// rows of weights at a time, request a step's weights for the next four as soon as they
// have been multiplied, and find the tokens in LDS, put there by the workgroup while its
// first weights travel:
//   one      lanes are 64 pieces of sixteen bytes of one row, as in a mat-vec, and a lane
//            takes the product of its own piece and its own piece of the token: one of
//            sixteen products, but every weight is read in contiguous KiB
//   several  the rows of a block are four rows of weights, its columns four tokens: all
//            products are used, and a load instruction reads 256 bytes of each row
// A piece's product is the same in both, and both add up pieces in the order of a lane
// that takes every 64th and then of wave_sum, so that a token's results do not depend on
// how many there are.  FP8: codes are exact in bf16, and the sixteen elements of a piece lie
// in one block of scales, which multiply their sum (see below).
// On the vector units every token is another FMA a weight and another read of its values.
// Hot weights (in the memory-side cache), us for 1, 2, 4, 8 tokens in a captured graph, on
// the vector units and now: 5120 -> 16480 in FP8 19.2, 33.2, 50.3, 82.6 and 17.5, 20.1, 21.1,
// 24.4; 6144 -> 5120 in FP8 8.8, 13.9, 21.4, 35.7 and 7.7, 12.2, 13.6, 18.7; 5120 -> 16480 in
// bf16 26.9, 31.9, 47.9, 70.3 and 27.0, 27.5, 30.0, 30.9 (169 MB: 6.3 TB/s).
typedef __attribute__((ext_vector_type(4))) short shortx4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float floatx4;

constexpr int kFewTokens = 8, kFewWaves = 8;
constexpr int kFewColumns = 9216;  // 8 tokens as bf16 in LDS: 144 KiB

// Eight FP8 codes (the lower or the upper eight of sixteen) as bf16, exactly.
__device__ inline bf16x8 fp8_to_bf16(const uint4& codes, int part) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  const uint32_t word[2] = {part == 0 ? codes.x : codes.z, part == 0 ? codes.y : codes.w};
  bf16x8 out;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bf16x2 low = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(word[i], 1.0f, false);
    const bf16x2 high = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(word[i], 1.0f, true);
    out[4 * i] = low[0], out[4 * i + 1] = low[1], out[4 * i + 2] = high[0], out[4 * i + 3] = high[1];
  }
  return out;
}

// acc += the products of eight elements a lane: column i of a block's lanes is lane i's
// piece of a token, row i lane i's piece of a row, so that lane i finds the product of its
// own two pieces in register i.
__device__ inline floatx4 mma_few(uint4 weights, uint4 tokens, floatx4 acc) {
  typedef __attribute__((ext_vector_type(2))) uint32_t uint32x2;
  const uint32x2 w[2] = {{weights.x, weights.y}, {weights.z, weights.w}}, t[2] = {{tokens.x, tokens.y}, {tokens.z, tokens.w}};
#pragma unroll
  for (int i = 0; i < 2; ++i)
    acc = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(shortx4, w[i]), __builtin_bit_cast(shortx4, t[i]), acc,
                                                 0, 0, 0);
  return acc;
}

// Sums of N values over the 64 lanes: lanes l / (64 / N) end with value l, added in the
// order of wave_sum.
template <int N>
__device__ inline float sums_of(float (&v)[N]) {
  int offset = 32;
#pragma unroll
  for (int n = N; n > 1; n /= 2, offset /= 2) {
    const bool upper = threadIdx.x & offset;
#pragma unroll
    for (int i = 0; i < n / 2; ++i) {
      float low = v[i], high = v[i + n / 2];
      asm("" : "+v"(low), "+v"(high));  // values: the compiler would choose between addresses
      const float kept = upper ? high : low, sent = upper ? low : high;
      v[i] = kept + __shfl_xor(sent, offset, 64);
    }
  }
  float sum = v[0];
#pragma unroll
  for (; offset > 0; offset /= 2) sum += __shfl_xor(sum, offset, 64);
  return sum;
}

struct FewArgs {
  const void* weights[kManyMax];
  const float* scales[kManyMax];  // FP8 only
  uint16_t* out[kManyMax];        // [tokens, rows]
  int rows[kManyMax];
  int first_block[kManyMax + 1];  // of quadruples of rows
  int matrices = 0;
  const uint16_t* tokens = nullptr;  // bf16 [count, cols]
  int cols = 0, count = 0;
};

constexpr int kFewRows = 4;
constexpr int kFewThreads = 64 * kFewWaves;

// Four rows of a matrix.
struct FewUnit {
  int which, row;
  __amdgpu_buffer_rsrc_t weights;  // those past the end read zeros
  const float* scales;
};
template <bool FP8>
__device__ inline FewUnit few_unit(const FewArgs& m, int unit) {
  const int row_bytes = m.cols * (FP8 ? 1 : 2);
  FewUnit u;
  u.which = 0;
#pragma unroll
  for (int i = 1; i < kManyMax; ++i) u.which += unit >= m.first_block[i];  // unused ones start at the end
  u.row = (unit - m.first_block[u.which]) * kFewRows;
  u.weights = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<unsigned char*>(static_cast<const unsigned char*>(m.weights[u.which]) +
                                 static_cast<size_t>(u.row) * row_bytes),
      0, min(kFewRows, m.rows[u.which] - u.row) * row_bytes, 0x00020000);
  u.scales = FP8 ? m.scales[u.which] + static_cast<size_t>(u.row / kGroup) * (m.cols / kGroup) : nullptr;
  return u;
}

// The tokens' way into LDS, eight values a thread and load.
template <bool FP8, int TOKENS>
struct FewTokens {
  static constexpr int kPieces = TOKENS * kFewColumns / 8;
  static constexpr int kLoads = (kPieces + kFewThreads - 1) / kFewThreads;
  typedef uint4 Values[kLoads];
  static __device__ __forceinline__ void request(const FewArgs& m, Values& values) {
    const int pieces = m.count * (m.cols / 8);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      if (i * kFewThreads >= pieces) break;
      values[i] = reinterpret_cast<const uint4*>(
          m.tokens)[min(i * kFewThreads + static_cast<int>(threadIdx.x), pieces - 1)];
    }
  }
  // place(token, column, eight bf16 values), scale(token, group, scale)
  template <class Place, class Scale>
  static __device__ __forceinline__ void store(const FewArgs& m, const Values& values, Place place, Scale scale) {
    const int pieces = m.count * (m.cols / 8);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      if (i * kFewThreads >= pieces) break;
      const int piece = i * kFewThreads + static_cast<int>(threadIdx.x);
      const int token = TOKENS == 1 ? 0 : piece / (m.cols / 8), c = (piece - token * (m.cols / 8)) * 8;
      uint4 v = values[i];
      if constexpr (FP8) {
        const uint32_t words[4] = {v.x, v.y, v.z, v.w};
        uint32_t largest = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) largest = max(largest, max(words[e] & 0x7fffu, words[e] >> 16 & 0x7fffu));
        const GroupQuantizer quantizer(row_max(largest));  // sixteen lanes hold a group
        uint32_t rounded[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float first, second;
          quantizer.round(__uint_as_float(words[e] << 16), __uint_as_float(words[e] & 0xffff0000u), first, second);
          rounded[e] = (__float_as_uint(first) >> 16) | (__float_as_uint(second) & 0xffff0000u);  // exact in bf16
        }
        v = make_uint4(rounded[0], rounded[1], rounded[2], rounded[3]);
        if (piece < pieces && c % kGroup == 0) scale(token, c / kGroup, quantizer.scale);
      }
      if (piece >= pieces) break;  // whole groups of sixteen lanes
      place(token, c, v);
    }
  }
};

// Barrier for LDS: weights stay in flight.
__device__ inline void few_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// STEPS: of a panel, as many steps of 1 KiB of each row as the registers hold; rows longer
// than that are several panels.
template <bool FP8, int STEPS, int TOKENS>
__global__ void __launch_bounds__(kFewThreads)
imported_one_kernel(FewArgs m, int panels) {
  constexpr int R = kFewRows, kElements = FP8 ? 16 : 8;  // of a lane's piece
  constexpr int kStepColumns = 64 * kElements, kReads = kElements / 8;
  extern __shared__ uint4 few_lds[];  // [steps][TOKENS][kReads][64], then FP8: scales [steps][TOKENS][8]
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int steps = STEPS * panels, groups = m.cols / kGroup, units = m.first_block[m.matrices];
  const int row_bytes = m.cols * (FP8 ? 1 : 2);
  const bool whole = steps * kStepColumns == m.cols;
  float* token_scales = reinterpret_cast<float*>(few_lds + TOKENS * steps * kReads * 64);
  uint4 raw[STEPS][R];
  float scale[STEPS];
  auto request = [&](const FewUnit& u, int panel, int step) {
    const int at = (panel * STEPS + step) * 1024 + lane * 16;
    const bool exists = whole || at < row_bytes;
    if (FP8) scale[step] = u.scales[min(at / kGroup, groups - 1)];
#pragma unroll
    for (int r = 0; r < R; ++r)  // what lies past the end of a row reads zero
      raw[step][r] = __builtin_bit_cast(
          uint4, __builtin_amdgcn_raw_buffer_load_b128(u.weights, exists ? r * row_bytes + at : -1, 0, 0));
    if (FP8 && !whole) scale[step] = exists ? scale[step] : 0.0f;
  };

  // The tokens first (requests are answered in order), the weights behind them.
  using Tokens = FewTokens<FP8, TOKENS>;
  typename Tokens::Values values;
  Tokens::request(m, values);
  __builtin_amdgcn_sched_barrier(0);
  // a compute unit's waves lie far apart in the rows: where there are few, all of them
  // have work
  int unit = wave * gridDim.x + blockIdx.x;
  FewUnit now = few_unit<FP8>(m, min(unit, units - 1));
#pragma unroll
  for (int step = 0; step < STEPS; ++step) request(now, 0, step);
  __builtin_amdgcn_sched_barrier(0);
  if (!whole) {  // the pieces past the end, and their scales
    for (int i = threadIdx.x; i < TOKENS * steps * kReads * 64; i += kFewThreads) {
      const int step = i / (TOKENS * kReads * 64);
      if ((step * 64 + i % 64) * kElements >= m.cols) few_lds[i] = make_uint4(0, 0, 0, 0);
    }
    if (FP8)
      for (int i = threadIdx.x; i < TOKENS * steps * 8; i += kFewThreads)
        if (i / (TOKENS * 8) * 8 + i % 8 >= groups) token_scales[i] = 0.0f;
  }
  Tokens::store(
      m, values,
      [&](int token, int c, uint4 v) {
        const int at = c / kElements;  // the piece of the row
        few_lds[((at / 64 * TOKENS + token) * kReads + c % kElements / 8) * 64 + at % 64] = v;
      },
      [&](int token, int group, float s) { token_scales[(group / 8 * TOKENS + token) * 8 + group % 8] = s; });
  few_barrier();

  const bool odd = lane & 1, second = lane & 2;
  uint4 x[2][kReads];
  float x_scale[2] = {1.0f, 1.0f};
  // the lane's places in LDS move with the steps, a token's offset is part of the read
  constexpr int kStride = TOKENS * kReads * 64, kScaleStride = TOKENS * 8;
  const uint4* x_at = few_lds + lane;
  const float* scale_at = token_scales + lane / 8;
  auto read_token = [&](int slot, int t) {
#pragma unroll
    for (int k = 0; k < kReads; ++k) x[slot][k] = x_at[(t * kReads + k) * 64];
    if (FP8) x_scale[slot] = scale_at[t * 8];
  };
  read_token(0, 0);
  while (unit < units) {
    const int next_unit = unit + kFewWaves * gridDim.x;
    float sums[TOKENS * R];
#pragma unroll
    for (int i = 0; i < TOKENS * R; ++i) sums[i] = 0.0f;
    const int own_row = now.row, own_which = now.which;
    for (int panel = 0; panel < panels; ++panel) {
      const bool last = panel + 1 == panels;
      if (last) now = few_unit<FP8>(m, min(next_unit, units - 1));
      const int next_panel = last ? 0 : panel + 1;
#pragma unroll
      for (int step = 0; step < STEPS; ++step) {
        uint4 w[R][kReads];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int k = 0; k < kReads; ++k)
            w[r][k] = FP8 ? __builtin_bit_cast(uint4, fp8_to_bf16(raw[step][r], k)) : raw[step][r];
        const float weight_scale = FP8 ? scale[step] : 1.0f;
        __builtin_amdgcn_sched_barrier(0);
        request(now, next_panel, step);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < TOKENS; ++t) {
          // a token's values are read while the one before is multiplied
          const int slot = (step * TOKENS + t) % 2;
          if (t + 1 == TOKENS) {
            const bool first = step + 1 == STEPS && last;
            x_at = first ? few_lds + lane : x_at + kStride;
            scale_at = first ? token_scales + lane / 8 : scale_at + kScaleStride;
          }
          read_token(1 - slot, t + 1 < TOKENS ? t + 1 : 0);
          __builtin_amdgcn_sched_barrier(0);
          const float factor = weight_scale * x_scale[slot];
#pragma unroll
          for (int r = 0; r < R; ++r) {
            floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < kReads; ++k) acc = mma_few(w[r][k], x[slot][k], acc);
            const float low = odd ? acc[1] : acc[0], high = odd ? acc[3] : acc[2];
            const float product = second ? high : low;
            sums[t * R + r] = FP8 ? __builtin_fmaf(product, factor, sums[t * R + r]) : sums[t * R + r] + product;
            asm volatile("" : "+v"(sums[t * R + r]));  // here: the compiler would keep every acc to the end
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        // the last slot read is the first of the next panel
        if (STEPS * TOKENS % 2 == 1 && step + 1 == STEPS) {
#pragma unroll
          for (int k = 0; k < kReads; ++k) x[0][k] = x[1][k];
          x_scale[0] = x_scale[1];
        }
      }
    }
    const float sum = sums_of(sums);
    constexpr int kLanes = 64 / (TOKENS * R);
    const int index = lane / kLanes, token = index / R, row = own_row + index % R, rows = m.rows[own_which];
    if (lane % kLanes == 0 && row < rows && token < m.count)
      m.out[own_which][static_cast<size_t>(token) * rows + row] = float_to_bf16_bits(sum);
    unit = next_unit;
  }
}

// A step is 256 bytes of each of the four rows: lane 4 p + i holds piece p of row i and, of
// the tokens, piece p of token i (of tokens i and 4 + i where QUADS is two).  STEPS: of a
// panel, a multiple of four; step s belongs to the lanes 16 (s % 4) + p of the order of
// sums above.
template <bool FP8, int STEPS, int QUADS>
__global__ void __launch_bounds__(kFewThreads)
imported_several_kernel(FewArgs m, int panels) {
  static_assert(STEPS % 4 == 0);
  constexpr int kElements = FP8 ? 16 : 8;           // of a lane's piece
  constexpr int kStepColumns = 16 * kElements, kReads = kElements / 8;
  extern __shared__ uint4 few_lds[];  // [QUADS][steps][kReads][64], then FP8: scales [2 steps][8]
  const int lane = threadIdx.x % 64, i4 = lane % 4, block = lane / 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int steps = STEPS * panels, groups = m.cols / kGroup, units = m.first_block[m.matrices];
  const uint32_t row_bytes = m.cols * (FP8 ? 1 : 2);
  const bool whole = steps * kStepColumns == m.cols;
  float* token_scales = reinterpret_cast<float*>(few_lds + QUADS * steps * kReads * 64);
  const uint32_t row_start = i4 * row_bytes;
  uint4 raw[STEPS];
  auto request = [&](const FewUnit& u, int panel, int step) {
    const uint32_t at = (panel * STEPS + step) * 256;
    const SeveralPlace place = several_place(row_bytes, row_start, at, block);
    raw[step] = __builtin_bit_cast(
        uint4, __builtin_amdgcn_raw_buffer_load_b128(u.weights, place.lane, place.step, 0));
  };
  // a panel's scales: lane l holds that of group l of it
  auto request_scales = [&](const FewUnit& u, int panel) {
    const int group = panel * STEPS * 2 + lane;
    return FP8 ? u.scales[min(group, groups - 1)] : 0.0f;
  };

  using Tokens = FewTokens<FP8, 4 * QUADS>;
  typename Tokens::Values values;
  Tokens::request(m, values);
  __builtin_amdgcn_sched_barrier(0);
  int unit = wave * gridDim.x + blockIdx.x;
  FewUnit now = few_unit<FP8>(m, min(unit, units - 1));
  float scales = request_scales(now, 0);  // before the weights, which it would have to wait for
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int step = 0; step < STEPS; ++step) request(now, 0, step);
  __builtin_amdgcn_sched_barrier(0);
  if (!whole) {  // the pieces past the end, and their scales
    for (int i = threadIdx.x; i < QUADS * steps * kReads * 64; i += kFewThreads) {
      const int step = i / (kReads * 64) % steps;
      if ((step * 16 + i % 64 / 4) * kElements >= m.cols) few_lds[i] = make_uint4(0, 0, 0, 0);
    }
    if (FP8)
      for (int i = threadIdx.x; i < 2 * steps * kFewTokens; i += kFewThreads)
        if (i / kFewTokens >= groups) token_scales[i] = 0.0f;
  }
  Tokens::store(
      m, values,
      [&](int token, int c, uint4 v) {
        const int at = c / kElements;  // the piece of the row
        few_lds[((token / 4 * steps + at / 16) * kReads + c % kElements / 8) * 64 + at % 16 * 4 + token % 4] = v;
      },
      [&](int token, int group, float s) { token_scales[group * kFewTokens + token] = s; });
  few_barrier();

  // a step's tokens are read a step ahead
  uint4 t[2][QUADS][kReads];
  float token_scale[2][QUADS];
  auto read_tokens = [&](int slot, int panel, int step) {
    const int at = panel * STEPS + step;
#pragma unroll
    for (int j = 0; j < QUADS; ++j) {
#pragma unroll
      for (int k = 0; k < kReads; ++k) t[slot][j][k] = few_lds[((j * steps + at) * kReads + k) * 64 + lane];
      if (FP8) token_scale[slot][j] = token_scales[(2 * at + block / 8) * kFewTokens + 4 * j + i4];
    }
  };
  read_tokens(0, 0, 0);
  while (unit < units) {
    const int next_unit = unit + kFewWaves * gridDim.x;
    floatx4 total[QUADS][4];
#pragma unroll
    for (int j = 0; j < QUADS; ++j)
#pragma unroll
      for (int u = 0; u < 4; ++u) total[j][u] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const FewUnit own = now;
    for (int panel = 0; panel < panels; ++panel) {
      const bool last = panel + 1 == panels;
      if (last) now = few_unit<FP8>(m, min(next_unit, units - 1));
      const int next_panel = last ? 0 : panel + 1;
      const float next_scales = request_scales(now, next_panel);
#pragma unroll
      for (int step = 0; step < STEPS; ++step) {
        const int slot = step % 2, u = step % 4;
        read_tokens(1 - slot, step + 1 < STEPS ? panel : next_panel, step + 1 < STEPS ? step + 1 : 0);
        __builtin_amdgcn_sched_barrier(0);
        uint4 w[kReads];
#pragma unroll
        for (int k = 0; k < kReads; ++k)
          w[k] = FP8 ? __builtin_bit_cast(uint4, fp8_to_bf16(raw[step], k)) : raw[step];
        // pieces 0 .. 7 of a step of FP8 are one group, 8 .. 15 the next
        float weight_scale = 1.0f;
        if constexpr (FP8) {
          const float low = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(scales), 2 * step));
          const float high = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(scales), 2 * step + 1));
          weight_scale = block < 8 ? low : high;
          if (!whole) weight_scale = ((panel * STEPS + step) * 16 + block) * kElements < m.cols ? weight_scale : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < QUADS; ++j) {
          floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int k = 0; k < kReads; ++k) acc = mma_few(w[k], t[slot][j][k], acc);
          const float factor = FP8 ? weight_scale * token_scale[slot][j] : 1.0f;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            total[j][u][i] = FP8 ? __builtin_fmaf(acc[i], factor, total[j][u][i]) : total[j][u][i] + acc[i];
        }
        __builtin_amdgcn_sched_barrier(0);
        request(now, next_panel, step);
        __builtin_amdgcn_sched_barrier(0);
      }
      scales = next_scales;
    }
    // over the pieces; lanes 16 k + i end with row k of token i
    const int row = own.row + lane / 16;
#pragma unroll
    for (int j = 0; j < QUADS; ++j) {
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        v[i] = (total[j][0][i] + total[j][2][i]) + (total[j][1][i] + total[j][3][i]);
      const bool upper = lane & 32, odd = lane & 16;
      const float a = (upper ? v[2] : v[0]) + __shfl_xor(upper ? v[0] : v[2], 32, 64);
      const float b = (upper ? v[3] : v[1]) + __shfl_xor(upper ? v[1] : v[3], 32, 64);
      float sum = (odd ? b : a) + __shfl_xor(odd ? a : b, 16, 64);
      sum += __shfl_xor(sum, 8, 64);
      sum += __shfl_xor(sum, 4, 64);
      const int token = 4 * j + i4, rows = m.rows[own.which];
      if (lane % 16 < 4 && row < rows && token < m.count)
        m.out[own.which][static_cast<size_t>(token) * rows + row] = float_to_bf16_bits(sum);
    }
    unit = next_unit;
  }
}

// ---- more than eight tokens: the matrix cores --------------------------------
// out[t, r] = sum_k w[r, k] x[t, k], 16 or 32 rows x 16 or 32 tokens a tile.  bf16 weights and
// tokens are exact operands of v_mfma_f32_16x16x32_bf16.  FP8 codes are exact in bf16
// too, so FP8 weights are multiplied unscaled with the FP8 values of the quantized
// tokens on v_mfma_f32_16x16x32_bf16, and each block of 128 contraction elements is
// scaled once by (weight block scale) x (token group scale): the same products as (w
// s_w)(x s_x), summed in FP32 in a different order.  (v_mfma_f32_16x16x32_fp8_fp8 would
// take the codes as they are, but sums with fewer bits: 0.1 % of the results of 1024
// columns were more than a bf16 rounding off.)  The eight waves of a workgroup share a
// tile and take every eighth block; their partial tiles are added in wave order
// through LDS.

// Tokens as FP8 codes and their group scales [tokens, n / 128].  The codes are written
// in the order the matrix-core kernel reads them, so that each of its loads is one
// contiguous KiB: [pass of 32 tokens][block of 128 columns][half of the block][half of
// the tokens][lane = token % 16 + 16 q][16], the lane's elements being columns 128
// block + 64 half + 16 q .. + 15.
__global__ void __launch_bounds__(kGroup)
imported_token_fp8_kernel(const uint16_t* x, int n, unsigned char* codes, float* scales) {
  __shared__ uint32_t largest[2];
  const int token = blockIdx.y, block = blockIdx.x, c = threadIdx.x;
  x += static_cast<size_t>(token) * n;
  const uint16_t bits = x[block * kGroup + c];  // n is a multiple of 128
  const float v = bf16_bits_to_float(bits);
  const uint32_t mine = lanes_max(bits & 0x7fffu, 64);
  if (threadIdx.x % 64 == 0) largest[threadIdx.x / 64] = mine;
  __syncthreads();
  const GroupQuantizer quantizer(max(largest[0], largest[1]));
  const size_t piece = ((static_cast<size_t>(token / 32) * gridDim.x + block) * 2 + c / 64) * 2 + token % 32 / 16;
  codes[(piece * 64 + token % 16 + c % 64 / 16 * 16) * 16 + c % 16] =
      static_cast<unsigned char>(quantizer.code(v));
  if (threadIdx.x == 0) scales[static_cast<size_t>(token) * gridDim.x + block] = quantizer.scale;
}

constexpr int kTileWaves = 8;  // waves that split a tile's contraction

// Several matrices in one launch, numbered as in MatVecArgs.
struct TileManyArgs {
  const void* weights[kManyMax];
  const float* weight_scales[kManyMax];
  uint16_t* out[kManyMax];
  int rows[kManyMax];
  int first_block[kManyMax + 1];
  int matrices = 0, tile_rows = 16;
  const void* tokens = nullptr;         // bf16 [count, cols]; FP8: one pass in operand order
  const float* token_scales = nullptr;  // FP8 only: [count, cols / 128]
  int cols = 0, count = 0;              // count <= 32
};

// The matrix of a tile and its first row there.
struct TilePlace {
  int which, row;
};
__device__ inline TilePlace tile_place(const TileManyArgs& m, int tile) {
  int which = 0;
  while (which + 1 < m.matrices && tile >= m.first_block[which + 1]) ++which;
  return {which, (tile - m.first_block[which]) * m.tile_rows};
}

// The partial tiles of the waves (`elements` of 64 lanes each) added in wave order; element
// e belongs to rows .. of the store.  Requests stay in flight across the barrier.
template <int ELEMENTS, typename Store>
__device__ inline void add_waves(float (&partial)[kTileWaves][ELEMENTS][64], const float (&own)[ELEMENTS], int wave,
                                 int lane, Store store) {
#pragma unroll
  for (int i = 0; i < ELEMENTS; ++i) partial[wave][i][lane] = own[i];
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
  for (int k = 0; k < (ELEMENTS + kTileWaves - 1) / kTileWaves; ++k) {
    const int e = k * kTileWaves + wave;
    if (ELEMENTS % kTileWaves != 0 && e >= ELEMENTS) break;
    float sum = partial[0][e][lane];
#pragma unroll
    for (int w = 1; w < kTileWaves; ++w) sum += partial[w][e][lane];
    store(e, sum);
  }
}

// bf16, the same walk over tiles of 16 rows as below.  Lane (q, n16) covers elements 32 s +
// 8 q .. + 7 of each block of weight row n16 and of tokens n16 (and 16 + n16): operands of
// v_mfma_f32_16x16x32_bf16 as they lie in memory, four lanes a 64-byte piece of a row.
// Bound by the addresses of those pieces, sixteen rows a load.  5120 -> 16480, 9, 16 and 32
// tokens (at any element: global memory takes wide accesses unaligned): 62.7, 75.1 and 98.3
// us with one tile of 32 rows a workgroup, 36.7, 37.7 and 75.5
// so (32 tokens take twice the registers, so that the rows travel in several passes).
template <int BLOCKS, int TOKEN_PARTS, bool ONE_PASS>
__global__ void __launch_bounds__(64 * kTileWaves)
imported_tile_bf16_kernel(TileManyArgs m, int passes) {
  if constexpr (ONE_PASS) passes = 1;
  constexpr int STEPS = kGroup / 32;
  __shared__ float partial[2][kTileWaves][4 * TOKEN_PARTS][64];
  const int lane = threadIdx.x % 64, n = lane % 16, q = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int groups = m.cols / kGroup, tiles = m.first_block[m.matrices];
  auto block_of = [&](int pass, int b) { return wave + kTileWaves * (pass * BLOCKS + b); };
  const uint32_t lane_at = (static_cast<uint32_t>(n) * m.cols + 8 * q) * 2;
  uint4 raw[BLOCKS][STEPS], x[BLOCKS][STEPS][TOKEN_PARTS];
  auto request = [&](const __amdgpu_buffer_rsrc_t& rows, int pass, int b) {
    const uint32_t at = min(block_of(pass, b), groups - 1) * (kGroup * 2);
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
      raw[b][s] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rows, lane_at, at + 64 * s, 0));
  };
  // rows past the end read zeros
  auto rows_of = [&](int tile) {
    const TilePlace place = tile_place(m, tile);
    const size_t first = static_cast<size_t>(place.row) * m.cols * 2;
    const int rows = min(m.tile_rows, m.rows[place.which] - place.row);
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<unsigned char*>(static_cast<const unsigned char*>(m.weights[place.which]) + first), 0,
        rows * m.cols * 2, 0x00020000);
  };
  auto load_tokens = [&](int pass) {
#pragma unroll
    for (int j = 0; j < TOKEN_PARTS; ++j) {
      // tokens past the end repeat the last one and are not stored
      const uint16_t* token = static_cast<const uint16_t*>(m.tokens) +
                              static_cast<size_t>(min(16 * j + n, m.count - 1)) * m.cols + 8 * q;
#pragma unroll
      for (int b = 0; b < BLOCKS; ++b) {
        const int g = block_of(pass, b);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
          x[b][s][j] = *reinterpret_cast<const uint4*>(token + min(g, groups - 1) * kGroup + 32 * s);
          if (g >= groups) x[b][s][j] = make_uint4(0, 0, 0, 0);  // a block past the end
        }
      }
    }
  };
  load_tokens(0);
  __builtin_amdgcn_sched_barrier(0);
  {
    const __amdgpu_buffer_rsrc_t rows = rows_of(blockIdx.x);
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) request(rows, 0, b);
  }
  __builtin_amdgcn_sched_barrier(0);
  int buffer = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, buffer ^= 1) {
    const TilePlace place = tile_place(m, tile);
    const int rows = m.rows[place.which];
    floatx4 total[TOKEN_PARTS];
#pragma unroll
    for (int j = 0; j < TOKEN_PARTS; ++j) total[j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int pass = 0; pass < passes; ++pass) {
      if (!ONE_PASS && (pass > 0 || tile != static_cast<int>(blockIdx.x))) load_tokens(pass);
      const int next_pass = pass + 1 < passes ? pass + 1 : 0;
      const int next_tile = next_pass > 0 ? tile : min(tile + static_cast<int>(gridDim.x), tiles - 1);
      const __amdgpu_buffer_rsrc_t next_rows = rows_of(next_tile);
#pragma unroll
      for (int b = 0; b < BLOCKS; ++b) {
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
#pragma unroll
          for (int j = 0; j < TOKEN_PARTS; ++j)
            total[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, raw[b][s]),
                                                               __builtin_bit_cast(bf16x8, x[b][s][j]), total[j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        request(next_rows, next_pass, b);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    float own[4 * TOKEN_PARTS];
#pragma unroll
    for (int i = 0; i < 4 * TOKEN_PARTS; ++i) own[i] = total[i / 4][i % 4];
    // element e is row 4 q + e % 4, token 16 (e / 4) + n
    add_waves(partial[buffer], own, wave, lane, [&](int e, float sum) {
      const int row = place.row + 4 * q + e % 4, token = 16 * (e / 4) + n;
      if (row < min(rows, place.row + m.tile_rows) && token < m.count)
        m.out[place.which][static_cast<size_t>(token) * rows + row] = float_to_bf16_bits(sum);
    });
  }
}

// FP8: one workgroup a compute unit that walks over tiles.  A wave's blocks of the
// contraction are the same in every tile: their tokens stay in registers, and each
// block of weights is requested for the next tile as soon as its registers have been
// multiplied, so that HBM never waits for a tile's products and sums (one tile a
// workgroup, the compute units went idle between 516 tiles of 5120 columns: 37 us
// against 25).  BLOCKS: a wave's blocks, as many as its registers hold; wider matrices
// take several passes a tile, for each of which the tokens are loaded again.  Lane (q,
// n16) covers elements 16 q .. + 15 of each half block of weight row n16 of each of
// PARTS 16-row parts (A operands) and of tokens n16 and 16 + n16 (B operands).
// TOKEN_PARTS: one for up to sixteen tokens.
template <int BLOCKS, int PARTS, int TOKEN_PARTS, bool ONE_PASS>
__global__ void __launch_bounds__(64 * kTileWaves)
imported_tile_fp8_kernel(TileManyArgs m, int passes) {
  if constexpr (ONE_PASS) passes = 1;
  __shared__ float partial[2][kTileWaves][4 * TOKEN_PARTS * PARTS][64];
  const int lane = threadIdx.x % 64, n = lane % 16, q = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int groups = m.cols / kGroup, tiles = m.first_block[m.matrices];
  auto block_of = [&](int pass, int b) { return wave + kTileWaves * (pass * BLOCKS + b); };
  const uint32_t lane_at = static_cast<uint32_t>(n) * m.cols + 16 * q;
  uint4 raw[BLOCKS][2][PARTS], x[BLOCKS][2][TOKEN_PARTS];  // [block][half][rows or tokens]
  float group_scale[BLOCKS][TOKEN_PARTS];
  // rows past the end read zeros
  auto request = [&](const __amdgpu_buffer_rsrc_t& rows, int pass, int b) {
    const uint32_t at = min(block_of(pass, b), groups - 1) * kGroup;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int t = 0; t < PARTS; ++t)
        raw[b][half][t] = __builtin_bit_cast(
            uint4, __builtin_amdgcn_raw_buffer_load_b128(rows, lane_at + 16 * t * m.cols, at + 64 * half, 0));
  };
  auto rows_of = [&](int tile) {
    const TilePlace place = tile_place(m, tile);
    const size_t first = static_cast<size_t>(place.row) * m.cols;
    const int rows = min(m.tile_rows, m.rows[place.which] - place.row);
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<unsigned char*>(static_cast<const unsigned char*>(m.weights[place.which]) + first), 0,
        rows * m.cols, 0x00020000);
  };
  auto load_tokens = [&](int pass) {
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) {
      const int g = min(block_of(pass, b), groups - 1);
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int t = 0; t < TOKEN_PARTS; ++t)
          x[b][half][t] = static_cast<const uint4*>(m.tokens)[((g * 2 + half) * 2 + t) * 64 + lane];
#pragma unroll
      for (int t = 0; t < TOKEN_PARTS; ++t)  // tokens past the end are not stored
        group_scale[b][t] = m.token_scales[static_cast<size_t>(min(16 * t + n, m.count - 1)) * groups + g];
    }
  };
  load_tokens(0);
  {
    const __amdgpu_buffer_rsrc_t rows = rows_of(blockIdx.x);
#pragma unroll
    for (int b = 0; b < BLOCKS; ++b) request(rows, 0, b);
  }
  __builtin_amdgcn_sched_barrier(0);
  int buffer = 0;
  for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x, buffer ^= 1) {
    const TilePlace place = tile_place(m, tile);
    const int rows = m.rows[place.which];
    const float* block_scale = m.weight_scales[place.which] + static_cast<size_t>(place.row / kGroup) * groups;
    // a tile of other than 16 rows may reach into the next 128, which have scales of their own
    const int own_rows = kGroup - place.row % kGroup;
    const bool crosses = PARTS > 1 && own_rows < min(m.tile_rows, rows - place.row);
    floatx4 total[PARTS][TOKEN_PARTS];
#pragma unroll
    for (int i = 0; i < PARTS; ++i)
#pragma unroll
      for (int j = 0; j < TOKEN_PARTS; ++j) total[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int pass = 0; pass < passes; ++pass) {
      if (!ONE_PASS && (pass > 0 || tile != static_cast<int>(blockIdx.x))) load_tokens(pass);
      const int next_pass = pass + 1 < passes ? pass + 1 : 0;
      const int next_tile = next_pass > 0 ? tile : min(tile + static_cast<int>(gridDim.x), tiles - 1);
      const __amdgpu_buffer_rsrc_t next_rows = rows_of(next_tile);
#pragma unroll
      for (int b = 0; b < BLOCKS; ++b) {
        // a block past the end contributes nothing (its scale is read in range)
        const int g = block_of(pass, b);
        const float weight_scale = g < groups ? block_scale[min(g, groups - 1)] : 0.0f;
        const float next_scale =
            PARTS > 1 && g < groups ? block_scale[min(g, groups - 1) + (crosses ? groups : 0)] : 0.0f;
        floatx4 acc[PARTS][TOKEN_PARTS];
#pragma unroll
        for (int i = 0; i < PARTS; ++i)
#pragma unroll
          for (int j = 0; j < TOKEN_PARTS; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        // the tokens are converted here for every tile: converted once they would take
        // twice the registers, which the compiler does not see
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int j = 0; j < TOKEN_PARTS; ++j)
            asm volatile("" : "+v"(x[b][half][j].x), "+v"(x[b][half][j].y), "+v"(x[b][half][j].z),
                              "+v"(x[b][half][j].w));
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int part = 0; part < 2; ++part) {
            bf16x8 w[PARTS], t[TOKEN_PARTS];
#pragma unroll
            for (int i = 0; i < PARTS; ++i) w[i] = fp8_to_bf16(raw[b][half][i], part);
#pragma unroll
            for (int j = 0; j < TOKEN_PARTS; ++j) t[j] = fp8_to_bf16(x[b][half][j], part);
#pragma unroll
            for (int i = 0; i < PARTS; ++i)
#pragma unroll
              for (int j = 0; j < TOKEN_PARTS; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i], t[j], acc[i][j], 0, 0, 0);
          }
        __builtin_amdgcn_sched_barrier(0);
        request(next_rows, next_pass, b);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < PARTS; ++i)
#pragma unroll
          for (int j = 0; j < TOKEN_PARTS; ++j) {
            if (PARTS == 1 || !crosses) {
              total[i][j] += acc[i][j] * (weight_scale * group_scale[b][j]);
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                total[i][j][e] +=
                    acc[i][j][e] * ((16 * i + 4 * q + e < own_rows ? weight_scale : next_scale) * group_scale[b][j]);
            }
          }
      }
    }
    constexpr int kElements = 4 * TOKEN_PARTS * PARTS;
    float own[kElements];
#pragma unroll
    for (int i = 0; i < kElements; ++i) own[i] = total[i / (4 * TOKEN_PARTS)][i / 4 % TOKEN_PARTS][i % 4];
    // element e is row 16 (e / (4 TOKEN_PARTS)) + 4 q + e % 4, token 16 (e / 4 % TOKEN_PARTS) + n
    add_waves(partial[buffer], own, wave, lane, [&](int e, float sum) {
      const int row = place.row + 16 * (e / (4 * TOKEN_PARTS)) + 4 * q + e % 4;
      const int token = 16 * (e / 4 % TOKEN_PARTS) + n;
      if (row < min(rows, place.row + m.tile_rows) && token < m.count)
        m.out[place.which][static_cast<size_t>(token) * rows + row] = float_to_bf16_bits(sum);
    });
  }
}

// The rows of a tile: at most 16 PARTS, and as few as leave the longest list of a workgroup as
// long as with that many, so that all lists have about as many bytes: 5120 -> 16480 is 1030 tiles
// of 16 rows, five for six workgroups and four for the others, or 1269 of 13.  bf16, 14 tokens:
// 5120 -> 16480 36.8 -> 32.2 us, 6144 -> 5120 (320 tiles, 512 so) 22.8 -> 17.7; 30 tokens 77.4 ->
// 72.1, 37.2 -> 32.8.  FP8 6144 -> 5120 (160 tiles of 32 rows, 256 of 20), 11 tokens 11.9 -> 10.6
// us, 32 13.6 -> 12.5.  FP8 tiles of 16 rows are bound by their conversions as much as by their
// bytes (5120 -> 16480 in tiles of 13, 11 tokens 21.1 -> 20.7, 32 23.4 -> 24.4): they stay whole.
// Fewer than 256 whole tiles become tiles of few rows on all compute units.  The tokens, which
// each loads then, come from the L2 and at the same time; whole and so, 9 / 16 / 32 tokens: bf16
// 5120 -> 256 12.7 / 14.4 / 18.0 and 6.6 / 8.2 / 12.9 us (1 row), 768 13.0 / 14.7 / 18.5 and 8.0 /
// 9.4 / 14.1 (3), 1024 13.1 / 14.8 / 18.6 and 8.5 / 10.1 / 14.6 (4), 768 -> 768 4.1 / 4.1 / 4.7 and
// 3.1 / 3.2 / 3.9; FP8 5120 -> 1024 13.6 / 14.3 / 17.0 and 9.3 / 9.8 / 12.6 (4), 768 -> 768 6.3 / 6.4
// / 6.7 and 5.2 / 5.3 / 5.8.  Fewer rows still make second tiles: 5120 -> 1024 bf16 in tiles of 2
// 9.3 / 10.8 / 24.6.
long long tiles_of(int matrices, const int* rows, int tile_rows) {
  long long tiles = 0;
  for (int i = 0; i < matrices; ++i) tiles += (rows[i] + tile_rows - 1) / tile_rows;
  return tiles;
}
int balanced_rows(int matrices, const int* rows, int most) {
  const long long turns = (tiles_of(matrices, rows, most) + 255) / 256;
  int tile_rows = most;
  while (tile_rows > 1 && tiles_of(matrices, rows, tile_rows - 1) <= 256 * turns) --tile_rows;
  return tile_rows;
}

// Where every compute unit walks over several tiles they have up to 16 rows (shorter ends: 516 x
// 32 rows of 5120 columns 27.4 us in tiles of 32 rows, 24.7 in tiles of 16).  Fewer have
// up to 32, for the tokens, as many bytes as a tile's weights, are loaded for one tile only
// (160 x 32 rows of 6144 columns: 14.3 us, 15.5 in tiles of 16).
int fp8_parts(int matrices, const int* rows) { return tiles_of(matrices, rows, 32) >= 256 ? 1 : 2; }

template <int PARTS, int TOKEN_PARTS>
void launch_fp8_tiles(hipStream_t s, const TileManyArgs& t) {
  const int groups = t.cols / kGroup, owned = (groups + kTileWaves - 1) / kTileWaves;  // blocks of a wave
  const unsigned grid = std::min(t.first_block[t.matrices], 256);
  int passes = 1;
  auto launch = [&](auto kernel) { kernel<<<grid, 64 * kTileWaves, 0, s>>>(t, passes); };
  // As many blocks as a wave's registers hold for the next tile; where a workgroup has one
  // tile of 32 rows and nothing to request ahead for, as few as its first request: the
  // products begin when that has arrived.  6144 -> 5120, 9 and 32 tokens: 16.7 us in one
  // pass of six blocks, 14.1 in two of three and 17.2; 5120 -> 5120 14.1 and 18.6 in one
  // pass of five, 13.6 and 16.9.
  constexpr int kMost = PARTS == 2 ? 4 : 6;
  if (owned > kMost) {
    passes = (owned + 3) / 4;
    return (owned + passes - 1) / passes == 3 ? launch(imported_tile_fp8_kernel<3, PARTS, TOKEN_PARTS, false>)
                                              : launch(imported_tile_fp8_kernel<4, PARTS, TOKEN_PARTS, false>);
  }
  switch (owned) {
    case 1: return launch(imported_tile_fp8_kernel<1, PARTS, TOKEN_PARTS, true>);
    case 2: return launch(imported_tile_fp8_kernel<2, PARTS, TOKEN_PARTS, true>);
    case 3: return launch(imported_tile_fp8_kernel<3, PARTS, TOKEN_PARTS, true>);
    case 4: return launch(imported_tile_fp8_kernel<4, PARTS, TOKEN_PARTS, true>);
    case 5: if constexpr (kMost == 6) return launch(imported_tile_fp8_kernel<5, PARTS, TOKEN_PARTS, true>);
    default: if constexpr (kMost == 6) return launch(imported_tile_fp8_kernel<6, PARTS, TOKEN_PARTS, true>);
  }
}

template <int TOKEN_PARTS>
void launch_bf16_tiles(hipStream_t s, const TileManyArgs& t) {
  const int owned = (t.cols / kGroup + kTileWaves - 1) / kTileWaves;
  const unsigned grid = std::min(t.first_block[t.matrices], 256);
  int passes = 1;
  auto launch = [&](auto kernel) { kernel<<<grid, 64 * kTileWaves, 0, s>>>(t, passes); };
  constexpr int kMost = TOKEN_PARTS == 1 ? 6 : 3;
  if (owned > kMost) {
    passes = (owned + kMost - 1) / kMost;
    return launch(imported_tile_bf16_kernel<kMost, TOKEN_PARTS, false>);
  }
  switch (owned) {
    case 1: return launch(imported_tile_bf16_kernel<1, TOKEN_PARTS, true>);
    case 2: return launch(imported_tile_bf16_kernel<2, TOKEN_PARTS, true>);
    case 3: return launch(imported_tile_bf16_kernel<3, TOKEN_PARTS, true>);
    case 4: if constexpr (kMost == 6) return launch(imported_tile_bf16_kernel<4, TOKEN_PARTS, true>);
    case 5: if constexpr (kMost == 6) return launch(imported_tile_bf16_kernel<5, TOKEN_PARTS, true>);
    default: if constexpr (kMost == 6) return launch(imported_tile_bf16_kernel<6, TOKEN_PARTS, true>);
  }
}

template <bool FP8, int TOKENS>
void launch_one(hipStream_t s, const FewArgs& a) {
  const int steps = (a.cols + (FP8 ? 1023 : 511)) / (FP8 ? 1024 : 512);
  const int panels = (steps + 5) / 6, of_panel = (steps + panels - 1) / panels;
  const unsigned grid = std::min(a.first_block[a.matrices], 256);
  const size_t lds = static_cast<size_t>(TOKENS) * of_panel * panels * (FP8 ? 2048 + 32 : 1024);
  auto launch = [&](auto kernel) { kernel<<<grid, kFewThreads, lds, s>>>(a, panels); };
  switch (of_panel) {
    case 1: return launch(imported_one_kernel<FP8, 1, TOKENS>);
    case 2: return launch(imported_one_kernel<FP8, 2, TOKENS>);
    case 3: return launch(imported_one_kernel<FP8, 3, TOKENS>);
    case 4: return launch(imported_one_kernel<FP8, 4, TOKENS>);
    case 5: return launch(imported_one_kernel<FP8, 5, TOKENS>);
    default: return launch(imported_one_kernel<FP8, 6, TOKENS>);
  }
}
template <bool FP8, int QUADS>
void launch_several(hipStream_t s, const FewArgs& a) {
  const int steps = (a.cols + (FP8 ? 255 : 127)) / (FP8 ? 256 : 128);
  int panels = (steps + 23) / 24;
  auto panel_steps = [&] { return ((steps + panels - 1) / panels + 3) / 4 * 4; };
  // what the panels hold past the end must not take more LDS than the widest rows do
  while (panel_steps() * panels > kFewColumns / (FP8 ? 256 : 128)) ++panels;
  const int of_panel = panel_steps();
  const unsigned grid = std::min(a.first_block[a.matrices], 256);
  const size_t lds = static_cast<size_t>(of_panel) * panels * (QUADS * (FP8 ? 2048 : 1024) + (FP8 ? 2 * kFewTokens * 4 : 0));
  auto launch = [&](auto kernel) { kernel<<<grid, kFewThreads, lds, s>>>(a, panels); };
  switch (of_panel) {
    case 4: return launch(imported_several_kernel<FP8, 4, QUADS>);
    case 8: return launch(imported_several_kernel<FP8, 8, QUADS>);
    case 12: return launch(imported_several_kernel<FP8, 12, QUADS>);
    case 16: return launch(imported_several_kernel<FP8, 16, QUADS>);
    case 20: return launch(imported_several_kernel<FP8, 20, QUADS>);
    default: return launch(imported_several_kernel<FP8, 24, QUADS>);
  }
}
// Two tokens of FP8 weights take 21.7 us in the kernel for one and 19.6 in the other (5120
// -> 16480), two of bf16 weights, which need no conversion, 27.6 and 29.0.
template <bool FP8>
void launch_few(hipStream_t s, const FewArgs& a) {
  if (a.count == 1) return launch_one<FP8, 1>(s, a);
  if constexpr (!FP8)
    if (a.count == 2) return launch_one<FP8, 2>(s, a);
  return a.count <= 4 ? launch_several<FP8, 1>(s, a) : launch_several<FP8, 2>(s, a);
}

// The matrix cores take bf16 and FP8 weights whose rows are whole 128-element blocks: up
// to eight tokens of rows that fit in LDS, and more.  Everything else, and up to eight
// tokens of longer rows, is the vector path's; what up to eight tokens take does not
// depend on their number, so that a token's results do not either.  Weights are read by
// buffer loads, which take whole words; up to eight tokens in pieces of sixteen bytes, more
// at any element.
bool matrix_cores(int storage, int matrices, const void* const* weights, const void* input, int tokens, int input_dim) {
  if (storage == PLUTO_HIP_MATRIX_F32 || input_dim % kGroup != 0) return false;
  auto aligned = [](const void* p, unsigned bytes) { return reinterpret_cast<uintptr_t>(p) % bytes == 0; };
  for (int i = 0; i < matrices; ++i)
    if (!aligned(weights[i], 4)) return false;
  if (tokens <= kFewTokens && input_dim > kFewColumns) return false;
  return tokens > kFewTokens || aligned(input, 16);
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
  return align_up(padded * input_dim, 256);
}
}  // namespace

size_t dense_imported_workspace_bytes(int tokens, int input_dim) {
  // FP32 tokens (vector path), or their FP8 codes, in whole passes of 32 tokens, and
  // the group scales (matrix-core path)
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
  const bool matrix = matrix_cores(storage, matrices, weights, input, tokens, input_dim);
  if (matrix && tokens <= kFewTokens) {
    FewArgs a;
    fill(a, a.scales, 4);
    a.tokens = static_cast<const uint16_t*>(input);
    a.count = tokens;
    fp8 ? launch_few<true>(s, a) : launch_few<false>(s, a);
    return launch_status();
  }
  if (!matrix) {
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
  const int parts = fp8 ? fp8_parts(matrices, output_dims) : 1;
  t.tile_rows = fp8 && parts == 1 ? 16 : balanced_rows(matrices, output_dims, 16 * parts);
  fill(t, t.weight_scales, t.tile_rows);
  const unsigned char* token_bytes = static_cast<const unsigned char*>(input);
  if (fp8) {
    unsigned char* codes = static_cast<unsigned char*>(workspace);
    float* token_scales = reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                                   tile_values_bytes(tokens, input_dim));
    imported_token_fp8_kernel<<<groups, kGroup, 0, s>>>(static_cast<const uint16_t*>(input),
                                                        input_dim, codes, token_scales);
    token_bytes = codes;
    t.token_scales = token_scales;
  }
  for (int done = 0; done < tokens; done += 32) {
    t.count = tokens - done < 32 ? tokens - done : 32;
    t.tokens = token_bytes + static_cast<size_t>(done) * input_dim * (fp8 ? 1 : 2);
    if (!fp8)
      t.count <= 16 ? launch_bf16_tiles<1>(s, t) : launch_bf16_tiles<2>(s, t);
    else if (parts == 1)
      t.count <= 16 ? launch_fp8_tiles<1, 1>(s, t) : launch_fp8_tiles<1, 2>(s, t);
    else
      t.count <= 16 ? launch_fp8_tiles<2, 1>(s, t) : launch_fp8_tiles<2, 2>(s, t);
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
