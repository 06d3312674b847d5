// Gated delta-net: chunked linear-attention scan for gfx950, plus the
// token-by-token recurrence.
//
// Recurrence (RecurrenceForward, src/llm/layers/sequence_delta_net.cc:55-102;
// DeltaRecurrenceKernel, src/llm/layers/util/cached_attention_ops.cc:205-251),
// per head, state S in R^{dk x dv}:
//     S <- a_t S;  d_t = b_t (v_t - S^T k_t);  S <- S + k_t d_t^T;  o_t = S^T q_t
// with a_t = exp(g_t) and b_t = beta_t.
//
// Chunked form used here (C = 64 tokens, c_i = g_1 + .. + g_i inside a chunk,
// S0 = state entering the chunk, K and Q with their normalisation and scale):
//     A[i,j]  = b_i exp(c_i - c_j) (k_i . k_j)        for j <  i
//     T  = (I + A)^-1
//     D  = T diag(b) (V - diag(exp(c)) K S0)          (the d_t of the chunk)
//     O  = diag(exp(c)) Q S0 + (M o Q K^T) D,   M[i,j] = exp(c_i - c_j), j <= i
//     S  = exp(c_C) S0 + (diag(exp(c_C - c)) K)^T D
// Only differences c_i - c_j <= 0 are exponentiated, so nothing overflows.
// Every diagonal factor is applied in FP32 to matrix-core results, so the
// products themselves take the raw bf16 rows of K and Q as they lie in memory.
//
// Kernel 1 (gdn_chunk_prepare, one workgroup per chunk, fully parallel): the
// two Gram matrices on the matrix cores from the raw bf16 inputs, T by a block
// forward substitution on the matrix cores, and 14 KiB per chunk written out:
// T and M o (Q K^T) as bf16 matrix-core operands, and the per-token factors.  For the layer
// it also makes the rows of K, Q and V from the layer's inputs.
// Kernel 2 (gdn_chunk_scan, one workgroup per (sequence, head, 16 state
// columns)): walks the chunks with v_mfma_f32_16x16x32_bf16, the state in FP32
// accumulator registers of one wave, a second wave computing the outputs, two
// more streaming each chunk's 14 KiB and its raw K, Q and V rows into LDS.
// State columns are independent, which is what gives the sequential part
// 8 x batch x heads way parallelism.
#include "gdn.h"
#include "gdn_activation.h"

#include <type_traits>

namespace pluto_hip {
namespace {

constexpr int C = 64;     // tokens per chunk
constexpr int DK = 128;   // key width of the chunked path
constexpr int DV = 128;   // value width of the chunked path
constexpr int SLICES = DV / 16;

typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4_t;
typedef __attribute__((ext_vector_type(4))) short shortx4;

__device__ inline bf16x8 bits_to_bf16x8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// Contraction-slot order of an operand that multiplies two stacked 16x16
// accumulator tiles: slot (hq, e) of 32-block kb is element
// 32*kb + 16*(e/4) + 4*hq + e%4 (see file header of mfma_tile.h for the
// 32x32 analogue).

__device__ inline floatx4 mfma16(bf16x8 a, bf16x8 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Two stacked accumulator tiles as the B operand of a 32-deep product.
__device__ inline bf16x8 tiles_to_operand(const floatx4& lo, const floatx4& hi) {
  bf16x8 out;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    out[e] = static_cast<__bf16>(lo[e]);
    out[4 + e] = static_cast<__bf16>(hi[e]);
  }
  return out;
}

// Two stacked accumulator tiles as a pair of B (or, read the other way, A)
// operands whose sum carries about 16 mantissa bits: hi = bf16(v), lo =
// bf16(v - hi).
__device__ inline void split_operand(const floatx4& first, const floatx4& second, bf16x8& hi,
                                     bf16x8& lo) {
  uint32_t high[4], low[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const floatx4& from = i < 2 ? first : second;
    const float v0 = from[2 * (i % 2)], v1 = from[2 * (i % 2) + 1];
    high[i] = pack_bf16(v0, v1);
    low[i] = pack_bf16(v0 - __uint_as_float(high[i] << 16), v1 - __uint_as_float(high[i] & 0xffff0000u));
  }
  hi = bits_to_bf16x8(make_uint4(high[0], high[1], high[2], high[3]));
  lo = bits_to_bf16x8(make_uint4(low[0], low[1], low[2], low[3]));
}

// One tile so, and the product of two of sixteen contraction elements.
struct SplitTile {
  shortx4 hi, lo;
};
__device__ inline SplitTile split_operand(const floatx4& v) {
  const uint32_t high[2] = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
  uint32_t low[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
    low[i] = pack_bf16(v[2 * i] - __uint_as_float(high[i] << 16), v[2 * i + 1] - __uint_as_float(high[i] & 0xffff0000u));
  return {__builtin_bit_cast(shortx4, make_uint2(high[0], high[1])), __builtin_bit_cast(shortx4, make_uint2(low[0], low[1]))};
}
__device__ inline floatx4 product16(const SplitTile& a, const SplitTile& b, floatx4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.hi, b.hi, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.lo, b.hi, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.hi, b.lo, c, 0, 0, 0);
}

// Sum of the squares of eight or four bf16 numbers, and of sixteen neighbouring lanes' values.
template <int WORDS>
__device__ inline float squares(const uint32_t (&words)[WORDS]) {
  float even = 0.0f, odd = 0.0f;
#pragma unroll
  for (int i = 0; i < WORDS; ++i) {
    const float low = __uint_as_float(words[i] << 16), high = __uint_as_float(words[i] & 0xffff0000u);
    even += low * low;
    odd += high * high;
  }
  return even + odd;
}
__device__ inline float squares(const uint4& v) { return squares<4>({v.x, v.y, v.z, v.w}); }
__device__ inline float squares(const uint2& v) { return squares<2>({v.x, v.y}); }
__device__ inline float row_sum(float v) {
  auto step = [&](auto control) {
    v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), decltype(control)::value, 0xf, 0xf, true));
  };
  step(std::integral_constant<int, 0xB1>());   // quad_perm 1, 0, 3, 2
  step(std::integral_constant<int, 0x4E>());   // quad_perm 2, 3, 0, 1
  step(std::integral_constant<int, 0x141>());  // row_half_mirror
  step(std::integral_constant<int, 0x140>());  // row_mirror
  return v;
}

// Once the Gram matrices are done the rows of K and Q make room for A, and A in turn for
// the finished inverse.  The kernel is a chain of short, barrier-separated phases and lives on
// occupancy: 35 KiB for one head, four workgroups of four waves a compute unit; 80 KiB for
// three, two of twelve waves.
template <int HEADS>
struct ChunkSmem {
  using Rows = uint16_t[C][DK + 8];     // raw K or Q rows (bf16)
  using Square = float[C][C + 4];       // strictly lower triangular A (FP32) and the blocks of its solve
  using Operand = uint16_t[C][C + 8];   // (I + A)^-1; M o (Q K^T) with all factors: bf16
  static_assert(sizeof(Rows) == sizeof(Square) && sizeof(Operand) <= sizeof(Rows));
  unsigned char blocks[HEADS < 2 ? 2 : HEADS][sizeof(Rows)];
  unsigned char products[HEADS < 2 ? 0 : HEADS][sizeof(Operand)];
  float cum[HEADS][C];      // inclusive cumulative log decay
  float beta[HEADS][C];
  float inv_k[C];           // 1/|k| (or 1)
  float q_factor[C];        // q_scale / |q| (or q_scale)
  __device__ Rows& k() { return *reinterpret_cast<Rows*>(blocks[0]); }
  __device__ Rows& q() { return *reinterpret_cast<Rows*>(blocks[1]); }
  __device__ Square& a(int head) { return *reinterpret_cast<Square*>(blocks[head]); }
  __device__ Operand& t(int head) { return *reinterpret_cast<Operand*>(blocks[head]); }
  __device__ Operand& a2(int head) {
    return *reinterpret_cast<Operand*>(HEADS < 2 ? blocks[1] : products[head]);
  }
};

// One head's 128 channels of a chunk through the convolution and SiLU, four channels and
// eight rows a thread of 256.  The rows go to memory, where the sequential kernel reads
// them, and to LDS with zeros beyond the sequence, the sums of their squares to `use_square`.
template <typename UseSquare>
__device__ inline void convolve_head(const uint16_t* in, const float* weight, uint16_t* out, long long stride,
                                     int t0, int valid, int tid, bool store, uint16_t (*rows)[DK + 8],
                                     UseSquare&& use_square) {
  constexpr int kRun = 8;
  const int c0 = 4 * (tid % 32), first = tid / 32 * kRun;
  uint2 raw[kRun + 3];
#pragma unroll
  for (int j = 0; j < kRun + 3; ++j) {
    // rows behind the sequence are not used, those before it are zero
    raw[j] = *reinterpret_cast<const uint2*>(in + min(max(first + j - 3, -t0), valid - 1) * stride + c0);
    if (j < 3 && t0 + first + j < 3) raw[j] = make_uint2(0, 0);
  }
  float w[4][4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float4 v = *reinterpret_cast<const float4*>(weight + 4 * (c0 + e));
    w[e][0] = v.x, w[e][1] = v.y, w[e][2] = v.z, w[e][3] = v.w;
  }
#pragma unroll
  for (int j = 0; j < kRun; ++j) {
    float x[4][4];  // channel, tap
#pragma unroll
    for (int tap = 0; tap < 4; ++tap) {
      x[0][tap] = __uint_as_float(raw[j + tap].x << 16), x[1][tap] = __uint_as_float(raw[j + tap].x & 0xffff0000u);
      x[2][tap] = __uint_as_float(raw[j + tap].y << 16), x[3][tap] = __uint_as_float(raw[j + tap].y & 0xffff0000u);
    }
    const int row = first + j;
    const uint2 post = make_uint2(convolved_pair(x[0], w[0], x[1], w[1]), convolved_pair(x[2], w[2], x[3], w[3]));
    if (store && row < valid) *reinterpret_cast<uint2*>(out + row * stride + c0) = post;
    if (rows) {
      *reinterpret_cast<uint2*>(&rows[row][c0]) = post;
      float square = row_sum(squares(post));
      square += __shfl_xor(square, 16, 64);
      if (tid % 32 == 0) use_square(row, row < valid ? square : 0.0f);
    }
  }
  if (rows && valid < C) {
#pragma unroll
    for (int j = 0; j < kRun; ++j)
      if (first + j >= valid) *reinterpret_cast<uint2*>(&rows[first + j][c0]) = make_uint2(0, 0);
  }
}

// A workgroup of 256 HEADS threads prepares a chunk for HEADS value heads of one key head.
// LAYER: from the layer's inputs; the rows of K and Q are convolved once for the heads of a
// workgroup, and every head's V on the way.  8191 tokens of 16/48 heads: 112 us for 427 MB;
// as passes of their own the convolution took 67, the gates 5 and the preparation 63, of 16/16
// heads 57 and 43 + 5 + 27.  Vector instructions are 60 % of it (42 million; 50 with an
// activation that carries a division's correction, factors rounded one by one, zeros in the
// operands of the solve and every wave substituting its own block).
template <int HEADS, bool LAYER>
__global__ void __launch_bounds__(256 * HEADS)
__attribute__((amdgpu_waves_per_eu(HEADS == 3 ? 6 : 4)))
gdn_chunk_prepare(GdnArgs a, GdnLayerInputs layer) {
  __shared__ __attribute__((aligned(16))) ChunkSmem<HEADS> sm;
  const int local = HEADS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / 256);  // of the workgroup's heads
  const int tid = threadIdx.x % 256, wave = tid / 64, lane = tid % 64;
  const int chunks = (a.length + C - 1) / C;
  const int group = a.value_heads / a.key_heads, parts = group / HEADS;
  // chunks of a head after each other; LAYER: heads of a chunk, neighbouring columns of its rows
  const int unit = LAYER ? blockIdx.x % (a.key_heads * parts) : blockIdx.x / chunks % a.value_heads;
  const int chunk = LAYER ? blockIdx.x / (a.key_heads * parts) % chunks : blockIdx.x % chunks;
  const int seq = blockIdx.x / (a.key_heads * parts) / chunks;
  const int head = HEADS * unit + local, key_head = unit / parts, part = unit % parts;
  const int bh = seq * a.value_heads + head;
  const int t0 = chunk * C;
  const int valid = min(C, a.length - t0);
  const long long token0 = static_cast<long long>(seq) * a.length + t0;
  uint16_t(&sm_k)[C][DK + 8] = sm.k(), (&sm_q)[C][DK + 8] = sm.q();
  float(&sm_a)[C][C + 4] = sm.a(local);
  uint16_t(&sm_t)[C][C + 8] = sm.t(local), (&sm_a2)[C][C + 8] = sm.a2(local);
  float(&sm_cum)[C] = sm.cum[local], (&sm_beta)[C] = sm.beta[local];

  // sequence_delta_net.cc:84-85: x * rsqrt(sum(x^2) + 1e-6)
  auto use_k = [&](int row, float square) { sm.inv_k[row] = a.normalize_qk ? rsqrtf(square + 1e-6f) : 1.0f; };
  auto use_q = [&](int row, float square) {
    sm.q_factor[row] = a.normalize_qk ? a.q_scale * rsqrtf(square + 1e-6f) : a.q_scale;
  };
  // the convolution of a head's columns; `which` is the place of its rows in GdnArgs
  auto convolve = [&](const uint16_t* which, int column, int thread, bool store, uint16_t (*rows)[DK + 8], auto&& use) {
    const int at = static_cast<int>(which - a.q) + column;
    convolve_head(layer.qkv + token0 * a.q_token_stride + at, layer.conv_weight + 4 * at,
                  const_cast<uint16_t*>(a.q) + token0 * a.q_token_stride + at, a.q_token_stride, t0, valid, thread,
                  store, rows, use);
  };
  // sixteen rows of a head's V
  auto convolve_v = [&](int of, int quarter) {
    convolve(a.v, (head - local + of) * DV, 64 * quarter + lane, true, nullptr, [](int, float) {});
  };
  if constexpr (LAYER) {
    // the first head's waves have K, the second's Q, the third's its V
    if (local == 0) convolve(a.k, key_head * DK, tid, part == 0, sm_k, use_k);
    if (local == (HEADS == 1 ? 0 : 1)) convolve(a.q, key_head * DK, tid, part == 0, sm_q, use_q);
    if (local == 2) convolve_v(2, wave);
  } else {
    // ---- stage K and Q rows (16-byte pieces), zero beyond the sequence --------
    // Sixteen lanes hold a row and add up its squares as it arrives (read back from LDS
    // one channel at a time, four lanes a row: 83 us at 8191 tokens of 48 heads, 78 so).
    constexpr int kLoads = C * (DK / 8) / 256;
    const int c8 = tid % (DK / 8);
    uint4 kb[kLoads], qb[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int row = i * (256 / (DK / 8)) + tid / (DK / 8);
      kb[i] = qb[i] = make_uint4(0, 0, 0, 0);
      if (row < valid) {
        kb[i] = *reinterpret_cast<const uint4*>(a.k + (token0 + row) * a.k_token_stride + key_head * DK + 8 * c8);
        qb[i] = *reinterpret_cast<const uint4*>(a.q + (token0 + row) * a.q_token_stride + key_head * DK + 8 * c8);
      }
    }
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int row = i * (256 / (DK / 8)) + tid / (DK / 8);
      *reinterpret_cast<uint4*>(&sm_k[row][8 * c8]) = kb[i];
      *reinterpret_cast<uint4*>(&sm_q[row][8 * c8]) = qb[i];
      const float kk = row_sum(squares(kb[i])), qq = row_sum(squares(qb[i]));
      if (c8 == 0) use_k(row, kk), use_q(row, qq);
    }
  }
  if (wave == (local + 1) % 4) {
    float g = 0.0f, b = 0.0f;
    if (lane < valid) {
      const long long at = (token0 + lane) * a.value_heads + head;
      if constexpr (LAYER) {
        g = log_decay_of(bf16_bits_to_float(layer.a[at]) + layer.dt_bias[head], layer.a_log[head]);
        b = round_to_bf16(beta_of(bf16_bits_to_float(layer.b[at])));
      } else {
        g = a.log_decay[at];
        b = a.beta[at];
      }
    }
    // inclusive prefix sum over the 64 lanes
    for (int offset = 1; offset < 64; offset <<= 1) {
      const float up = __shfl_up(g, offset, 64);
      if (lane >= offset) g += up;
    }
    sm_cum[lane] = g;
    sm_beta[lane] = b;
  }
  __syncthreads();

  // ---- Gram matrices on the matrix cores: wave (ti, tj) owns a 32x32 tile --
  {
    const int ti = wave / 2, tj = wave % 2;
    const int h = lane / 32, n = lane % 32;
    float a2v[16], av[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      a2v[i] = 0.0f;
      av[i] = 0.0f;
    }
    if (tj <= ti) {
      floatx16 gk, gq;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        gk[i] = 0.0f;
        gq[i] = 0.0f;
      }
#pragma unroll
      for (int ks = 0; ks < DK / 16; ++ks) {
        const bf16x8 kr = bits_to_bf16x8(*reinterpret_cast<const uint4*>(&sm_k[32 * ti + n][16 * ks + 8 * h]));
        const bf16x8 qr = bits_to_bf16x8(*reinterpret_cast<const uint4*>(&sm_q[32 * ti + n][16 * ks + 8 * h]));
        const bf16x8 kc = bits_to_bf16x8(*reinterpret_cast<const uint4*>(&sm_k[32 * tj + n][16 * ks + 8 * h]));
        gk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kr, kc, gk, 0, 0, 0);
        gq = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qr, kc, gq, 0, 0, 0);
      }
      const int col = 32 * tj + n;  // token j
      const float cum_j = sm_cum[col], inv_kj = sm.inv_k[col];
      // four rows a register quad; values are chosen, not branched around: a branch with
      // a read of LDS in it for each of 32 elements took 7400 of the kernel's 21000 cycles
      // (78 us; 70 so)
      const int above = col - 32 * ti - 4 * h;  // of the lane's first row
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row0 = 32 * ti + 8 * j + 4 * h;  // token i
        const floatx4 cum = *reinterpret_cast<const floatx4*>(&sm_cum[row0]),
                      beta = *reinterpret_cast<const floatx4*>(&sm_beta[row0]),
                      inv_k = *reinterpret_cast<const floatx4*>(&sm.inv_k[row0]),
                      q_factor = *reinterpret_cast<const floatx4*>(&sm.q_factor[row0]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float decay = __expf(fminf(cum[e] - cum_j, 0.0f)) * inv_kj;
          float k = beta[e] * inv_k[e] * decay * gk[4 * j + e], q = decay * q_factor[e] * gq[4 * j + e];
          asm("" : "+v"(k), "+v"(q));
          av[4 * j + e] = above < 8 * j + e ? k : 0.0f;
          a2v[4 * j + e] = above <= 8 * j + e ? q : 0.0f;
        }
      }
    }
    __syncthreads();  // nobody reads the rows of K and Q any more
#pragma unroll
    for (int i = 0; i < 16; i += 2) {
      const int row = 32 * ti + 8 * (i / 4) + 4 * h + (i % 4);
      sm_a[row][32 * tj + n] = av[i];  // the tile above the diagonal is zero
      sm_a[row + 1][32 * tj + n] = av[i + 1];
      const uint32_t pair = pack_bf16(a2v[i], a2v[i + 1]);
      sm_a2[row][32 * tj + n] = static_cast<uint16_t>(pair);
      sm_a2[row + 1][32 * tj + n] = static_cast<uint16_t>(pair >> 16);
    }
  }
  __syncthreads();

  // ---- T = (I + A)^-1 by blocks of 16 rows on the matrix cores.  With T_b the
  // inverse of diagonal block b of I + A, block row b of the solve X of
  // (I + A) X = R is  X_b = T_b (R_b - sum_{k<b} A_bk X_k).
  // Every factor enters as a sum of two bf16 numbers (value = hi + lo, products
  // hi*hi + lo*hi + hi*lo), which keeps the result to about 2^-16 relative.
  //
  // T_b by forward substitution on the identity: sixteen lanes a block, lane = column, by
  // one wave of a head's (of each head's another, which the hardware deals to another SIMD);
  // the result replaces the diagonal block of A, which nothing else reads.  The other waves
  // convolve the V that are left meanwhile (behind the kernel's end, all of them: 112 us at
  // 8191 tokens of 16/48 heads).
  if (wave == local) {
    const int base = 16 * (lane / 16), column = lane % 16;
    float t[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float acc = (i == column) ? 1.0f : 0.0f;
#pragma unroll
      for (int j4 = 0; j4 < (i + 3) / 4; ++j4) {
        const float4 row = *reinterpret_cast<const float4*>(&sm_a[base + i][base + 4 * j4]);
        acc -= row.x * t[4 * j4];
        if (4 * j4 + 1 < i) acc -= row.y * t[4 * j4 + 1];
        if (4 * j4 + 2 < i) acc -= row.z * t[4 * j4 + 2];
        if (4 * j4 + 3 < i) acc -= row.w * t[4 * j4 + 3];
      }
      t[i] = acc;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) sm_a[base + i][base + column] = t[i];
  }
  if constexpr (LAYER) {
    const int turn = wave == local ? 3 * HEADS + local : 3 * local + wave - (wave > local);
    if (turn < 4 * min(HEADS, 2)) convolve_v(turn / 4, turn % 4);
  }
  __syncthreads();

  // Wave w solves columns 16 w .. 16 w + 15 of X for R = I: X_b = 0 above the
  // diagonal block, X_w = T_w, and the blocks below follow from the recurrence.
  // x[b] is the 16x16 tile of block row b in accumulator order: lane (hq, m)
  // holds rows 16 b + 4 hq + r of column 16 w + m.
  {
    const int hq = lane / 16, m = lane % 16;
    const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    floatx4 x[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      x[b] = zero;
      if (b < wave) continue;  // uniform over the wave
      if (b == wave) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[b][e] = sm_a[16 * b + 4 * hq + e][16 * b + m];
        continue;
      }
      // r = sum [A_b,k0 | A_b,k1] [X_k0; X_k1]: contraction slot (hq, e) is row
      // 4 hq + e % 4 of block k0 (e < 4) or k1
      floatx4 r = zero;
#pragma unroll
      for (int k0 = 0; k0 < b; k0 += 2) {
        if (k0 + 1 < wave) continue;  // both blocks of X are zero
        const floatx4 first = *reinterpret_cast<const floatx4*>(&sm_a[16 * b + m][16 * k0 + 4 * hq]);
        if (k0 + 1 == b) {
          r = product16(split_operand(first), split_operand(x[k0]), r);
        } else {
          const floatx4 second = *reinterpret_cast<const floatx4*>(&sm_a[16 * b + m][16 * k0 + 16 + 4 * hq]);
          bf16x8 a_hi, a_lo, b_hi, b_lo;
          split_operand(first, second, a_hi, a_lo);
          split_operand(x[k0], x[k0 + 1], b_hi, b_lo);
          r = mfma16(a_hi, b_hi, r);
          r = mfma16(a_lo, b_hi, r);
          r = mfma16(a_hi, b_lo, r);
        }
      }
      // X_b = -T_b r
      const floatx4 t = *reinterpret_cast<const floatx4*>(&sm_a[16 * b + m][16 * b + 4 * hq]);
      x[b] = -product16(split_operand(t), split_operand(r), zero);
    }
    __syncthreads();  // every wave has read what it needs of A: T takes its place
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const uint32_t pair = pack_bf16(x[b][e], x[b][e + 1]);
        sm_t[16 * b + 4 * hq + e][16 * wave + m] = static_cast<uint16_t>(pair);
        sm_t[16 * b + 4 * hq + e + 1][16 * wave + m] = static_cast<uint16_t>(pair >> 16);
      }
  }
  __syncthreads();

  // ---- what the sequential kernel reads of this chunk -------------------------
  char* out = a.workspace + (static_cast<size_t>(bh) * chunks + chunk) * kGdnChunkBytes;
  uint4* t_out = reinterpret_cast<uint4*>(out + kGdnOffsetT);
  uint4* a2_out = reinterpret_cast<uint4*>(out + kGdnOffsetA2);
  // T and M o (Q K^T) as matrix-core operands over tokens j: fragment
  // (tile, kb), lane (hq, m) = row 16 tile + m, slot (hq, e) = column
  // 32 kb + 16 (e / 4) + 4 hq + e % 4; the two fragments above the diagonal
  // are zero and are not stored
  for (int piece = tid; piece < 6 * 64; piece += 256) {
    const int f = piece / 64, l = piece % 64;
    const int tile = f < 2 ? f : 2 + (f - 2) / 2, kb = f < 2 ? 0 : (f - 2) % 2;
    const int hq = l / 16, m = l % 16;
    const int row = 16 * tile + m, lo = 32 * kb + 4 * hq;
    uint2 w0 = *reinterpret_cast<const uint2*>(&sm_t[row][lo]);
    uint2 w1 = *reinterpret_cast<const uint2*>(&sm_t[row][lo + 16]);
    t_out[piece] = make_uint4(w0.x, w0.y, w1.x, w1.y);
    w0 = *reinterpret_cast<const uint2*>(&sm_a2[row][lo]);
    w1 = *reinterpret_cast<const uint2*>(&sm_a2[row][lo + 16]);
    a2_out[piece] = make_uint4(w0.x, w0.y, w1.x, w1.y);
  }
  // per-token factors, and the decay of the whole chunk
  float* factors = reinterpret_cast<float*>(out + kGdnOffsetFactors);
  const float cum_last = sm_cum[C - 1];
  if (tid < C) {
    const float grown = __expf(sm_cum[tid]);
    factors[tid] = sm_beta[tid];
    factors[C + tid] = sm_beta[tid] * grown * sm.inv_k[tid];
    factors[2 * C + tid] = sm.q_factor[tid] * grown;
    factors[3 * C + tid] = __expf(cum_last - sm_cum[tid]) * sm.inv_k[tid];
  } else if (tid < 2 * C) {
    // the rest of the block is loaded with it: keep it defined
    factors[4 * C + tid - C] = tid == C ? __expf(cum_last) : 0.0f;
  }
}

// LDS stage of the sequential kernel for one chunk: the chunk's scratch as it
// sits in memory (T | A2 | factors, 14 KiB), the raw K and Q rows gathered
// into matrix-core operand order (16 KiB each), and the 16 value columns of each
// of the workgroup's slices (2 KiB).
constexpr int kStageScratch = 0;
constexpr int kStageK = static_cast<int>(kGdnChunkBytes);
constexpr int kStageQ = kStageK + 16384;
constexpr int kStageV = kStageQ + 16384;
constexpr int scan_stage_bytes(int slices) { return kStageV + 2048 * slices; }
constexpr int kScanStages = 2;

typedef __attribute__((address_space(3))) unsigned char lds_byte;
typedef __attribute__((address_space(3))) const uint32x4 lds_u32x4;
typedef __attribute__((address_space(3))) const floatx4 lds_f32x4;
__device__ inline bf16x8 words_to_bf16x8(uint32x4 v) { return __builtin_bit_cast(bf16x8, v); }

// One direct-to-LDS load of 16 bytes per lane: lane l fetches
// descriptor base + voffset(l) + soffset and the hardware writes it at LDS
// byte lds_address + 16 l.  Only voffset is checked against the size in the
// descriptor (a lane beyond it reads zeros).  Issued as inline assembly on
// purpose: the compiler does not see an LDS write, so it does not make later
// reads of the OTHER stage wait for this load; the kernel orders the accesses
// itself with s_waitcnt vmcnt (see gdn_chunk_scan).
__device__ inline void lds_dma_16(uint32x4 descriptor, uint32_t lds_address, uint32_t voffset,
                                  uint32_t soffset) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen lds"
      :
      : "s"(lds_address), "v"(voffset), "s"(descriptor), "s"(soffset)
      : "memory", "m0");
}

// LDS transpose read of four 16-bit elements per lane (ds_read_b64_tr_b16):
// within every group of 16 lanes, source lane 4 kk + b supplies the 8 bytes at
// its address, and lane 4 b + e receives element e of source lanes b, b + 4,
// b + 8, b + 12 (kk = 0..3, in that order).
__device__ inline uint2 lds_transposed(const lds_byte* address) {
  const shortx4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) shortx4*)(address));
  return __builtin_bit_cast(uint2, v);
}

// K and Q operands sit in the stage in fragments of 64 slots of 16 bytes,
// fragment 4 tile + kb: logical lane (hq, m) holds token 16 tile + m, channels
// 32 kb + 8 hq .. + 7.  A token's four pieces occupy four consecutive slots, so
// the four lanes that fill them fetch 64 contiguous bytes; the pieces are
// rotated by m / 4 within those slots, which spreads both the operand reads
// (16 tokens at a fixed piece) and the transpose reads of K (four tokens at
// each of the four pieces) over the LDS banks.
__device__ inline int operand_slot(int hq, int m) { return 4 * m + ((hq + m / 4) & 3); }

// Where the loaders fetch a chunk from: one buffer descriptor per source, and
// the lane's own byte offset into each.
struct ScanSources {
  uint32x4 scratch, k, q, v;
  uint32_t k_lane, q_lane, v_lane;
  uint32_t k_row_bytes, q_row_bytes, v_row_bytes;
};

// The direct-to-LDS loads of one chunk, 1 KiB each: 14 of scratch, 16 of K,
// 16 of Q, 2 of V a slice.  Loader wave LOADER of LOADERS issues every LOADERS-th.
constexpr int kFillScratch = static_cast<int>(kGdnChunkBytes) / 1024;
constexpr int scan_fill_loads(int slices) { return kFillScratch + 16 + 16 + 2 * slices; }
template <int LOADER, int LOADERS, int WG_SLICES>
__device__ __forceinline__ void scan_fill(uint32_t stage_address, const ScanSources& src, int chunk,
                                          int lane) {
  const uint32_t lane_bytes = static_cast<uint32_t>(lane) * 16u;
  const uint32_t row0 = static_cast<uint32_t>(chunk) * C;
  // fully unrolled: a lone wave issues a loop's scalar bookkeeping far slower
  // than the memory pipeline takes loads
#pragma unroll
  for (int f = LOADER; f < scan_fill_loads(WG_SLICES); f += LOADERS) {
    if (f < kFillScratch) {
      lds_dma_16(src.scratch, stage_address + f * 1024, lane_bytes,
                 static_cast<uint32_t>(chunk) * static_cast<uint32_t>(kGdnChunkBytes) + f * 1024);
    } else if (f < kFillScratch + 32) {
      // rows past the end of the sequence lie beyond the descriptor's size and
      // read zeros: the whole offset goes through the checked lane offset
      const int g = (f - kFillScratch) % 16, tile = g / 4, kb = g % 4;
      if (f < kFillScratch + 16)
        lds_dma_16(src.k, stage_address + kStageK + g * 1024,
                   src.k_lane + (row0 + 16 * tile) * src.k_row_bytes + 64 * kb, 0);
      else
        lds_dma_16(src.q, stage_address + kStageQ + g * 1024,
                   src.q_lane + (row0 + 16 * tile) * src.q_row_bytes + 64 * kb, 0);
    } else {
      const int slice = (f - kFillScratch - 32) / 2, half = (f - kFillScratch - 32) % 2;
      lds_dma_16(src.v, stage_address + kStageV + slice * 2048 + half * 1024,
                 src.v_lane + (row0 + 32 * half) * src.v_row_bytes + 32 * slice, 0);
    }
  }
}

// Loader waves per workgroup, and what each needs at run time: the fill for its
// index, and a wait that lets exactly its share of one (the younger) fill stay
// in flight.
constexpr int kScanLoaders = 2;
constexpr int scan_fill_share(int loader, int slices) {
  return (scan_fill_loads(slices) - loader + kScanLoaders - 1) / kScanLoaders;
}
// (a wave whose two fills exceed the 63 operations its vector-memory counter
// holds merely stalls at the issue of the last few loads)
static_assert(scan_fill_share(0, 2) <= 63, "the wait for the older fill must be encodable");
template <int WG_SLICES>
__device__ __forceinline__ void scan_fill_as(int loader, uint32_t stage_address,
                                             const ScanSources& src, int chunk, int lane) {
  if (loader == 0) scan_fill<0, kScanLoaders, WG_SLICES>(stage_address, src, chunk, lane);
  else scan_fill<1, kScanLoaders, WG_SLICES>(stage_address, src, chunk, lane);
}
template <int WG_SLICES>
__device__ __forceinline__ void scan_wait_older_fill(int loader) {
  if (loader == 0)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(scan_fill_share(0, WG_SLICES)) : "memory");
  else
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(scan_fill_share(1, WG_SLICES)) : "memory");
}

// Pulls a slice's eighth of a future chunk (its scratch, its K rows and
// its Q rows; the eight slices of a (sequence, head) share all three) and
// its own V columns through L2 so that it is there by the time the workgroups fetch it for real:
// the loader waves cannot keep enough real loads in flight to cover the latency
// of HBM.  These are full-width loads (1 KiB per instruction): what bounds a
// compute unit is the number of requests it has in flight, and a narrow load
// per cache sector is one request per lane.  They go straight to an LDS dump
// area nobody reads, so they need no registers and the issuing wave never waits
// for them.
constexpr int kScanAhead = 4;
__device__ inline void scan_touch(const ScanSources& src, uint32_t dump_address, int chunk,
                                  int slice, uint32_t v_column_bytes, int lane) {
  const uint32_t lane_bytes = static_cast<uint32_t>(lane) * 16u;
  // scratch: 14 KiB / 8 = 1792 bytes, two loads (the second runs into the
  // next slice's share, or past the end of the scratch, where it reads zeros)
  const uint32_t scratch = static_cast<uint32_t>(chunk) * static_cast<uint32_t>(kGdnChunkBytes) +
                           static_cast<uint32_t>(slice) * (kGdnChunkBytes / SLICES) + lane_bytes;
#pragma unroll
  for (int i = 0; i < 2; ++i) lds_dma_16(src.scratch, dump_address, scratch + i * 1024, 0);
  // K and Q: eight token rows of 256 bytes each, four rows a load
  const uint32_t row = static_cast<uint32_t>(chunk) * C + 8 * slice + lane / 16;
  const uint32_t piece = (lane % 16) * 16u;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    lds_dma_16(src.k, dump_address, (row + 4 * i) * src.k_row_bytes + piece, 0);
    lds_dma_16(src.q, dump_address, (row + 4 * i) * src.q_row_bytes + piece, 0);
  }
  // V: the slice's 16 columns belong to this workgroup alone
#pragma unroll
  for (int half = 0; half < 2; ++half)
    lds_dma_16(src.v, dump_address,
               src.v_lane + (static_cast<uint32_t>(chunk) * C + 32 * half) * src.v_row_bytes +
                   v_column_bytes,
               0);
}

// One workgroup per (sequence, head, slice of 16 state columns): the chain wave (the
// sequential dependence from state to state: P = K S0, D, the state update),
// the output wave (Q S0, the causal product with D, the stores, and the loads
// that warm L2), and kScanLoaders loader waves.  A stage holds one chunk.  The
// two computing waves move the chunk's operands into registers as their matrix
// instructions need them; once the last read is issued the stage goes back to
// the loaders, which stream chunk c+2 into it (asynchronous direct-to-LDS
// loads), so each loader has two fills in flight.  Two workgroup barriers per
// chunk order everything: "landed" (the stage is complete, and the chain wave
// has published the state entering the chunk as a bf16 operand) and "free" (both
// computing waves are done with the stage, and the chain wave has published D).
// A wave that issues long runs of loads stalls at issue while the memory
// pipeline digests them, which is why the chain wave issues none.
//
// WG_SLICES = 2: a workgroup of six waves walks two slices of a head from one
// copy of the stage, a chain and an output wave each.  A compute unit holds one
// workgroup, and 48 heads are 384 single slices, one and a half rounds of the
// chip that take two; as 192 pairs they take one (8191 tokens: 290 -> 192 us).
constexpr int scan_threads(int slices) { return 64 * (2 * slices + kScanLoaders); }

// The workgroup barriers that hand an LDS stage over.  A loader arrives at the
// "landed" barrier once the stage's direct-to-LDS loads are complete (the
// caller waits for them); the computing wave arrives at the "free" barrier once
// its LDS reads are done, without waiting for its own vector-memory operations
// (output stores, L2 touches), which nobody in the workgroup depends on.
__device__ __forceinline__ void scan_barrier() { asm volatile("s_barrier" ::: "memory"); }
__device__ __forceinline__ void scan_handover_compute() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

struct ScanContext {
  uint16_t* out;
  int length, value_heads;
  int slice, local, lane, hq, m, seq, head;  // local: the slice within the workgroup
};

__device__ inline float bf16_half(uint32_t word, int upper) {
  return __builtin_bit_cast(float, upper ? (word & 0xffff0000u) : (word << 16));
}

// What the chain wave hands to the output wave through LDS, one 16-byte slot a
// lane: the state entering the chunk as four operands, D as two.
struct ScanExchange {
  uint32x4 state[4][64];
  uint32x4 d[2][64];
};
typedef __attribute__((address_space(3))) ScanExchange lds_exchange;

__device__ inline uint32x4 bf16x8_to_words(bf16x8 v) { return __builtin_bit_cast(uint32x4, v); }

// The chain wave's share of one chunk.  The state s[t] holds rows
// 16 t + 4 hq + r of the slice's column m, where row rho stands for key channel
// 32 (rho / 32) + 8 ((rho % 16) / 4) + 4 ((rho / 16) % 2) + rho % 4: with that
// order the raw rows of K and Q are matrix-core operands as they are (eight
// consecutive channels per lane).  `sb` is the state as operands, which the
// caller has already published; on return it is the next chunk's.
__device__ __forceinline__ void chain_step(const ScanContext ctx, const lds_byte* stage,
                                           lds_exchange* exchange, floatx4 (&s)[8],
                                           bf16x8 (&sb)[4]) {
  const int lane = ctx.lane, hq = ctx.hq, m = ctx.m;
  const int slot = operand_slot(hq, m);
  lds_u32x4* k_in = (lds_u32x4*)(stage + kStageK) + slot;
  lds_u32x4* t_in = (lds_u32x4*)(stage + kStageScratch + kGdnOffsetT) + lane;
  // factor n of rows 16 i + 4 hq .. + 3: four consecutive floats
  lds_f32x4* factor_in = (lds_f32x4*)(stage + kStageScratch + kGdnOffsetFactors) + hq;
  const float decay =
      *(const __attribute__((address_space(3))) float*)(stage + kStageScratch + kGdnOffsetFactors + 4 * C * 4);
  // as a source lane of the transpose reads: token row kk of a group of four,
  // 8-byte piece b of the row
  const int kk = m / 4, piece = m % 4;
  const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f};

  // LDS reads are issued well ahead of the matrix instructions that consume
  // them (a read takes about as long as four matrix instructions): the K
  // fragments one token tile ahead, everything the later phases need during the
  // phase before.
  uint32x4 k_reg[2][4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) k_reg[0][kb] = k_in[kb * 64];
  uint2 v_reg[4];
  floatx4 f1[4], f2[4], f4[4];
  uint32x4 t_reg[6];  // (i, kb) = (0,0) (1,0) (2,0) (2,1) (3,0) (3,1): T is lower triangular
  floatx4 p[4];
  // P = K S0, token tile by token tile
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i + 1 < 4) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) k_reg[(i + 1) % 2][kb] = k_in[(4 * (i + 1) + kb) * 64];
    }
    if (i == 0) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v_reg[j] = lds_transposed(stage + kStageV + 2048 * ctx.local + (16 * j + 4 * hq + kk) * 32 + 8 * piece);
        f1[j] = factor_in[4 * j];
      }
    } else if (i == 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) f2[j] = factor_in[16 + 4 * j];
      t_reg[0] = t_in[0 * 64];
      t_reg[1] = t_in[1 * 64];
      t_reg[2] = t_in[2 * 64];
    } else if (i == 2) {
      t_reg[3] = t_in[3 * 64];
      t_reg[4] = t_in[4 * 64];
      t_reg[5] = t_in[5 * 64];
#pragma unroll
      for (int j = 0; j < 4; ++j) f4[j] = factor_in[48 + 4 * j];
    }
    __builtin_amdgcn_sched_barrier(0);
    floatx4 acc = zero;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) acc = mfma16(words_to_bf16x8(k_reg[i % 2][kb]), sb[kb], acc);
    p[i] = acc;
    __builtin_amdgcn_sched_barrier(0);
  }
  // S = exp(c_C) S0 + K^T (diag(exp(c_C - c) / |k|) D): row tile t = 2 kb + j
  // of the state is channels 32 kb + 8 b + 4 j + e for operand row 4 b + e,
  // read from the K fragments through the transposing LDS path; tokens
  // 32 tb + 16 jt + 4 hq + kk, jt = 0, 1
  uint2 kt_reg[2][8][2];
  auto read_kt = [&](int tb) {
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int kb = t / 2, j = t % 2;
      const lds_byte* base = stage + kStageK + 8 * j;
#pragma unroll
      for (int jt = 0; jt < 2; ++jt)
        kt_reg[tb][t][jt] = lds_transposed(
            base + (((2 * tb + jt) * 4 + kb) * 64 + operand_slot(piece, 4 * hq + kk)) * 16);
    }
  };
  read_kt(0);
  __builtin_amdgcn_sched_barrier(0);
  // R = diag(beta) V - diag(beta exp(c) / |k|) P, then D = T R
  floatx4 rt[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint2 v = v_reg[i];
    rt[i][0] = f1[i][0] * bf16_half(v.x, 0) - f2[i][0] * p[i][0];
    rt[i][1] = f1[i][1] * bf16_half(v.x, 1) - f2[i][1] * p[i][1];
    rt[i][2] = f1[i][2] * bf16_half(v.y, 0) - f2[i][2] * p[i][2];
    rt[i][3] = f1[i][3] * bf16_half(v.y, 1) - f2[i][3] * p[i][3];
  }
  bf16x8 r_op[2];
  r_op[0] = tiles_to_operand(rt[0], rt[1]);
  r_op[1] = tiles_to_operand(rt[2], rt[3]);
  __builtin_amdgcn_sched_barrier(0);
  read_kt(1);
  __builtin_amdgcn_sched_barrier(0);
  floatx4 d[4];
  {
    constexpr int first[4] = {0, 1, 2, 4};  // index of (i, 0) in t_reg
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      floatx4 acc = zero;
#pragma unroll
      for (int kb = 0; kb < (i < 2 ? 1 : 2); ++kb)
        acc = mfma16(words_to_bf16x8(t_reg[first[i] + kb]), r_op[kb], acc);
      d[i] = acc;
    }
  }
  // the two roles of D: as it is for the outputs (published for the output
  // wave), scaled by exp(c_C - c) / |k| for the state
  bf16x8 ds[2];
  {
    floatx4 scaled[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) scaled[i] = d[i] * f4[i];
    exchange->d[0][lane] = bf16x8_to_words(tiles_to_operand(d[0], d[1]));
    exchange->d[1][lane] = bf16x8_to_words(tiles_to_operand(d[2], d[3]));
    ds[0] = tiles_to_operand(scaled[0], scaled[1]);
    ds[1] = tiles_to_operand(scaled[2], scaled[3]);
  }
  // every read of the stage has been issued, D is on its way to LDS
  scan_handover_compute();
#pragma unroll
  for (int t = 0; t < 8; ++t) s[t] = s[t] * decay;
#pragma unroll
  for (int tb = 0; tb < 2; ++tb) {
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const uint32x4 words = {kt_reg[tb][t][0].x, kt_reg[tb][t][0].y, kt_reg[tb][t][1].x,
                              kt_reg[tb][t][1].y};
      s[t] = mfma16(words_to_bf16x8(words), ds[tb], s[t]);
    }
  }
  // the next chunk's operands, published before its "landed" barrier
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    sb[kb] = tiles_to_operand(s[2 * kb], s[2 * kb + 1]);
    exchange->state[kb][lane] = bf16x8_to_words(sb[kb]);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// The output wave's share of one chunk:
// O = diag(q_scale exp(c) / |q|) Q S0 + (M o Q K^T) D.
__device__ __forceinline__ void output_step(const ScanContext ctx, int chunk, const lds_byte* stage,
                                            const lds_exchange* exchange) {
  const int slice = ctx.slice, lane = ctx.lane, hq = ctx.hq, m = ctx.m;
  lds_u32x4* q_in = (lds_u32x4*)(stage + kStageQ) + operand_slot(hq, m);
  lds_u32x4* a2_in = (lds_u32x4*)(stage + kStageScratch + kGdnOffsetA2) + lane;
  lds_f32x4* factor_in = (lds_f32x4*)(stage + kStageScratch + kGdnOffsetFactors) + hq;
  const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  bf16x8 sb[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) sb[kb] = words_to_bf16x8(exchange->state[kb][lane]);
  uint32x4 q_reg[2][4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) q_reg[0][kb] = q_in[kb * 64];
  uint32x4 a2_reg[6];  // (i, kb) = (0,0) (1,0) (2,0) (2,1) (3,0) (3,1): causal
  floatx4 f3[4];
  floatx4 o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i + 1 < 4) {
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) q_reg[(i + 1) % 2][kb] = q_in[(4 * (i + 1) + kb) * 64];
    }
    if (i == 1) {
      a2_reg[0] = a2_in[0 * 64];
      a2_reg[1] = a2_in[1 * 64];
      a2_reg[2] = a2_in[2 * 64];
    } else if (i == 2) {
      a2_reg[3] = a2_in[3 * 64];
      a2_reg[4] = a2_in[4 * 64];
      a2_reg[5] = a2_in[5 * 64];
#pragma unroll
      for (int j = 0; j < 4; ++j) f3[j] = factor_in[32 + 4 * j];
    }
    __builtin_amdgcn_sched_barrier(0);
    floatx4 acc = zero;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) acc = mfma16(words_to_bf16x8(q_reg[i % 2][kb]), sb[kb], acc);
    o[i] = acc;
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = o[i] * f3[i];
  // done with the stage; D follows the barrier
  scan_handover_compute();
  bf16x8 db[2];
  db[0] = words_to_bf16x8(exchange->d[0][lane]);
  db[1] = words_to_bf16x8(exchange->d[1][lane]);
  {
    constexpr int first[4] = {0, 1, 2, 4};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int kb = 0; kb < (i < 2 ? 1 : 2); ++kb)
        o[i] = mfma16(words_to_bf16x8(a2_reg[first[i] + kb]), db[kb], o[i]);
    }
  }
  // outputs: rows 16i + 4hq + r of the chunk, column 16*slice + m
  uint16_t* out_row = ctx.out +
      ((static_cast<long long>(ctx.seq) * ctx.length + chunk * C + 4 * hq) * ctx.value_heads + ctx.head) * DV +
      16 * slice + m;
  const long long row_step = static_cast<long long>(ctx.value_heads) * DV;
  if (chunk * C + C <= ctx.length) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) out_row[(16 * i + r) * row_step] = float_to_bf16_bits(o[i][r]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (chunk * C + 16 * i + 4 * hq + r < ctx.length)
          out_row[(16 * i + r) * row_step] = float_to_bf16_bits(o[i][r]);
  }
}

__device__ inline uint32x4 raw_descriptor(const void* base, uint32_t bytes) {
  const uint64_t address = reinterpret_cast<uint64_t>(base);
  // base address, no stride, size in bytes, data format
  return uint32x4{static_cast<uint32_t>(address), static_cast<uint32_t>(address >> 32) & 0xffffu,
                  bytes, 0x00020000u};
}

template <int WG_SLICES>
__global__ void __launch_bounds__(scan_threads(WG_SLICES))
gdn_chunk_scan(GdnArgs a) {
  constexpr int kScanStageBytes = scan_stage_bytes(WG_SLICES);
  __shared__ __attribute__((aligned(1024))) unsigned char stages[kScanStages * kScanStageBytes];
  __shared__ __attribute__((aligned(256))) unsigned char dump[1024];
  __shared__ __attribute__((aligned(16))) ScanExchange exchanges[WG_SLICES];
  const int lane = threadIdx.x % 64, hq = lane / 16, m = lane % 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int chunks = (a.length + C - 1) / C;
  // The workgroups of one (sequence, head) read the same operands: keep them
  // on one XCD so that its L2 serves all but the first read.
  int logical = blockIdx.x;
  if (gridDim.x % 8 == 0) logical = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  constexpr int kGroups = SLICES / WG_SLICES;
  const int first_slice = logical % kGroups * WG_SLICES;
  const int bh = logical / kGroups;
  const int head = bh % a.value_heads, seq = bh / a.value_heads;
  const int key_head = head / (a.value_heads / a.key_heads);
  float* state = a.state + static_cast<size_t>(bh) * DK * DV;

  ScanSources src;
  src.scratch = raw_descriptor(a.workspace + static_cast<size_t>(bh) * chunks * kGdnChunkBytes,
                               static_cast<uint32_t>(chunks * kGdnChunkBytes));
  const long long first_token = static_cast<long long>(seq) * a.length;
  src.k_row_bytes = static_cast<uint32_t>(a.k_token_stride * 2);
  src.q_row_bytes = static_cast<uint32_t>(a.q_token_stride * 2);
  src.v_row_bytes = static_cast<uint32_t>(a.v_token_stride * 2);
  src.k = raw_descriptor(a.k + first_token * a.k_token_stride + key_head * DK,
                         static_cast<uint32_t>(a.length - 1) * src.k_row_bytes + DK * 2);
  src.q = raw_descriptor(a.q + first_token * a.q_token_stride + key_head * DK,
                         static_cast<uint32_t>(a.length - 1) * src.q_row_bytes + DK * 2);
  src.v = raw_descriptor(a.v + first_token * a.v_token_stride + head * DV + 16 * first_slice,
                         static_cast<uint32_t>(a.length - 1) * src.v_row_bytes + 16 * WG_SLICES * 2);
  {
    // LDS slot `lane` of a K or Q fragment belongs to the logical lane whose
    // operand_slot it is: token lane / 4 of the tile, piece (lane % 4 - token / 4) mod 4
    const uint32_t token = static_cast<uint32_t>(lane / 4);
    const uint32_t part = static_cast<uint32_t>((lane % 4 - lane / 16) & 3);
    src.k_lane = token * src.k_row_bytes + 16u * part;
    src.q_lane = token * src.q_row_bytes + 16u * part;
    // V: two slots a token (16 columns = 32 bytes)
    src.v_lane = static_cast<uint32_t>(lane / 2) * src.v_row_bytes + 16u * (lane % 2);
  }
  // chunk c lives in stage c % 2; every address within a stage is then the
  // stage's base plus a constant
  const uint32_t stage0_address = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_byte*)stages));
  const uint32_t stage1_address = stage0_address + kScanStageBytes;
  const uint32_t dump_address =
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_byte*)dump));

  // Every wave passes two barriers per chunk: "landed" and "free".
  if (wave >= 2 * WG_SLICES) {
    const int loader = wave - 2 * WG_SLICES;
    scan_fill_as<WG_SLICES>(loader, stage0_address, src, 0, lane);
    if (chunks > 1) scan_fill_as<WG_SLICES>(loader, stage1_address, src, 1, lane);
    for (int chunk = 0; chunk < chunks; ++chunk) {
      // loads complete in issue order: all but the younger fill have landed
      if (chunk + 1 < chunks) scan_wait_older_fill<WG_SLICES>(loader);
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      scan_barrier();  // landed
      scan_barrier();  // free
      if (chunk + 2 < chunks)
        scan_fill_as<WG_SLICES>(loader, (chunk & 1) ? stage1_address : stage0_address, src, chunk + 2,
                                lane);
    }
    return;
  }

  const int local = wave % WG_SLICES, slice = first_slice + local;
  const lds_byte* stage_base = (const lds_byte*)stages;
  lds_exchange* exchange = (lds_exchange*)&exchanges[local];
  ScanContext ctx;
  ctx.out = a.out;
  ctx.length = a.length;
  ctx.value_heads = a.value_heads;
  ctx.slice = slice;
  ctx.local = local;
  ctx.lane = lane;
  ctx.hq = hq;
  ctx.m = m;
  ctx.seq = seq;
  ctx.head = head;
  // (the loaders share the output waves' SIMDs)
  if (wave < WG_SLICES) {
    for (int chunk = 2; chunk < min(kScanAhead + 2, chunks); ++chunk)
      scan_touch(src, dump_address, chunk, slice, 32 * local, lane);
    for (int chunk = 0; chunk < chunks; ++chunk) {
      if (chunk + 2 + kScanAhead < chunks)
        scan_touch(src, dump_address, chunk + 2 + kScanAhead, slice, 32 * local, lane);
      scan_barrier();  // landed
      // passes the "free" barrier once it has read all it needs of the stage,
      // and has read D by the time it returns
      output_step(ctx, chunk, stage_base + (chunk & 1) * kScanStageBytes, exchange);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    return;
  }

  // state rows in operand order (see chain_step)
  floatx4 s[8];
#pragma unroll
  for (int t = 0; t < 8; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      s[t][r] = state[(32 * (t / 2) + 8 * hq + 4 * (t % 2) + r) * DV + 16 * slice + m];
  bf16x8 sb[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    sb[kb] = tiles_to_operand(s[2 * kb], s[2 * kb + 1]);
    exchange->state[kb][lane] = bf16x8_to_words(sb[kb]);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  for (int chunk = 0; chunk < chunks; ++chunk) {
    scan_barrier();  // landed
    // passes the "free" barrier once it has read all it needs of the stage
    chain_step(ctx, stage_base + (chunk & 1) * kScanStageBytes, exchange, s, sb);
  }
#pragma unroll
  for (int t = 0; t < 8; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      state[(32 * (t / 2) + 8 * hq + 4 * (t % 2) + r) * DV + 16 * slice + m] = s[t][r];
}

// Token-by-token recurrence, any widths up to 128 x 256: one workgroup per
// (sequence, head), one thread per state column, the column's state in
// registers.  This is the reference's own loop structure
// (sequence_delta_net.cc:79-101); it serves shapes the chunked path does not
// specialise and cross-checks the chunked scan on the device.
__global__ void __launch_bounds__(256)
gdn_recurrence_kernel(GdnArgs a, int out_dtype) {
  __shared__ float ks[128];
  __shared__ float qs[128];
  const int bh = blockIdx.x;
  const int head = bh % a.value_heads, seq = bh / a.value_heads;
  const int key_head = head / (a.value_heads / a.key_heads);
  const int kd = a.key_dim, vd = a.value_dim;
  const int column = threadIdx.x;
  const bool active = column < vd;
  float* state = a.state + static_cast<size_t>(bh) * kd * vd;
  float s[128];
#pragma unroll
  for (int d = 0; d < 128; ++d) s[d] = (d < kd && active) ? state[d * vd + column] : 0.0f;
  for (int t = 0; t < a.length; ++t) {
    const long long token = static_cast<long long>(seq) * a.length + t;
    __syncthreads();
    if (threadIdx.x < 128) {
      const int d = threadIdx.x;
      ks[d] = d < kd ? load_element(a.k, token * a.k_token_stride + key_head * kd + d, a.in_dtype) : 0.0f;
      qs[d] = d < kd ? load_element(a.q, token * a.q_token_stride + key_head * kd + d, a.in_dtype) : 0.0f;
    }
    __syncthreads();
    float k_factor = 1.0f, q_factor = a.q_scale;
    if (a.normalize_qk) {
      float kk = 1e-6f, qq = 1e-6f;
      for (int d = 0; d < kd; ++d) {
        kk += ks[d] * ks[d];
        qq += qs[d] * qs[d];
      }
      k_factor = rsqrtf(kk);
      q_factor = a.q_scale * rsqrtf(qq);
    }
    const long long scalar = token * a.value_heads + head;
    const float decay = __expf(a.log_decay[scalar]);
    const float beta = a.beta[scalar];
    float value = 0.0f;
    if (active) value = load_element(a.v, token * a.v_token_stride + head * vd + column, a.in_dtype);
    float prediction = 0.0f;
#pragma unroll
    for (int d = 0; d < 128; ++d) {
      if (d < kd) {
        s[d] *= decay;
        prediction += s[d] * (ks[d] * k_factor);
      }
    }
    const float delta = (value - prediction) * beta;
    float output = 0.0f;
#pragma unroll
    for (int d = 0; d < 128; ++d) {
      if (d < kd) {
        s[d] += (ks[d] * k_factor) * delta;
        output += s[d] * (qs[d] * q_factor);
      }
    }
    if (active) {
      const long long at = (token * a.value_heads + head) * vd + column;
      if (out_dtype == PLUTO_HIP_BF16)
        static_cast<uint16_t*>(a.out_any)[at] = float_to_bf16_bits(output);
      else
        static_cast<float*>(a.out_any)[at] = a.round_output ? round_to_bf16(output) : output;
    }
  }
#pragma unroll
  for (int d = 0; d < 128; ++d)
    if (d < kd && active) state[d * vd + column] = s[d];
}

}  // namespace

bool gdn_chunked_supported(const GdnArgs& a, int chunk) {
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  // the sequential kernel addresses a sequence's rows through 32-bit offsets
  auto in_range = [&](long long token_stride) {
    return token_stride > 0 && token_stride * 2 * a.length < (1LL << 31);
  };
  if (!in_range(a.q_token_stride) || !in_range(a.k_token_stride) || !in_range(a.v_token_stride))
    return false;
  return chunk == C && a.key_dim == DK && a.value_dim == DV && a.in_dtype == PLUTO_HIP_BF16 &&
         a.q_token_stride % 8 == 0 && a.k_token_stride % 8 == 0 && a.v_token_stride % 8 == 0 &&
         aligned(a.q) && aligned(a.k) && aligned(a.v) && aligned(a.workspace);
}

// While every head of a chunk gets a compute unit of its own, three heads of one key head are
// prepared faster by a workgroup each (six by one for every two), though each convolves the
// rows of K and Q: the one workgroup's 12 waves share a compute unit while others idle.  The whole forward of 16/48 heads,
// three a workgroup and one: 17 tokens 29.2 and 25.6 us, 320 (240 heads of chunks) 39.7 and
// 37.4, 400 (336) 45.2 and 44.4, 700 (528) 51.2 and 55.9, 8191 348 and 377; of 4/12 heads 1400
// (264) 59.0 and 58.0, 2000 (384) 68.8 and 69.4.  (17 tokens took 27.0 with the convolution and
// the gates as passes of their own.)
constexpr unsigned kAlonePreparations = 256;

bool gdn_layer_rows_supported(const GdnLayerInputs& layer, int taps) {
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  return taps == 4 && aligned(layer.qkv) && aligned(layer.conv_weight);
}

int launch_gdn_chunked(hipStream_t stream, const GdnArgs& a, const GdnLayerInputs* layer) {
  const long long chunks = (a.length + C - 1) / C;
  const long long heads = static_cast<long long>(a.batch) * a.value_heads;
  if (heads * chunks > 0x7fffffffLL) return PLUTO_HIP_EINVAL;
  if (kernel_enabled(kAuxiliaryKernel)) {
    const int group = a.value_heads / a.key_heads;
    const unsigned blocks = static_cast<unsigned>(heads * chunks);
    if (layer == nullptr)
      gdn_chunk_prepare<1, false><<<blocks, 256, 0, stream>>>(a, {});
    else if (group % 3 == 0 && blocks > kAlonePreparations)
      gdn_chunk_prepare<3, true><<<blocks / 3, 768, 0, stream>>>(a, *layer);
    else if (group % 2 == 0)
      gdn_chunk_prepare<2, true><<<blocks / 2, 512, 0, stream>>>(a, *layer);
    else
      gdn_chunk_prepare<1, true><<<blocks, 256, 0, stream>>>(a, *layer);
  }
  int status = launch_status();
  if (status != 0) return status;
  if (!kernel_enabled(kMainKernel)) return 0;
  // one workgroup a compute unit: two slices a workgroup where that saves a round
  int device = 0, units = 0;
  status = static_cast<int>(hipGetDevice(&device));
  if (status == 0)
    status = static_cast<int>(
        hipDeviceGetAttribute(&units, hipDeviceAttributeMultiprocessorCount, device));
  if (status != 0) return status;
  auto rounds = [&](long long workgroups) { return (workgroups + units - 1) / units; };
  if (rounds(heads * SLICES / 2) < rounds(heads * SLICES))
    gdn_chunk_scan<2><<<static_cast<unsigned>(heads * SLICES / 2), scan_threads(2), 0, stream>>>(a);
  else
    gdn_chunk_scan<1><<<static_cast<unsigned>(heads * SLICES), scan_threads(1), 0, stream>>>(a);
  return launch_status();
}

int launch_gdn_recurrence(hipStream_t stream, const GdnArgs& a, int out_dtype) {
  if (a.key_dim > 128 || a.value_dim > 256) return PLUTO_HIP_EUNSUPPORTED;
  gdn_recurrence_kernel<<<a.batch * a.value_heads, 256, 0, stream>>>(a, out_dtype);
  return launch_status();
}

}  // namespace pluto_hip
