// FullyConnectedLayer, trainable path (src/llm/layers/fully_connected.cc):
//   DenseForwardKernel         :97-131   y = bias + x w        (FP32 accumulate)
//   DenseInputGradientKernel   :134-164  dx = dy w^T
//   DenseWeightGradientKernel  :167-196  dw = x^T dy
//   DenseBias*GradientKernel   :198-247  db = column sums of dy, fixed order
// Operands are multiplied as 16-bit values (bf16 for bf16 activations, IEEE
// half for FP32 activations: MmaType, :31-33) and summed in FP32.  The FP32
// master matrix [input_dim, output_dim] and the FP32 gradient are converted
// to 16 bits once per call; the products then run on v_mfma_f32_32x32x16_*
// from LDS tiles filled by direct-to-LDS loads:
//   y and dx:      rows of both operands are contiguous along the contraction
//                  (x and w^T; dy and w) -> 16-byte row reads
//   dw:            the contraction runs over tokens, both operands (x, dy) are
//                  read through the LDS transpose read; the token range is
//                  split over workgroups and the slices are added in a fixed
//                  order
// Widths that are not multiples of 64 take a one-thread-per-element kernel
// with the same operand rounding.
#include "dense.h"

#include "mfma_tile.h"

#include <algorithm>

namespace pluto_hip {
namespace {

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 256;
constexpr int kDepth = 64;        // contraction elements per LDS tile
constexpr int kBiasRows = 256;    // fully_connected.cc:38

template <bool HALF>
__device__ inline floatx16 mma(uint4 a, uint4 b, floatx16 c) {
  if constexpr (HALF)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(halfx8, a),
                                                  __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

template <bool HALF>
__device__ inline uint16_t to_operand(float value) {
  if constexpr (HALF) {
    const _Float16 h = static_cast<_Float16>(value);
    return __builtin_bit_cast(uint16_t, h);
  } else {
    return float_to_bf16_bits(value);
  }
}

template <bool HALF>
__device__ inline float operand_value(float value) {
  if constexpr (HALF)
    return static_cast<float>(static_cast<_Float16>(value));
  else
    return round_to_bf16(value);
}

// out[i] = operand(in[i]): eight elements a thread where both are aligned, thread `index`
// of `threads`.
template <bool HALF>
__device__ inline void convert_elements(const float* in, long long total, uint16_t* out,
                                        long long index, long long threads) {
  const bool wide = reinterpret_cast<uintptr_t>(in) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
  const long long eights = wide ? total / 8 : 0;
  for (long long i = index; i < eights; i += threads) {
    const float4 a = *reinterpret_cast<const float4*>(in + 8 * i);
    const float4 b = *reinterpret_cast<const float4*>(in + 8 * i + 4);
    ushort4 lo, hi;
    lo.x = to_operand<HALF>(a.x), lo.y = to_operand<HALF>(a.y), lo.z = to_operand<HALF>(a.z);
    lo.w = to_operand<HALF>(a.w), hi.x = to_operand<HALF>(b.x), hi.y = to_operand<HALF>(b.y);
    hi.z = to_operand<HALF>(b.z), hi.w = to_operand<HALF>(b.w);
    *reinterpret_cast<ushort4*>(out + 8 * i) = lo;
    *reinterpret_cast<ushort4*>(out + 8 * i + 4) = hi;
  }
  for (long long i = 8 * eights + index; i < total; i += threads) out[i] = to_operand<HALF>(in[i]);
}

// Four neighbouring values in one access at any address of their type: global memory
// takes wide accesses unaligned, the types keep the compiler from assuming more.
struct __attribute__((packed, aligned(4))) FourFloats {
  float x, y, z, w;
};
struct __attribute__((packed, aligned(2))) FourHalves {
  uint32_t low, high;
};

// What a product needs converted, in one launch: the first blocks transpose the matrix
// [rows, cols] to out [cols, rows] by tiles of 64 (both are multiples), the rest convert the
// input.  Sixteen bytes an access on both sides: 512 rows of 768 -> 2304 4.3 us, of 3072 ->
// 768 4.5 (5.0 and 6.6 an element an access with tiles of 32).
template <bool HALF>
__global__ void __launch_bounds__(256)
convert_forward_kernel(const float* matrix, int rows, int cols, uint16_t* out, int tiles,
                       const float* input, long long elements, uint16_t* input16) {
  if (static_cast<int>(blockIdx.x) >= tiles) {
    convert_elements<HALF>(input, elements, input16, (blockIdx.x - tiles) * 256LL + threadIdx.x,
                           (gridDim.x - tiles) * 256LL);
    return;
  }
  constexpr int kEdge = 64, kPitch = kEdge + 4;
  __shared__ __attribute__((aligned(16))) uint16_t tile[kEdge][kPitch];
  const int across = cols / kEdge;
  const int c0 = blockIdx.x % across * kEdge, r0 = blockIdx.x / across * kEdge;
  {
    const int quad = threadIdx.x % 16, row = threadIdx.x / 16;
    FourFloats v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = *reinterpret_cast<const FourFloats*>(matrix + static_cast<long long>(r0 + row + 16 * i) * cols + c0 + 4 * quad);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ushort4 four;
      four.x = to_operand<HALF>(v[i].x), four.y = to_operand<HALF>(v[i].y);
      four.z = to_operand<HALF>(v[i].z), four.w = to_operand<HALF>(v[i].w);
      *reinterpret_cast<ushort4*>(&tile[row + 16 * i][4 * quad]) = four;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int chunk = threadIdx.x % 8, column = threadIdx.x / 8 + 32 * i;
    uint32_t words[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      words[e] = tile[8 * chunk + 2 * e][column] | static_cast<uint32_t>(tile[8 * chunk + 2 * e + 1][column]) << 16;
    *reinterpret_cast<uint4*>(out + static_cast<long long>(c0 + column) * rows + r0 + 8 * chunk) =
        make_uint4(words[0], words[1], words[2], words[3]);
  }
}

struct ProductArgs {
  const uint16_t* left = nullptr;    // [m_rows, depth]   -> output rows
  const uint16_t* right = nullptr;   // [n_rows, depth]   -> output columns
  const float* bias = nullptr;       // optional [n_rows]
  void* out = nullptr;               // [m_rows, n_rows], bf16 or fp32
  int m_rows = 0, n_rows = 0, depth = 0;
  bool out_bf16 = false;
};

// Workgroup barrier that leaves queued global loads in flight (the library
// barrier waits for them too).
__device__ inline void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int COUNT>
__device__ inline void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(COUNT) : "memory");
}

// out[m, n] = bias[n] + sum_k left[m, k] right[n, k]; depth % 64 == 0.  A
// workgroup of four waves, arranged 2 x 2, owns a 64 x (64 JN) tile and each wave
// a 32 x (32 JN) part of it.  Two LDS stages of 64 contraction elements: one is
// filled while the other is multiplied.  GROUPS: as many such sets of four waves share the
// tile, each with every GROUPS-th stage of the contraction, and add their sums through LDS
// in order.  A step is a chain of waits of 0.5 us (memory, barrier, LDS; eight stages in
// flight took 0.44), which several workgroups on a compute unit cover for each other;
// where there are too few of them, the groups do: 256 rows, 768 -> 2304 and its input
// gradient take 8.0 and 18.6 us with one group, 6.1 and 11.8 with four; 512 rows 9.4 and
// 19.2, 9.3 (two groups: 288 workgroups) and 12.7; 2000 rows of 2304 -> 768 20.4 and 18.1
// (two).
template <bool HALF, int JN, int GROUPS>
__global__ void __launch_bounds__(kThreads * GROUPS)
product_rows_kernel(ProductArgs a) {
  constexpr int KS = kDepth / 16;  // matrix instructions along the contraction per stage
  constexpr int TM = 64, TN = 64 * JN;
  constexpr int kLeftBytes = TM * kDepth * 2, kRightBytes = TN * kDepth * 2;
  constexpr int kStageBytes = kLeftBytes + kRightBytes;
  constexpr int LEFT_LOADS = TM * (kDepth / 8) / kThreads;
  constexpr int RIGHT_LOADS = TN * (kDepth / 8) / kThreads;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * GROUPS * kStageBytes];
  const int tid = threadIdx.x % kThreads, wave = tid / 64, lane = tid % 64;
  const int group = GROUPS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / kThreads);
  const int h = lane / 32, n = lane % 32;
  const int n_tiles = (a.n_rows + TN - 1) / TN;
  const int logical = xcd_logical_block();
  const int m0 = (logical / n_tiles) * TM, n0 = (logical % n_tiles) * TN;
  const int wm = 32 * (wave / 2), wn = 32 * JN * (wave % 2);
  uint32_t left_fill[LEFT_LOADS], right_fill[RIGHT_LOADS];
#pragma unroll
  for (int i = 0; i < LEFT_LOADS; ++i)
    left_fill[i] = tile_fill_offset<kDepth>((wave * LEFT_LOADS + i) * 64 + lane, a.depth);
#pragma unroll
  for (int i = 0; i < RIGHT_LOADS; ++i)
    right_fill[i] = tile_fill_offset<kDepth>((wave * RIGHT_LOADS + i) * 64 + lane, a.depth);
  // Rows 32 apart share the swizzle: block j of a quarter is 32 j rows further.
  constexpr int kBlockStep = 32 * (kDepth / 8) * 16;
  int left_read[KS], right_read[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    left_read[ks] = tile_row_read<kDepth>(wm + n, 2 * ks + h);
    right_read[ks] = tile_row_read<kDepth>(wn + n, 2 * ks + h);
  }
  // acc[jn]: a lane holds output column n0 + wn + 32 jn + n of rows
  // m0 + wm + 8 q + 4 h + i (element 4 q + i)
  floatx16 acc[JN];
#pragma unroll
  for (int jn = 0; jn < JN; ++jn) {
    const int column = n0 + wn + 32 * jn + n;
    const float start = (group == 0 && a.bias && column < a.n_rows) ? a.bias[column] : 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[jn][i] = start;
  }
  const uint16_t* left = a.left + static_cast<long long>(m0) * a.depth;
  const uint16_t* right = a.right + static_cast<long long>(n0) * a.depth;
  const int steps = a.depth / kDepth;
  // turn t of group g is step t GROUPS + g
  auto fill_stage = [&](int turn) {
    const int step = turn * GROUPS + group;
    if (step >= steps) return;
    unsigned char* stage = lds + (2 * group + turn % 2) * kStageBytes;
    tile_fill<kDepth, LEFT_LOADS>(stage, wave, left + step * kDepth, a.depth, m0, a.m_rows,
                                  left_fill);
    tile_fill<kDepth, RIGHT_LOADS>(stage + kLeftBytes, wave, right + step * kDepth, a.depth, n0,
                                   a.n_rows, right_fill);
  };
  fill_stage(0);
  for (int turn = 0; turn * GROUPS < steps; ++turn) {
    wait_loads<0>();
    lds_barrier();
    fill_stage(turn + 1);
    if (turn * GROUPS + group >= steps) break;  // the last turn
    const unsigned char* left_tile = lds + (2 * group + turn % 2) * kStageBytes;
    const unsigned char* right_tile = left_tile + kLeftBytes;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint4 r[JN];
      const uint4 l = *reinterpret_cast<const uint4*>(left_tile + left_read[ks]);
#pragma unroll
      for (int j = 0; j < JN; ++j)
        r[j] = *reinterpret_cast<const uint4*>(right_tile + right_read[ks] + j * kBlockStep);
#pragma unroll
      for (int jn = 0; jn < JN; ++jn) acc[jn] = mma<HALF>(l, r[jn], acc[jn]);
    }
  }
  if constexpr (GROUPS > 1) {
    // the groups' sums in order; group g finishes registers 16 / GROUPS g ..
    static_assert(JN == 1 && GROUPS * kThreads * 16 * 4 <= sizeof(lds));
    float (*sums)[16][kThreads] = reinterpret_cast<float (*)[16][kThreads]>(lds);
    lds_barrier();  // every group is done with its stages
#pragma unroll
    for (int i = 0; i < 16; ++i) sums[group][i][tid] = acc[0][i];
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (i / (16 / GROUPS) != group) continue;
      float sum = sums[0][i][tid];
#pragma unroll
      for (int g = 1; g < GROUPS; ++g) sum += sums[g][i][tid];
      acc[0][i] = sum;
    }
  }
  // 32 lanes store 32 consecutive columns of a row: 64 or 128 contiguous bytes
#pragma unroll
  for (int jn = 0; jn < JN; ++jn) {
    const int column = n0 + wn + 32 * jn + n;
    if (column >= a.n_rows) continue;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if (GROUPS > 1 && i / (16 / GROUPS) != group) continue;
      const int row = m0 + wm + 8 * (i / 4) + 4 * h + i % 4;
      if (row >= a.m_rows) continue;
      const long long at = static_cast<long long>(row) * a.n_rows + column;
      if (a.out_bf16)
        static_cast<uint16_t*>(a.out)[at] = float_to_bf16_bits(acc[jn][i]);
      else
        static_cast<float*>(a.out)[at] = acc[jn][i];
    }
  }
}

// The same product with one wave a SIMD: four waves, arranged 2 x 2, each with a (32 JM) x
// (32 JN) part of a (64 JM) x (64 JN) tile, which read each operand from LDS for JN or
// JM matrix instructions.  Nothing but the wave itself fills the matrix pipe: a row of
// the left operand is read again for the next 16-element step as soon as it has been
// multiplied, the right operand a step ahead; the barrier of a stage stands before its
// last step (whose operands are in registers), and the fills of the stage after
// next, one every other instruction, follow it.  WORDS: the output starts at a word;
// between two words a store of four bf16 values is slower than four stores of one (16384
// x 768 -> 3072: 131 us, 116 so, 104 at a word; the choice is not made in the kernel, where
// it cost the others 5 %).
template <bool HALF, int JM, int JN, bool WORDS>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(1, 1)))
product_rows_wide_kernel(ProductArgs a) {
  constexpr int KS = kDepth / 16;
  constexpr int TM = 64 * JM, TN = 64 * JN;
  constexpr int kLeftBytes = TM * kDepth * 2, kStageBytes = kLeftBytes + TN * kDepth * 2;
  constexpr int LEFT_LOADS = TM * (kDepth / 8) / 256, RIGHT_LOADS = TN * (kDepth / 8) / 256;
  constexpr int LOADS = LEFT_LOADS + RIGHT_LOADS;
  static_assert(LOADS <= 3 * (JM * JN / 2), "the fills stand between the instructions of three steps");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kStageBytes];
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int h = lane / 32, n = lane % 32;
  const int n_tiles = (a.n_rows + TN - 1) / TN;
  const int logical = xcd_logical_block();
  const int m0 = __builtin_amdgcn_readfirstlane(logical / n_tiles * TM);
  const int n0 = __builtin_amdgcn_readfirstlane(logical % n_tiles * TN);
  const int wm = 32 * JM * (wave / 2), wn = 32 * JN * (wave % 2);
  // loads of a wave are eight rows apart, which keeps the swizzle: one lane offset.
  // Columns beyond the contraction are rows of their own to the descriptor; those of
  // the last stages read zeros or another row's start into a stage nobody reads.
  const int32x4 left = make_rsrc(a.left + static_cast<long long>(m0) * a.depth,
                                 static_cast<uint32_t>(static_cast<long long>(a.m_rows - m0) * a.depth * 2));
  const int32x4 right = make_rsrc(a.right + static_cast<long long>(n0) * a.depth,
                                  static_cast<uint32_t>(static_cast<long long>(a.n_rows - n0) * a.depth * 2));
  uint32_t fill_at[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i)
    fill_at[i] = i < LEFT_LOADS ? tile_fill_offset<kDepth>((wave * LEFT_LOADS + i) * 64 + lane, a.depth)
                                : tile_fill_offset<kDepth>((wave * RIGHT_LOADS + i - LEFT_LOADS) * 64 + lane, a.depth);
  const uint32_t left_stage = lds_address(lds) + wave * LEFT_LOADS * 1024;
  const uint32_t right_stage = lds_address(lds) + kLeftBytes + wave * RIGHT_LOADS * 1024;
  auto fill = [&](int stage, int i) {
    if (i < LEFT_LOADS)
      lds_fill_at<16>(left, left_stage + stage * kStageBytes + i * 1024, fill_at[i]);
    else
      lds_fill_at<16>(right, right_stage + stage * kStageBytes + (i - LEFT_LOADS) * 1024, fill_at[i]);
    fill_at[i] += kDepth * 2;
  };
  constexpr int kBlockStep = 32 * (kDepth / 8) * 16;
  int left_read[KS], right_read[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    left_read[ks] = tile_row_read<kDepth>(wm + n, 2 * ks + h);
    right_read[ks] = kLeftBytes + tile_row_read<kDepth>(wn + n, 2 * ks + h);
  }
  floatx16 acc[JM][JN];
#pragma unroll
  for (int jn = 0; jn < JN; ++jn) {
    const int column = n0 + wn + 32 * jn + n;
    const float start = (a.bias && column < a.n_rows) ? a.bias[column] : 0.0f;
#pragma unroll
    for (int jm = 0; jm < JM; ++jm)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[jm][jn][i] = start;
  }
  const int steps = a.depth / kDepth;
  uint4 l[JM], r[2][JN];
  auto read_left = [&](int stage, int ks, int j) {
    l[j] = *reinterpret_cast<const uint4*>(lds + left_read[ks] + stage * kStageBytes + j * kBlockStep);
  };
  auto read_right = [&](int stage, int ks, int j) {
    r[ks & 1][j] = *reinterpret_cast<const uint4*>(lds + right_read[ks] + stage * kStageBytes + j * kBlockStep);
  };
  // the products of step ks, the reads of step `next` of a stage behind their operands'
  // last use, and fills first .. first + JM JN / 2 - 1 of a stage between
  auto multiply = [&](int ks, int next_stage, int next, int fill_stage, int first) {
#pragma unroll
    for (int jm = 0; jm < JM; ++jm) {
#pragma unroll
      for (int jn = 0; jn < JN; ++jn) {
        const int i = jm * JN + jn;
        acc[jm][jn] = mma<HALF>(l[jm], r[ks & 1][jn], acc[jm][jn]);
        __builtin_amdgcn_sched_barrier(0);
        if (first >= 0 && i % 2 == 1 && first + i / 2 < LOADS) {
          fill(fill_stage, first + i / 2);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (jm == 0) read_right(next_stage, next, jn);
      }
      read_left(next_stage, next, jm);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr int PART = JM * JN / 2;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) fill(0, i);
  wait_loads<0>();
  lds_barrier();
#pragma unroll
  for (int j = 0; j < JN; ++j) read_right(0, 0, j);
#pragma unroll
  for (int j = 0; j < JM; ++j) read_left(0, 0, j);
#pragma unroll
  for (int i = 0; i < PART && i < LOADS; ++i) fill(1, i);
  __builtin_amdgcn_sched_barrier(0);
  for (int step = 0; step < steps; step += 2) {
#pragma unroll
    for (int stage = 0; stage < 2; ++stage) {
      if (stage == 1 && step + 1 >= steps) break;
      multiply(0, stage, 1, stage ^ 1, PART);
      multiply(1, stage, 2, stage ^ 1, 2 * PART);
      multiply(2, stage, 3, stage ^ 1, -1);
      // the next stage has landed, and every wave has read the last of this one
      wait_loads<0>();
      lds_barrier();
      multiply(3, stage ^ 1, 0, stage, 0);
    }
  }
  wait_loads<0>();  // no fill may land after the workgroup has given its LDS back
  if constexpr (!WORDS) {
#pragma unroll
    for (int jm = 0; jm < JM; ++jm)
#pragma unroll
      for (int jn = 0; jn < JN; ++jn) {
        const int column = n0 + wn + 32 * jn + n;
        if (column >= a.n_rows) continue;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int row = m0 + wm + 32 * jm + 8 * (i / 4) + 4 * h + i % 4;
          if (row < a.m_rows)
            static_cast<uint16_t*>(a.out)[static_cast<long long>(row) * a.n_rows + column] =
                float_to_bf16_bits(acc[jm][jn][i]);
        }
      }
    return;
  }
  // four rows of one column a lane -> four columns of one row: 128 (or 64) contiguous
  // bytes of eight rows a store
  const int row0 = m0 + wm + 4 * h + n % 4, column0 = n0 + wn + n / 4 * 4;
#pragma unroll
  for (int jm = 0; jm < JM; ++jm)
#pragma unroll
    for (int jn = 0; jn < JN; ++jn)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx16& c = acc[jm][jn];
        const float4 v = quad_transpose(make_float4(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]));
        const int row = row0 + 32 * jm + 8 * q, column = column0 + 32 * jn;
        if (row >= a.m_rows || column >= a.n_rows) continue;
        const long long at = static_cast<long long>(row) * a.n_rows + column;
        if (a.out_bf16)
          *reinterpret_cast<FourHalves*>(static_cast<uint16_t*>(a.out) + at) = {pack_bf16(v.x, v.y),
                                                                               pack_bf16(v.z, v.w)};
        else
          *reinterpret_cast<FourFloats*>(static_cast<float*>(a.out) + at) = {v.x, v.y, v.z, v.w};
      }
}

// A tile of a product: its size, the time of a 64-element step of one workgroup when a
// compute unit has it alone, and per workgroup when compute units are full, in units of
// 10 ns.
struct Tile {
  int rows, columns, alone, full;
};
constexpr Tile kWideTile = {256, 192, 108, 125};   // product_rows_wide_kernel
constexpr Tile kMediumTile = {64, 128, 58, 35};    // product_rows_kernel<2>
constexpr Tile kSmallTile = {64, 64, 50, 20};      // product_rows_kernel<1>

// The time of a product with one kind of tiles: its steps, and the filling of the first
// stages and the stores at about five of them, as often as compute units take turns.
long long product_time(const Tile& t, int rows, int columns, int slices, int steps) {
  constexpr long long kComputeUnits = 256;
  const long long tiles = 1LL * ((rows + t.rows - 1) / t.rows) * ((columns + t.columns - 1) / t.columns) * slices;
  const long long turns = (tiles + kComputeUnits - 1) / kComputeUnits;
  return (steps + 5LL) * std::max<long long>(t.alone, turns * t.full);
}

// 16384 x 768 -> 2304 and its input gradient take 72 and 53 us in wide tiles (89 and 75 in
// tiles of 128 x 128 or, with eight waves, 256 x 256); 4096 x 2304 -> 768 26 us in small
// ones (33, 64) and 500 rows of it 16 (28, 58).
template <bool HALF>
void launch_product_rows(hipStream_t s, const ProductArgs& p) {
  auto blocks = [&](const Tile& t) {
    return static_cast<unsigned>((p.m_rows + t.rows - 1) / t.rows) *
           static_cast<unsigned>((p.n_rows + t.columns - 1) / t.columns);
  };
  auto time = [&](const Tile& t) { return product_time(t, p.m_rows, p.n_rows, 1, p.depth / kDepth); };
  const long long wide = time(kWideTile), medium = time(kMediumTile), small = time(kSmallTile);
  if (wide <= medium && wide <= small) {
    if constexpr (!HALF) {  // FP32 activations have FP32 results
      if (p.out_bf16 && reinterpret_cast<uintptr_t>(p.out) % 4 != 0) {
        product_rows_wide_kernel<HALF, 4, 3, false><<<blocks(kWideTile), 256, 0, s>>>(p);
        return;
      }
    }
    product_rows_wide_kernel<HALF, 4, 3, true><<<blocks(kWideTile), 256, 0, s>>>(p);
  } else if (medium <= small) {
    product_rows_kernel<HALF, 2, 1><<<blocks(kMediumTile), kThreads, 0, s>>>(p);
  } else if (blocks(kSmallTile) <= 256) {
    product_rows_kernel<HALF, 1, 4><<<blocks(kSmallTile), 4 * kThreads, 0, s>>>(p);
  } else if (blocks(kSmallTile) <= 512) {
    product_rows_kernel<HALF, 1, 2><<<blocks(kSmallTile), 2 * kThreads, 0, s>>>(p);
  } else {
    product_rows_kernel<HALF, 1, 1><<<blocks(kSmallTile), kThreads, 0, s>>>(p);
  }
}

struct GramArgs {
  const uint16_t* left = nullptr;   // [rows, m_cols]
  const uint16_t* right = nullptr;  // [rows, n_cols]
  float* out = nullptr;             // [slices, m_cols, n_cols] partial sums
  int rows = 0, m_cols = 0, n_cols = 0, slices = 1;
};

// out[slice][m, n] = sum over the slice's rows r of left[r, m] right[r, n];
// m_cols and n_cols are multiples of 64.  A workgroup owns a 128 x 128 tile
// and one slice of the rows; both operands come from row-major [64 rows, 128]
// LDS tiles through the transpose read, 16 rows a contraction step.
template <bool HALF>
__global__ void __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(2, 2)))
product_columns_kernel(GramArgs a) {
  constexpr int kRows = 64;   // rows per LDS tile
  constexpr int kWidth = 128;
  constexpr int kBytes = kRows * kWidth * 2;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[4 * kBytes];
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int h = lane / 32, n = lane % 32;
  const int n_tiles = (a.n_cols + kWidth - 1) / kWidth, m_tiles = (a.m_cols + kWidth - 1) / kWidth;
  // The tiles of a slice read the same rows: neighbours share an XCD's L2.  Dealt out to all
  // of them, 16000 rows of 768 -> 768 took 39.8 us instead of 25.2; in wide tiles, 16384 rows
  // of 768 -> 2304, 62.2 instead of 57.5 (353 MB from beyond the L2).
  const int logical = xcd_contiguous_block();
  const int tile = logical % (n_tiles * m_tiles), slice = logical / (n_tiles * m_tiles);
  const int m0 = (tile / n_tiles) * kWidth, n0 = (tile % n_tiles) * kWidth;
  const int wm = 64 * (wave / 2), wn = 64 * (wave % 2);
  const int per_slice = ((a.rows + a.slices - 1) / a.slices + kRows - 1) / kRows * kRows;
  const int first = slice * per_slice, last = min(first + per_slice, a.rows);
  constexpr int LOADS = kRows * (kWidth / 8) / kThreads;  // 4
  uint32_t left_fill[LOADS], right_fill[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    left_fill[i] = tile_fill_offset<kWidth>((wave * LOADS + i) * 64 + lane, a.m_cols);
    right_fill[i] = tile_fill_offset<kWidth>((wave * LOADS + i) * 64 + lane, a.n_cols);
  }
  int left_read[2], right_read[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    left_read[j] = tile_transpose_read<kWidth>(lane, (wm + 32 * j) / 32);
    right_read[j] = tile_transpose_read<kWidth>(lane, (wn + 32 * j) / 32);
  }
  floatx16 acc[2][2];
#pragma unroll
  for (int jm = 0; jm < 2; ++jm)
#pragma unroll
    for (int jn = 0; jn < 2; ++jn)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[jm][jn][i] = 0.0f;
  // A tile may be wider than what is left of a row (widths are multiples of
  // 64, tiles 128 wide): those columns then hold the start of the next row,
  // which only reaches output elements that are not stored.  The descriptor
  // ends with row `last - 1`, so nothing is read beyond the slice.
  auto fill_tile = [&](unsigned char* tile, const uint16_t* matrix, int stride, int col0, int r0,
                       const uint32_t* offsets) {
    const long long begin = static_cast<long long>(r0) * stride + col0;
    const long long left_elements = static_cast<long long>(last) * stride - begin;
    const int32x4 rsrc = make_rsrc(
        matrix + begin, left_elements <= 0 ? 0u : static_cast<uint32_t>(left_elements * 2));
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      lds_fill<16>(rsrc, tile + (wave * LOADS + i) * 1024, offsets[i]);
  };
  auto fill_stage = [&](int step) {
    unsigned char* stage = lds + (step & 1) * 2 * kBytes;
    const int r0 = first + step * kRows;
    fill_tile(stage, a.left, a.m_cols, m0, r0, left_fill);
    fill_tile(stage + kBytes, a.right, a.n_cols, n0, r0, right_fill);
  };
  const int steps = first < last ? (last - first + kRows - 1) / kRows : 0;
  if (steps > 0) fill_stage(0);
  for (int step = 0; step < steps; ++step) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (step + 1 < steps) fill_stage(step + 1);
    const unsigned char* left_tile = lds + (step & 1) * 2 * kBytes;
    const unsigned char* right_tile = left_tile + kBytes;
#pragma unroll
    for (int s2 = 0; s2 < kRows / 16; ++s2) {
      uint4 l[2], r[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        l[j] = __builtin_bit_cast(uint4, tile_transposed_operand<kWidth>(left_tile, left_read[j], s2));
        r[j] = __builtin_bit_cast(uint4, tile_transposed_operand<kWidth>(right_tile, right_read[j], s2));
      }
#pragma unroll
      for (int jm = 0; jm < 2; ++jm)
#pragma unroll
        for (int jn = 0; jn < 2; ++jn) acc[jm][jn] = mma<HALF>(l[jm], r[jn], acc[jm][jn]);
    }
  }
  float* out = a.out + static_cast<long long>(slice) * a.m_cols * a.n_cols;
#pragma unroll
  for (int jm = 0; jm < 2; ++jm)
#pragma unroll
    for (int jn = 0; jn < 2; ++jn) {
      const int column = n0 + wn + 32 * jn + n;
      if (column >= a.n_cols) continue;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = m0 + wm + 32 * jm + 8 * (i / 4) + 4 * h + i % 4;
        if (row < a.m_cols) out[static_cast<long long>(row) * a.n_cols + column] = acc[jm][jn][i];
      }
    }
}

// The same in (64 JM) x (64 JN) tiles with one wave a SIMD, as product_rows_wide_kernel.
template <bool HALF, int JM, int JN>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(1, 1)))
product_columns_wide_kernel(GramArgs a) {
  constexpr int kRows = 64, KS = kRows / 16;
  constexpr int TM = 64 * JM, TN = 64 * JN;
  constexpr int kLeftBytes = kRows * TM * 2, kStageBytes = kLeftBytes + kRows * TN * 2;
  constexpr int LEFT_LOADS = kRows * (TM / 8) / 256, RIGHT_LOADS = kRows * (TN / 8) / 256;
  constexpr int LOADS = LEFT_LOADS + RIGHT_LOADS;
  static_assert(LOADS <= 3 * (JM * JN / 2), "the fills stand between the instructions of three steps");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kStageBytes];
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int h = lane / 32, n = lane % 32;
  const int n_tiles = (a.n_cols + TN - 1) / TN, m_tiles = (a.m_cols + TM - 1) / TM;
  const int logical = xcd_contiguous_block();
  const int tile = logical % (n_tiles * m_tiles);
  const int slice = __builtin_amdgcn_readfirstlane(logical / (n_tiles * m_tiles));
  const int m0 = __builtin_amdgcn_readfirstlane(tile / n_tiles * TM);
  const int n0 = __builtin_amdgcn_readfirstlane(tile % n_tiles * TN);
  const int wm = 32 * JM * (wave / 2), wn = 32 * JN * (wave % 2);
  const int per_slice = ((a.rows + a.slices - 1) / a.slices + kRows - 1) / kRows * kRows;
  const int first = slice * per_slice, last = min(first + per_slice, a.rows);
  const int steps = first < last ? (last - first + kRows - 1) / kRows : 0;
  // Columns beyond a matrix are the start of its next row, which only reaches output
  // elements that are not stored; rows beyond the slice read zeros.
  auto source = [&](const uint16_t* matrix, int stride, int col0) {
    const long long elements = static_cast<long long>(last - first) * stride - col0;
    return make_rsrc(matrix + static_cast<long long>(first) * stride + col0,
                     elements <= 0 ? 0u : static_cast<uint32_t>(elements * 2));
  };
  const int32x4 left = source(a.left, a.m_cols, m0), right = source(a.right, a.n_cols, n0);
  uint32_t fill_at[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i)
    fill_at[i] = i < LEFT_LOADS ? tile_fill_offset<TM>((wave * LEFT_LOADS + i) * 64 + lane, a.m_cols)
                                : tile_fill_offset<TN>((wave * RIGHT_LOADS + i - LEFT_LOADS) * 64 + lane, a.n_cols);
  const uint32_t left_stage = lds_address(lds) + wave * LEFT_LOADS * 1024;
  const uint32_t right_stage = lds_address(lds) + kLeftBytes + wave * RIGHT_LOADS * 1024;
  auto fill = [&](int stage, int i) {
    if (i < LEFT_LOADS)
      lds_fill_at<16>(left, left_stage + stage * kStageBytes + i * 1024, fill_at[i]);
    else
      lds_fill_at<16>(right, right_stage + stage * kStageBytes + (i - LEFT_LOADS) * 1024, fill_at[i]);
    fill_at[i] += kRows * 2 * (i < LEFT_LOADS ? a.m_cols : a.n_cols);
  };
  // blocks of 32 columns two apart share the swizzle
  int left_read[2], right_read[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    left_read[j] = tile_transpose_read<TM>(lane, wm / 32 + j);
    right_read[j] = kLeftBytes + tile_transpose_read<TN>(lane, wn / 32 + j);
  }
  floatx16 acc[JM][JN];
#pragma unroll
  for (int jm = 0; jm < JM; ++jm)
#pragma unroll
    for (int jn = 0; jn < JN; ++jn)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[jm][jn][i] = 0.0f;
  uint4 l[JM], r[2][JN];
  auto read_left = [&](int stage, int ks, int j) {
    l[j] = __builtin_bit_cast(uint4, tile_transposed_operand<TM>(lds + stage * kStageBytes + j / 2 * 128,
                                                                 left_read[j % 2], ks));
  };
  auto read_right = [&](int stage, int ks, int j) {
    r[ks & 1][j] = __builtin_bit_cast(uint4, tile_transposed_operand<TN>(lds + stage * kStageBytes + j / 2 * 128,
                                                                         right_read[j % 2], ks));
  };
  auto multiply = [&](int ks, int next_stage, int next, int fill_stage, int first_fill) {
#pragma unroll
    for (int jm = 0; jm < JM; ++jm) {
#pragma unroll
      for (int jn = 0; jn < JN; ++jn) {
        const int i = jm * JN + jn;
        acc[jm][jn] = mma<HALF>(l[jm], r[ks & 1][jn], acc[jm][jn]);
        __builtin_amdgcn_sched_barrier(0);
        if (first_fill >= 0 && i % 2 == 1 && first_fill + i / 2 < LOADS) {
          fill(fill_stage, first_fill + i / 2);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (jm == 0) read_right(next_stage, next, jn);
      }
      read_left(next_stage, next, jm);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr int PART = JM * JN / 2;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) fill(0, i);
  wait_loads<0>();
  lds_barrier();
#pragma unroll
  for (int j = 0; j < JN; ++j) read_right(0, 0, j);
#pragma unroll
  for (int j = 0; j < JM; ++j) read_left(0, 0, j);
#pragma unroll
  for (int i = 0; i < PART && i < LOADS; ++i) fill(1, i);
  __builtin_amdgcn_sched_barrier(0);
  for (int step = 0; step < steps; step += 2) {
#pragma unroll
    for (int stage = 0; stage < 2; ++stage) {
      if (stage == 1 && step + 1 >= steps) break;
      multiply(0, stage, 1, stage ^ 1, PART);
      multiply(1, stage, 2, stage ^ 1, 2 * PART);
      multiply(2, stage, 3, stage ^ 1, -1);
      wait_loads<0>();
      lds_barrier();
      multiply(3, stage ^ 1, 0, stage, 0);
    }
  }
  wait_loads<0>();  // no fill may land after the workgroup has given its LDS back
  float* out = a.out + static_cast<long long>(slice) * a.m_cols * a.n_cols;
  const int row0 = m0 + wm + 4 * h + n % 4, column0 = n0 + wn + n / 4 * 4;
#pragma unroll
  for (int jm = 0; jm < JM; ++jm)
#pragma unroll
    for (int jn = 0; jn < JN; ++jn)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx16& c = acc[jm][jn];
        const float4 v = quad_transpose(make_float4(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]));
        const int row = row0 + 32 * jm + 8 * q, column = column0 + 32 * jn;
        if (row < a.m_cols && column < a.n_cols)
          *reinterpret_cast<float4*>(out + static_cast<long long>(row) * a.n_cols + column) = v;
      }
}

// The ends of both weight gradients in one launch: the first blocks add the slices of the
// matrix gradient (ascending), four elements a thread, the rest the partitions of the
// bias gradient.
template <bool ALIGNED>
__global__ void __launch_bounds__(256)
sum_partials_kernel(const float* slices, long long elements, int count, float* d_matrix, int matrix_blocks,
                    const float* partitions, int parts, int width, float* d_bias) {
  if (static_cast<int>(blockIdx.x) >= matrix_blocks) {
    const int c = (blockIdx.x - matrix_blocks) * 256 + threadIdx.x;
    if (c >= width) return;
    float sum = 0.0f;
#pragma unroll 16
    for (int p = 0; p < parts; ++p) sum += partitions[static_cast<long long>(p) * width + c];
    d_bias[c] = sum;
    return;
  }
  const long long i = 4 * (blockIdx.x * 256LL + threadIdx.x);
  if (i >= elements) return;  // widths are multiples of 64
  float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll 4
  for (int s = 0; s < count; ++s) {
    const float4 v = *reinterpret_cast<const float4*>(slices + s * elements + i);
    sum.x += v.x, sum.y += v.y, sum.z += v.z, sum.w += v.w;
  }
  if constexpr (ALIGNED)
    *reinterpret_cast<float4*>(d_matrix + i) = sum;
  else
    d_matrix[i] = sum.x, d_matrix[i + 1] = sum.y, d_matrix[i + 2] = sum.z, d_matrix[i + 3] = sum.w;
}

// Column sums of [rows, width] in two levels with a fixed order
// (fully_connected.cc:198-247: 256-row partitions, then the partitions), and
// optionally the 16-bit copy of the same values: the gradient is read once
// for both.  A workgroup takes 64 columns of a 256-row partition; thread
// (lane, quad) = (tid / 16, tid % 16) adds rows lane, lane + 16, ... of four
// adjacent columns, and the sixteen lanes' sums are added in ascending order.  The
// blocks beyond `tiles` make the 16-bit copies of the matrix and of the input.
template <bool HALF>
__global__ void __launch_bounds__(256)
column_partial_kernel(const float* in, int rows, int width, float* partial, uint16_t* copy, int tiles,
                      const float* matrix, long long matrix_elements, uint16_t* matrix16,
                      const float* input, long long input_elements, uint16_t* input16) {
  if (static_cast<int>(blockIdx.x) >= tiles) {
    const long long index = (blockIdx.x - tiles) * 256LL + threadIdx.x, threads = (gridDim.x - tiles) * 256LL;
    convert_elements<HALF>(matrix, matrix_elements, matrix16, index, threads);
    convert_elements<HALF>(input, input_elements, input16, index, threads);
    return;
  }
  __shared__ float lanes[16][64];
  const int quad = threadIdx.x % 16, lane = threadIdx.x / 16;
  const int across = (width + 63) / 64, column_block = blockIdx.x % across, part = blockIdx.x / across;
  const int c = column_block * 64 + quad * 4;
  const int r0 = part * kBiasRows, r1 = min(r0 + kBiasRows, rows);
  float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (width % 4 == 0 && c < width) {
    // all of a thread's rows are requested together (four at a time: 13.1 us at 256
    // rows of 2304, 55 at 16384; 8.0 and 47 so)
    float4 values[kBiasRows / 16];
#pragma unroll
    for (int i = 0; i < kBiasRows / 16; ++i)
      values[i] = *reinterpret_cast<const float4*>(
          in + static_cast<long long>(min(r0 + lane + 16 * i, r1 - 1)) * width + c);
#pragma unroll
    for (int i = 0; i < kBiasRows / 16; ++i) {
      const int r = r0 + lane + 16 * i;
      if (r >= r1) break;
      const long long at = static_cast<long long>(r) * width + c;
      const float4 value = values[i];
      sum[0] += value.x, sum[1] += value.y, sum[2] += value.z, sum[3] += value.w;
      if (copy) {
        ushort4 out;
        out.x = to_operand<HALF>(value.x), out.y = to_operand<HALF>(value.y);
        out.z = to_operand<HALF>(value.z), out.w = to_operand<HALF>(value.w);
        *reinterpret_cast<ushort4*>(copy + at) = out;
      }
    }
  } else {
    for (int r = r0 + lane; r < r1; r += 16)
      for (int e = 0; e < 4; ++e)
        if (c + e < width) {
          const float value = in[static_cast<long long>(r) * width + c + e];
          sum[e] += value;
          if (copy) copy[static_cast<long long>(r) * width + c + e] = to_operand<HALF>(value);
        }
  }
  for (int e = 0; e < 4; ++e) lanes[lane][quad * 4 + e] = sum[e];
  __syncthreads();
  const int column = column_block * 64 + threadIdx.x;
  if (threadIdx.x < 64 && column < width) {
    float total = lanes[0][threadIdx.x];
    for (int l = 1; l < 16; ++l) total += lanes[l][threadIdx.x];
    partial[static_cast<long long>(part) * width + column] = total;
  }
}

// Any shape: one thread per output element, operands rounded like the matrix
// cores' and summed in FP32 in ascending order.
//   mode 0: out[r, o] = bias[o] + sum_i x[r, i] w[i, o]   (x in `dtype`)
//   mode 1: out[r, i] = sum_o g[r, o] w[i, o]
//   mode 2: out[i, o] = sum_r x[r, i] g[r, o]
template <bool HALF>
__global__ void __launch_bounds__(256)
generic_dense_kernel(int mode, int dtype, const void* x, const float* w, const float* g,
                     const float* bias, int rows, int input_dim, int output_dim, void* out) {
  const long long i = blockIdx.x * 256LL + threadIdx.x;
  const long long total = mode == 0   ? 1LL * rows * output_dim
                          : mode == 1 ? 1LL * rows * input_dim
                                      : 1LL * input_dim * output_dim;
  if (i >= total) return;
  auto activation = [&](long long at) {
    return operand_value<HALF>(load_element(x, at, dtype));
  };
  float sum = 0.0f;
  if (mode == 0) {
    const int r = static_cast<int>(i / output_dim), o = static_cast<int>(i % output_dim);
    sum = bias[o];
    for (int k = 0; k < input_dim; ++k)
      sum += activation(1LL * r * input_dim + k) * operand_value<HALF>(w[1LL * k * output_dim + o]);
    store_element(out, i, dtype, sum);
    return;
  }
  if (mode == 1) {
    const int r = static_cast<int>(i / input_dim), k = static_cast<int>(i % input_dim);
    for (int o = 0; o < output_dim; ++o)
      sum += operand_value<HALF>(g[1LL * r * output_dim + o]) *
             operand_value<HALF>(w[1LL * k * output_dim + o]);
  } else {
    const int k = static_cast<int>(i / output_dim), o = static_cast<int>(i % output_dim);
    for (int r = 0; r < rows; ++r)
      sum += activation(1LL * r * input_dim + k) * operand_value<HALF>(g[1LL * r * output_dim + o]);
  }
  static_cast<float*>(out)[i] = sum;
}

unsigned blocks_for(long long elements, long long cap = 1LL << 20) {
  const long long blocks = (elements + 255) / 256;
  return static_cast<unsigned>(blocks < cap ? blocks : cap);
}

bool matrix_cores(int input_dim, int output_dim) {
  return input_dim % 64 == 0 && output_dim % 64 == 0;
}

// How the matrix gradient is computed: the kind of tiles and the slices of the rows, as
// many as fill the compute units once (one wide tile each or two of 128 x 128) but of
// at least 256 rows, whose partial sums are written and read again at about 5 TB/s.
struct WeightPlan {
  bool wide = false;
  int slices = 1;
};
WeightPlan weight_plan(int rows, int input_dim, int output_dim) {
  constexpr Tile kWide = {256, 192, 115, 130}, kSquare = {128, 128, 75, 60};
  auto plan = [&](const Tile& t, int resident, long long* time) {
    const long long tiles = 1LL * ((input_dim + t.rows - 1) / t.rows) * ((output_dim + t.columns - 1) / t.columns);
    const long long slices =
        std::max(1LL, std::min<long long>(resident / tiles, (rows + 255) / 256));
    const int steps = static_cast<int>(((rows + slices - 1) / slices + 63) / 64);
    *time = product_time(t, input_dim, output_dim, static_cast<int>(slices), steps) +
            (slices > 1 ? 8LL * slices * input_dim * output_dim / 50000 : 0);
    return static_cast<int>(slices);
  };
  long long wide_time = 0, square_time = 0;
  const int wide = plan(kWide, 256, &wide_time), square = plan(kSquare, 512, &square_time);
  return wide_time <= square_time ? WeightPlan{true, wide} : WeightPlan{false, square};
}

struct Layout {
  size_t matrix16, input16, gradient16, partial, bias_partial, total;
};

Layout layout(int dtype, int rows, int input_dim, int output_dim) {
  Layout l{};
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t offset = at;
    at += align_up(bytes, 256);
    return offset;
  };
  const size_t r = rows, in = input_dim, out = output_dim;
  l.matrix16 = take(in * out * 2);
  l.input16 = take(dtype == PLUTO_HIP_F32 ? r * in * 2 : 0);
  l.gradient16 = take(r * out * 2);
  l.partial = take(static_cast<size_t>(weight_plan(rows, input_dim, output_dim).slices) * in * out * 4);
  l.bias_partial = take(static_cast<size_t>((rows + kBiasRows - 1) / kBiasRows) * out * 4);
  l.total = at;
  return l;
}

template <bool HALF>
int forward(hipStream_t s, int dtype, const void* input, const float* matrix, const float* bias,
            int rows, int input_dim, int output_dim, void* output, char* scratch) {
  if (!matrix_cores(input_dim, output_dim)) {
    generic_dense_kernel<HALF><<<blocks_for(1LL * rows * output_dim), 256, 0, s>>>(
        0, dtype, input, matrix, nullptr, bias, rows, input_dim, output_dim, output);
    return launch_status();
  }
  const Layout l = layout(dtype, rows, input_dim, output_dim);
  uint16_t* matrix16 = reinterpret_cast<uint16_t*>(scratch + l.matrix16);  // w^T [out, in]
  const bool copied = dtype == PLUTO_HIP_F32;
  uint16_t* copy = reinterpret_cast<uint16_t*>(scratch + l.input16);
  const uint16_t* input16 = copied ? copy : static_cast<const uint16_t*>(input);
  const int tiles = (input_dim / 64) * (output_dim / 64);
  const long long elements = copied ? 1LL * rows * input_dim : 0;
  convert_forward_kernel<HALF><<<tiles + (copied ? blocks_for(elements / 8, 2048) : 0), 256, 0, s>>>(
      matrix, input_dim, output_dim, matrix16, tiles, static_cast<const float*>(input), elements, copy);
  ProductArgs p;
  p.left = input16;
  p.right = matrix16;
  p.bias = bias;
  p.out = output;
  p.m_rows = rows;
  p.n_rows = output_dim;
  p.depth = input_dim;
  p.out_bf16 = dtype == PLUTO_HIP_BF16;
  launch_product_rows<HALF>(s, p);
  return launch_status();
}

template <bool HALF>
int backward(hipStream_t s, int dtype, const void* input, const float* matrix,
             const float* d_output, int rows, int input_dim, int output_dim, float* d_input,
             float* d_matrix, float* d_bias, char* scratch) {
  const Layout l = layout(dtype, rows, input_dim, output_dim);
  // bias gradient: 256-row partitions, then the partitions in order
  float* bias_partial = reinterpret_cast<float*>(scratch + l.bias_partial);
  const int parts = (rows + kBiasRows - 1) / kBiasRows;
  const bool cores = matrix_cores(input_dim, output_dim);
  uint16_t* gradient16 = reinterpret_cast<uint16_t*>(scratch + l.gradient16);  // dy [rows, out]
  uint16_t* matrix16 = reinterpret_cast<uint16_t*>(scratch + l.matrix16);  // w [in, out]
  const bool copied = cores && dtype == PLUTO_HIP_F32;
  uint16_t* copy = reinterpret_cast<uint16_t*>(scratch + l.input16);
  const long long elements = 1LL * input_dim * output_dim;
  const long long matrix_elements = cores ? elements : 0, input_elements = copied ? 1LL * rows * input_dim : 0;
  const int tiles = (output_dim + 63) / 64 * parts;
  const long long converted = matrix_elements + input_elements;
  column_partial_kernel<HALF>
      <<<tiles + (converted > 0 ? blocks_for(converted / 8, 2048) : 0), 256, 0, s>>>(
          d_output, rows, output_dim, bias_partial, cores ? gradient16 : nullptr, tiles, matrix, matrix_elements,
          matrix16, static_cast<const float*>(input), input_elements, copy);
  const int bias_blocks = (output_dim + 255) / 256;
  if (!cores) {
    sum_partials_kernel<false><<<bias_blocks, 256, 0, s>>>(nullptr, 0, 0, nullptr, 0, bias_partial, parts,
                                                           output_dim, d_bias);
    generic_dense_kernel<HALF><<<blocks_for(1LL * rows * input_dim), 256, 0, s>>>(
        1, dtype, input, matrix, d_output, nullptr, rows, input_dim, output_dim, d_input);
    generic_dense_kernel<HALF><<<blocks_for(elements), 256, 0, s>>>(
        2, dtype, input, matrix, d_output, nullptr, rows, input_dim, output_dim, d_matrix);
    return launch_status();
  }
  const uint16_t* input16 = copied ? copy : static_cast<const uint16_t*>(input);
  // dx[r, i] = sum_o dy[r, o] w[i, o]
  ProductArgs p;
  p.left = gradient16;
  p.right = matrix16;
  p.out = d_input;
  p.m_rows = rows;
  p.n_rows = input_dim;
  p.depth = output_dim;
  launch_product_rows<HALF>(s, p);
  int status = launch_status();
  if (status != 0) return status;
  // dw[i, o] = sum_r x[r, i] dy[r, o], the rows in slices
  GramArgs g;
  g.left = input16;
  g.right = gradient16;
  g.rows = rows;
  g.m_cols = input_dim;
  g.n_cols = output_dim;
  const WeightPlan plan = weight_plan(rows, input_dim, output_dim);
  g.slices = plan.slices;
  g.out = g.slices == 1 ? d_matrix : reinterpret_cast<float*>(scratch + l.partial);
  auto weight_tiles = [&](int m, int n) {
    return static_cast<unsigned>((input_dim + m - 1) / m) * static_cast<unsigned>((output_dim + n - 1) / n);
  };
  const bool aligned = reinterpret_cast<uintptr_t>(d_matrix) % 16 == 0;
  if (plan.wide && (aligned || g.slices > 1))
    product_columns_wide_kernel<HALF, 4, 3><<<weight_tiles(256, 192) * g.slices, 256, 0, s>>>(g);
  else
    product_columns_kernel<HALF><<<weight_tiles(128, 128) * g.slices, kThreads, 0, s>>>(g);
  status = launch_status();
  if (status != 0) return status;
  const int matrix_blocks = g.slices == 1 ? 0 : static_cast<int>((elements / 4 + 255) / 256);
  const unsigned blocks = matrix_blocks + bias_blocks;
  if (aligned)
    sum_partials_kernel<true><<<blocks, 256, 0, s>>>(g.out, elements, g.slices, d_matrix, matrix_blocks,
                                                     bias_partial, parts, output_dim, d_bias);
  else
    sum_partials_kernel<false><<<blocks, 256, 0, s>>>(g.out, elements, g.slices, d_matrix, matrix_blocks,
                                                      bias_partial, parts, output_dim, d_bias);
  return launch_status();
}

}  // namespace

size_t dense_workspace_bytes(int dtype, int rows, int input_dim, int output_dim) {
  return layout(dtype, rows, input_dim, output_dim).total;
}

int launch_dense_forward(hipStream_t stream, int dtype, const void* input, const float* matrix,
                         const float* bias, int rows, int input_dim, int output_dim, void* output,
                         void* workspace) {
  char* scratch = static_cast<char*>(workspace);
  return dtype == PLUTO_HIP_BF16
             ? forward<false>(stream, dtype, input, matrix, bias, rows, input_dim, output_dim,
                              output, scratch)
             : forward<true>(stream, dtype, input, matrix, bias, rows, input_dim, output_dim,
                             output, scratch);
}

int launch_dense_backward(hipStream_t stream, int dtype, const void* input, const float* matrix,
                          const float* d_output, int rows, int input_dim, int output_dim,
                          float* d_input, float* d_matrix, float* d_bias, void* workspace) {
  char* scratch = static_cast<char*>(workspace);
  return dtype == PLUTO_HIP_BF16
             ? backward<false>(stream, dtype, input, matrix, d_output, rows, input_dim,
                               output_dim, d_input, d_matrix, d_bias, scratch)
             : backward<true>(stream, dtype, input, matrix, d_output, rows, input_dim, output_dim,
                              d_input, d_matrix, d_bias, scratch);
}

}  // namespace pluto_hip

using namespace pluto_hip;

extern "C" {

static int validate_dense(int dtype, int rows, int input_dim, int output_dim) {
  // fully_connected.cc:318-338: BF16 and FP32 activations are the trainable types
  if (dtype != PLUTO_HIP_F32 && dtype != PLUTO_HIP_BF16) return PLUTO_HIP_EUNSUPPORTED;
  if (rows <= 0 || input_dim <= 0 || output_dim <= 0) return PLUTO_HIP_EINVAL;
  if (static_cast<long long>(rows) * input_dim > 0x7fffffffLL ||
      static_cast<long long>(rows) * output_dim > 0x7fffffffLL ||
      static_cast<long long>(input_dim) * output_dim > 0x7fffffffLL)
    return PLUTO_HIP_ERANGE;
  return 0;
}

size_t pluto_hip_dense_workspace_bytes(int dtype, int rows, int input_dim, int output_dim) {
  if (validate_dense(dtype, rows, input_dim, output_dim) != 0) return 0;
  return dense_workspace_bytes(dtype, rows, input_dim, output_dim);
}

int pluto_hip_dense_forward(void* stream, int dtype, const void* input, const float* matrix,
                            const float* bias, int rows, int input_dim, int output_dim,
                            void* output, void* workspace, size_t workspace_bytes) {
  const int status = validate_dense(dtype, rows, input_dim, output_dim);
  if (status != 0) return status;
  if (!input || !matrix || !bias || !output) return PLUTO_HIP_EINVAL;
  if (!workspace || workspace_bytes < dense_workspace_bytes(dtype, rows, input_dim, output_dim))
    return PLUTO_HIP_EWORKSPACE;
  return launch_dense_forward(static_cast<hipStream_t>(stream), dtype, input, matrix, bias, rows,
                              input_dim, output_dim, output, workspace);
}

int pluto_hip_dense_backward(void* stream, int dtype, const void* input, const float* matrix,
                             const float* d_output, int rows, int input_dim, int output_dim,
                             float* d_input, float* d_matrix, float* d_bias, void* workspace,
                             size_t workspace_bytes) {
  const int status = validate_dense(dtype, rows, input_dim, output_dim);
  if (status != 0) return status;
  if (!input || !matrix || !d_output || !d_input || !d_matrix || !d_bias) return PLUTO_HIP_EINVAL;
  if (!workspace || workspace_bytes < dense_workspace_bytes(dtype, rows, input_dim, output_dim))
    return PLUTO_HIP_EWORKSPACE;
  return launch_dense_backward(static_cast<hipStream_t>(stream), dtype, input, matrix, d_output,
                               rows, input_dim, output_dim, d_input, d_matrix, d_bias, workspace);
}

}  // extern "C"
