// FP32 attention on the bf16 matrix cores: what the forward and backward kernels share.
//
// A workgroup of four waves owns 32 rows of one side, kept in LDS as pieces in operand
// order; every wave streams tiles of 32 rows of the other side of its own through an area
// of LDS, where a tile lies as pieces and is read both ways: by rows for the score
// products, transposed for those that contract over rows.
#pragma once

#include "bf16_pieces.h"

namespace pluto_hip {

// What pieces cannot hold: an infinity less itself is no number, and a number from 2^128 -
// 2^119 on rounds to one; a product beyond the range has parts of either sign beyond it.
// All of these leave an accumulator that is not finite (what a zero weight hides of them
// is hidden in either arithmetic), so a wave looks at its results when it is done, and
// where one is not finite repeats its tiles on the FP32 matrix instruction, which gives the
// infinity, the weight of zero for a score of minus infinity or the finite product.
template <int N>
__device__ inline bool all_finite(const floatx16 (&acc)[N]) {
  float probe[8] = {};  // zero times what is finite
#pragma unroll
  for (int k = 0; k < N; ++k)
#pragma unroll
    for (int i = 0; i < 16; ++i) probe[i % 8] = __builtin_fmaf(acc[k][i], 0.0f, probe[i % 8]);
  return ((probe[0] + probe[1]) + (probe[2] + probe[3])) + ((probe[4] + probe[5]) + (probe[6] + probe[7])) == 0.0f;
}

// Accumulator registers 8 s2 .. 8 s2 + 7 as a B operand.
__device__ inline Pieces split_accumulator(const floatx16& acc, int s2) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = acc[8 * s2 + e];
  return split_eight(x);
}

template <int D>
struct F32Rows {
  static constexpr int KS = D / 16, DB = D / 32;
  static constexpr int kWidth = D < 64 ? 64 : D;  // of a row in LDS: the swizzle permutes eight pieces
  static constexpr int kOwnBytes = 3 * KS * 1024;
  static constexpr int kPartBytes = 32 * kWidth * 2, kAreaBytes = 3 * kPartBytes;

  // A tile as it arrives: four channels a lane, whole rows next to each other (a lane's
  // channels of an operand at a time, 32 rows an access, the loads took twice as long as
  // everything else).
  static constexpr int kLanes = D / 4, kLoads = 32 * kLanes / 64;
  struct Raw {
    float4 v[kLoads];
  };
  // Rows `row_stride` floats apart, `valid` of which exist; the others read as zero.
  __device__ __forceinline__ static void request(Raw& raw, const float* base, long long row_stride, int valid, int lane) {
    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(base), 0,
        valid <= 0 ? 0 : static_cast<int>(((min(valid, 32) - 1) * row_stride + D) * 4), 0x00020000);
    const int bytes = static_cast<int>(row_stride * 4);
    int at = lane / kLanes * bytes + lane % kLanes * 16;
    asm volatile("" : "+v"(at));  // one register kept over a loop, not one a load
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      raw.v[i] = __builtin_bit_cast(
          float4, __builtin_amdgcn_raw_buffer_load_b128(rows, at + i * (64 / kLanes) * bytes, 0, 0));
  }

  // The workgroup's own rows: operand (part, ks) is 1 KiB, a lane's eight channels together.
  __device__ __forceinline__ static void keep_own(unsigned char* own, int ks, int lane, const Pieces& p) {
#pragma unroll
    for (int part = 0; part < 3; ++part)
      *reinterpret_cast<bf16x8*>(own + ((part * KS + ks) * 64 + lane) * 16) = p.part[part];
  }
  __device__ __forceinline__ static Pieces read_own(const unsigned char* own, int ks, int lane) {
    Pieces p;
#pragma unroll
    for (int part = 0; part < 3; ++part)
      p.part[part] = *reinterpret_cast<const bf16x8*>(own + ((part * KS + ks) * 64 + lane) * 16);
    return p;
  }

  // The wave's area: row-major tiles of the three pieces.  A wave's accesses to LDS are
  // carried out in order, so a tile may follow another without a wait.
  __device__ __forceinline__ static void keep(unsigned char* area, const Raw& raw, int lane) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int row = i * (64 / kLanes) + lane / kLanes, piece = lane % kLanes;
      const int at = tile_row_read<kWidth>(row, piece / 2) + piece % 2 * 8;
      uint32_t words[3][2];
      split_pair(raw.v[i].x, raw.v[i].y, words[0][0], words[1][0], words[2][0]);
      split_pair(raw.v[i].z, raw.v[i].w, words[0][1], words[1][1], words[2][1]);
#pragma unroll
      for (int part = 0; part < 3; ++part)
        *reinterpret_cast<uint2*>(area + part * kPartBytes + at) = make_uint2(words[part][0], words[part][1]);
    }
  }
  // A operand: row n, channels 16 ks + 8 h .. + 7
  __device__ __forceinline__ static Pieces read_rows(const unsigned char* area, int ks, int lane) {
    const int at = tile_row_read<kWidth>(lane % 32, 2 * ks + lane / 32);
    Pieces p;
#pragma unroll
    for (int part = 0; part < 3; ++part)
      p.part[part] = *reinterpret_cast<const bf16x8*>(area + part * kPartBytes + at);
    return p;
  }
  // A operand: channels 32 db + n of rows 16 s2 .. in accumulator order
  __device__ __forceinline__ static Pieces read_transposed(const unsigned char* area, int db, int s2, int lane) {
    Pieces p;
#pragma unroll
    for (int part = 0; part < 3; ++part)
      p.part[part] =
          tile_transposed_operand<kWidth>(area + part * kPartBytes, tile_transpose_read<kWidth>(lane, db), s2);
    return p;
  }

  // The two kinds of product on the FP32 matrix instruction, straight from memory; rows
  // beyond `valid` count as zero.  Rows of a tile by the lane's row of the other side:
  __device__ __forceinline__ static floatx16 exact_rows(const float* tile, long long row_stride, int valid,
                                                           const float* other, int lane) {
    const int h = lane / 32, n = lane % 32;
    const float* row = tile + (n < valid ? n : 0) * row_stride;
    floatx16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
#pragma unroll 4
    for (int c = 0; c < D; c += 2) {
      const float x = row[c + h];
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(n < valid ? x : 0.0f, other[c + h], acc, 0, 0, 0);
    }
    return acc;
  }
  // A tile's rows, transposed, by an accumulator.
  __device__ __forceinline__ static void exact_transposed(floatx16 (&acc)[DB], const float* tile, long long row_stride,
                                                             int valid, const floatx16& other, int lane) {
    const int h = lane / 32, n = lane % 32;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 8 * (i / 4) + 4 * h + i % 4;
      const float* channels = tile + (row < valid ? row : 0) * row_stride + n;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const float x = channels[32 * db];
        acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(row < valid ? x : 0.0f, other[i], acc[db], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
};

}  // namespace pluto_hip
