// LDS tiles of the FP32 attention kernels: a wave fills its own and reads them both
// ways, rows for the score products and single channels for the others.
#pragma once

#include "mfma_tile.h"

namespace pluto_hip {

// 32 rows of D floats in LDS, 16-byte piece c of row r at slot c ^ swizzle(r):
// the lanes of a row read (32 rows, same piece) spread over the banks.
template <int D>
struct F32Tile {
  static constexpr int kPieces = D / 4;
  static constexpr int kBytes = 32 * D * 4;
  static constexpr int kFillOps = kBytes / 1024;  // vector-memory operations of one fill
  __device__ static int swizzle(int row) { return row & (kPieces < 16 ? kPieces - 1 : 15); }
  // Queues the fill from global rows `row_bytes` apart, `valid` of which exist
  // (the rest read as zero).
  __device__ static void fill(unsigned char* tile, const float* base, long long row_stride,
                              int valid, int lane) {
    const int32x4 rsrc = make_rsrc(
        base, valid <= 0 ? 0u : static_cast<uint32_t>((min(valid, 32) - 1) * row_stride + D) * 4u);
#pragma unroll
    for (int i = 0; i < kBytes / 1024; ++i) {
      const int at = i * 64 + lane, row = at / kPieces, slot = at % kPieces;
      lds_fill<16>(rsrc, tile + i * 1024,
                   static_cast<uint32_t>(row * row_stride * 4 + (slot ^ swizzle(row)) * 16));
    }
  }
  // The same through registers, a tile ahead.
  struct Held {
    float4 v[kBytes / 1024];
  };
  __device__ static void request(Held& held, const float* base, long long row_stride, int valid,
                                 int lane) {
    const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(base), 0,
        valid <= 0 ? 0 : static_cast<int>(((min(valid, 32) - 1) * row_stride + D) * 4), 0x00020000);
#pragma unroll
    for (int i = 0; i < kBytes / 1024; ++i) {
      const int at = i * 64 + lane, row = at / kPieces, slot = at % kPieces;
      held.v[i] = __builtin_bit_cast(
          float4, __builtin_amdgcn_raw_buffer_load_b128(
                      rows, static_cast<int>(row * row_stride * 4) + (slot ^ swizzle(row)) * 16, 0, 0));
    }
  }
  __device__ static void place(unsigned char* tile, const Held& held, int lane) {
#pragma unroll
    for (int i = 0; i < kBytes / 1024; ++i)
      *reinterpret_cast<float4*>(tile + i * 1024 + lane * 16) = held.v[i];
  }
  __device__ static float4 row_piece(const unsigned char* tile, int row, int piece) {
    return *reinterpret_cast<const float4*>(tile + (row * kPieces + (piece ^ swizzle(row))) * 16);
  }
  __device__ static float element(const unsigned char* tile, int row, int channel) {
    return *reinterpret_cast<const float*>(
        tile + (row * kPieces + ((channel / 4) ^ swizzle(row))) * 16 + (channel % 4) * 4);
  }
};

// The lane's half (channels h D/2 ..) of one row.
template <int HALF>
__device__ inline void load_half_row(const float* row, float* out) {
#pragma unroll
  for (int j = 0; j < HALF / 4; ++j) {
    const float4 v = reinterpret_cast<const float4*>(row)[j];
    out[4 * j] = v.x; out[4 * j + 1] = v.y; out[4 * j + 2] = v.z; out[4 * j + 3] = v.w;
  }
}

// Until all but the last YOUNGER vector-memory operations of the wave are done.
template <int YOUNGER = 0>
__device__ inline void wait_fills() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");
}
__device__ inline void wait_reads() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

}  // namespace pluto_hip
