// FP32 matrix products on the bf16 matrix cores.
//
// An FP32 number is the sum of three bf16 numbers (8 + 8 + 8 mantissa bits), and a
// product of two such sums is six bf16 matrix products with FP32 sums: the three left
// out are 2^-25 of the product, less than one FP32 rounding.  Six v_mfma_f32_32x32x16_bf16
// take 192 cycles where the FP32 instruction needs 512 for the same depth, six
// v_mfma_f32_16x16x32_bf16 96 where it needs 256; making the pieces costs 44 cycles of
// vector instructions a pair of numbers.
// An infinity has no such pieces, and a number from 2^128 - 2^119 on, which rounds to one, not
// by rounding alone: what the kernels do about them stands beside them.
#pragma once

#include "mfma_tile.h"

namespace pluto_hip {

struct Pieces {
  bf16x8 part[3];
};

// acc + a b, smallest products first.
__device__ inline floatx16 mma_pieces(const Pieces& a, const Pieces& b, floatx16 acc) {
#pragma unroll
  for (int i = 2; i >= 0; --i)
#pragma unroll
    for (int j = 2 - i; j >= 0; --j) acc = mfma32(a.part[i], b.part[j], acc);
  return acc;
}

__device__ inline floatx4 mfma16(bf16x8 a, bf16x8 b, floatx4 acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}
// Two numbers as the packed words of their pieces.
__device__ inline void split_pair(float first, float second, uint32_t& high, uint32_t& middle, uint32_t& low) {
  high = pack_bf16(first, second);
  first -= __uint_as_float(high << 16);
  second -= __uint_as_float(high & 0xffff0000u);
  middle = pack_bf16(first, second);
  first -= __uint_as_float(middle << 16);
  second -= __uint_as_float(middle & 0xffff0000u);
  low = pack_bf16(first, second);
}
// Eight numbers' pieces in eleven steps of four instructions that do not wait for each
// other: an instruction that waits for the one before it takes twice the four cycles of
// one that does not, so the four pairs go side by side.
struct Splitter {
  static constexpr int kSteps = 11;
  float rest[8], taken[8];
  uint32_t words[3][4];
  __device__ Splitter(float4 a, float4 b) : rest{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w} {}
  // `step` is known at compile time; pin: here, not where the compiler would rather have it
  __device__ void operator()(int step, bool pin = false) {
    const int part = step / 5, what = step % 5;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (what == 0) {
        words[part][i] = pack_bf16(rest[2 * i], rest[2 * i + 1]);
      } else if (what <= 2) {
        const int e = 4 * (what - 1) + i;
        taken[e] = __uint_as_float(e % 2 == 0 ? words[part][e / 2] << 16 : words[part][e / 2] & 0xffff0000u);
      } else {
        rest[4 * (what - 3) + i] -= taken[4 * (what - 3) + i];
      }
    }
    auto keep = [](auto& a, auto& b, auto& c, auto& d) { asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d)); };
    if (!pin) return;
    if (what == 0) keep(words[part][0], words[part][1], words[part][2], words[part][3]);
    if (what == 1) keep(taken[0], taken[1], taken[2], taken[3]);
    if (what == 2) keep(taken[4], taken[5], taken[6], taken[7]);
    if (what == 3) keep(rest[0], rest[1], rest[2], rest[3]);
    if (what == 4) keep(rest[4], rest[5], rest[6], rest[7]);
  }
  __device__ Pieces pieces() const {
    Pieces out;
#pragma unroll
    for (int p = 0; p < 3; ++p)
      out.part[p] = as_bf16x8(make_uint4(words[p][0], words[p][1], words[p][2], words[p][3]));
    return out;
  }
};
__device__ inline Pieces split_eight(const float (&x)[8]) {
  Splitter split(make_float4(x[0], x[1], x[2], x[3]), make_float4(x[4], x[5], x[6], x[7]));
#pragma unroll
  for (int i = 0; i < Splitter::kSteps; ++i) split(i);
  return split.pieces();
}
__device__ inline Pieces split_eight(float4 a, float4 b) {
  const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  return split_eight(x);
}
}  // namespace pluto_hip
