// Causal attention of head width 256 to FP32 accuracy on the bf16 matrix cores:
// the attention core of the whole-sequence Qwen layer's backward
// (src/llm/layers/qwen_attention.cc:146-199, and the forward it repeats, :68-119)
// where queries, keys and values are bf16 and everything derived from them is
// FP32.
//
// An FP32 number is the exact sum of three bf16 numbers (8 + 8 + 8 mantissa
// bits).  A product of a bf16 and an FP32 operand is therefore three bf16 matrix
// products with FP32 sums, and one of two FP32 operands six: the terms left out
// are 2^-24 of the product, what one FP32 rounding costs.  Per 32 x 32 block of
// scores in products of depth 256: S 1, P V 3 (forward); S 1, dP 3, dQ 3; and
// S 1, dP 3, dK 3, dV 6.  At sixteen times the rate of the FP32 matrix
// instruction that is a third of its time.  T = 1024, 24/4 heads: 0.03, 0.06
// and 0.12 ms for the three kernels, where the kernels that multiply one element
// at a time took 3.9, 5.0 and 7.4 ms.
//
// Shape of the kernels as in flash_bwd_mfma.hip: four waves of 32 queries (keys)
// each, tiles of 32 rows of the other side through two LDS stages filled by
// direct-to-LDS loads, one barrier a tile, score tiles oriented so that their
// accumulator is the B operand of the product that follows.
#include "attn_split_mfma.h"

#include "mfma_tile.h"

namespace pluto_hip {
namespace {

constexpr int D = kSplitHeadDim;
constexpr int kThreads = 256, kRows = 32, kOwned = 128;
constexpr int KCH = D / 8, KS = D / 16, DB = D / 32;
constexpr int kLoads = kRows * KCH / kThreads;
constexpr int kTileBytes = kRows * D * 2;

struct Pieces {
  bf16x8 part[3];
};

// Accumulator registers 8 s2 .. 8 s2 + 7 as three B operands that add up to them.
__device__ inline Pieces split_accumulator(const floatx16& acc, int s2) {
  uint32_t words[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float first = acc[8 * s2 + 2 * i], second = acc[8 * s2 + 2 * i + 1];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const uint32_t bits = pack_bf16(first, second);
      words[p][i] = bits;
      first -= __uint_as_float(bits << 16);
      second -= __uint_as_float(bits & 0xffff0000u);
    }
  }
  Pieces out;
#pragma unroll
  for (int p = 0; p < 3; ++p)
    out.part[p] = as_bf16x8(make_uint4(words[p][0], words[p][1], words[p][2], words[p][3]));
  return out;
}

__device__ inline floatx16 zero16() {
  floatx16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.0f;
  return z;
}

__device__ inline void load_row_operand(const uint16_t* row, int h, bf16x8 (&out)[KS]) {
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    out[ks] = as_bf16x8(*reinterpret_cast<const uint4*>(row + 16 * ks + 8 * h));
}

// Where a wave's lanes read a tile, and what they fetch of one.
struct TileAccess {
  uint32_t fill[kLoads];
  int row_read[KS], tr_read[DB];
  __device__ TileAccess(int wave, int lane, long long row_stride) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      fill[i] = tile_fill_offset<D>((wave * kLoads + i) * 64 + lane, row_stride);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) row_read[ks] = tile_row_read<D>(lane % 32, 2 * ks + lane / 32);
#pragma unroll
    for (int db = 0; db < DB; ++db) tr_read[db] = tile_transpose_read<D>(lane, db);
  }
};
__device__ inline bf16x8 row_operand(const unsigned char* tile, int offset) {
  return as_bf16x8(*reinterpret_cast<const uint4*>(tile + offset));
}

__device__ inline void stage_ready() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
split_forward_kernel(SplitArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2][2 * kTileBytes];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const int T = a.length, head = blockIdx.x % a.heads;
  const int q0 = ((T + kOwned - 1) / kOwned - 1 - static_cast<int>(blockIdx.x) / a.heads) * kOwned;
  const long long q_row = 1LL * a.heads * D, kv_row = 1LL * (a.heads / a.group) * D;
  const uint16_t* k_base = a.k + head / a.group * D;
  const uint16_t* v_base = a.v + head / a.group * D;
  const int first_query = q0 + 32 * wave, query = first_query + n, query_load = min(query, T - 1);
  const TileAccess at(wave, lane, kv_row);
  const int tiles = (min(q0 + kOwned, T) - 1) / kRows + 1;
  auto fill = [&](int tile) {
    unsigned char* stage = lds[tile & 1];
    const int k0 = tile * kRows;
    tile_fill<D, kLoads>(stage, wave, k_base + k0 * kv_row, kv_row, k0, T, at.fill);
    tile_fill<D, kLoads>(stage + kTileBytes, wave, v_base + k0 * kv_row, kv_row, k0, T, at.fill);
  };
  fill(0);
  bf16x8 qf[KS];
  load_row_operand(a.q + query_load * q_row + head * D, h, qf);
  floatx16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = zero16();
  float running_max = kMasked, running_sum = 0.0f;  // of the scaled scores
  for (int tile = 0; tile < tiles; ++tile) {
    const int k0 = tile * kRows;
    stage_ready();
    if (tile + 1 < tiles) fill(tile + 1);
    if (k0 > first_query + 31) continue;  // every key follows my queries
    const unsigned char* k_tile = lds[tile & 1];
    const unsigned char* v_tile = k_tile + kTileBytes;
    floatx16 s = zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) s = mfma32(row_operand(k_tile, at.row_read[ks]), qf[ks], s);
    // register i = (key k0 + 8(i/4) + 4h + i%4, query n)
    const int limit = query_load - k0 - 4 * h;
    float tile_max = kMasked;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = 8 * (i / 4) + (i % 4) > limit ? kMasked : s[i] * a.scale;
      tile_max = fmaxf(tile_max, s[i]);
    }
    const float new_max = fmaxf(running_max, half_swap_max(tile_max));
    const float correction = __builtin_amdgcn_exp2f((running_max - new_max) * kLog2e);
    running_max = new_max;
    float tile_sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = s[i] == kMasked ? 0.0f : __builtin_amdgcn_exp2f((s[i] - new_max) * kLog2e);
      tile_sum += s[i];
    }
    running_sum = running_sum * correction + half_swap_sum(tile_sum);
    if (__any(correction != 1.0f)) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] *= correction;
    }
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const Pieces p = split_accumulator(s, s2);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const bf16x8 vt = tile_transposed_operand<D>(v_tile, at.tr_read[db], s2);
#pragma unroll
        for (int part = 2; part >= 0; --part) o[db] = mfma32(vt, p.part[part], o[db]);
      }
    }
  }
  if (query >= T) return;
  const float inverse = 1.0f / (running_sum > 0.0f ? running_sum : 1.0f);
  float* out = a.core + query * q_row + head * D + 4 * h;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<float4*>(out + 32 * db + 8 * j) =
          make_float4(o[db][4 * j] * inverse, o[db][4 * j + 1] * inverse,
                      o[db][4 * j + 2] * inverse, o[db][4 * j + 3] * inverse);
  if (h == 0) {
    a.maxima[1LL * head * T + query] = running_max;
    a.inverses[1LL * head * T + query] = inverse;
  }
}

// 32 lanes a row, eight channels a lane; a workgroup walks 64 rows of one head.
// WIDE: the caller's tensors are 16-byte aligned.
template <bool WIDE>
__global__ void __launch_bounds__(256)
split_gate_kernel(SplitArgs a, const uint16_t* __restrict__ qg, const float* __restrict__ dy,
                  float* __restrict__ dqg) {
  const int c = 8 * (threadIdx.x % 32), head = blockIdx.y;
  for (int i = 0; i < 64; i += 8) {
    const int row = blockIdx.x * 64 + i + threadIdx.x / 32;
    if (row >= a.length) continue;  // a row's lanes leave together
    const long long unit = 1LL * row * a.heads + head;
    float gate[8], core[8], grad[8], d_gate[8];
    load8<WIDE>(qg + (unit * 2 + 1) * D + c, gate);
    load8<WIDE>(dy + unit * D + c, grad);
    load8<true>(a.core + unit * D + c, core);
    float delta = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float sigmoid = 1.0f / (1.0f + expf(-gate[e]));
      d_gate[e] = grad[e] * round_to_bf16(core[e]) * sigmoid * (1.0f - sigmoid);
      grad[e] *= round_to_bf16(sigmoid);
      delta += grad[e] * core[e];
    }
    store8<WIDE>(dqg + (unit * 2 + 1) * D + c, d_gate);
#pragma unroll
    for (int part = 0; part < 3; ++part) {
      uint32_t words[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        words[k] = pack_bf16(grad[2 * k], grad[2 * k + 1]);
        grad[2 * k] -= __uint_as_float(words[k] << 16);
        grad[2 * k + 1] -= __uint_as_float(words[k] & 0xffff0000u);
      }
      *reinterpret_cast<uint4*>(a.d_core + part * a.piece + unit * D + c) =
          make_uint4(words[0], words[1], words[2], words[3]);
    }
#pragma unroll
    for (int offset = 16; offset > 0; offset >>= 1) delta += __shfl_xor(delta, offset, 64);
    if (c == 0) a.deltas[1LL * head * a.length + row] = delta;
  }
}

__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
split_dq_kernel(SplitArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2][2 * kTileBytes];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const int T = a.length, head = blockIdx.x % a.heads;
  const int q0 = ((T + kOwned - 1) / kOwned - 1 - static_cast<int>(blockIdx.x) / a.heads) * kOwned;
  const long long q_row = 1LL * a.heads * D, kv_row = 1LL * (a.heads / a.group) * D;
  const uint16_t* k_base = a.k + head / a.group * D;
  const uint16_t* v_base = a.v + head / a.group * D;
  const int first_query = q0 + 32 * wave, query = first_query + n, query_load = min(query, T - 1);
  const TileAccess at(wave, lane, kv_row);
  const int tiles = (min(q0 + kOwned, T) - 1) / kRows + 1;
  auto fill = [&](int tile) {
    unsigned char* stage = lds[tile & 1];
    const int k0 = tile * kRows;
    tile_fill<D, kLoads>(stage, wave, k_base + k0 * kv_row, kv_row, k0, T, at.fill);
    tile_fill<D, kLoads>(stage + kTileBytes, wave, v_base + k0 * kv_row, kv_row, k0, T, at.fill);
  };
  fill(0);
  bf16x8 qf[KS], gf[3][KS];
  load_row_operand(a.q + query_load * q_row + head * D, h, qf);
#pragma unroll
  for (int part = 0; part < 3; ++part)
    load_row_operand(a.d_core + part * a.piece + query_load * q_row + head * D, h, gf[part]);
  const long long stat = 1LL * head * T + query_load;
  const float maximum = a.maxima[stat], inverse = a.inverses[stat], delta = a.deltas[stat];
  floatx16 dq[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dq[db] = zero16();
  for (int tile = 0; tile < tiles; ++tile) {
    const int k0 = tile * kRows;
    stage_ready();
    if (tile + 1 < tiles) fill(tile + 1);
    if (k0 > first_query + 31) continue;
    const unsigned char* k_tile = lds[tile & 1];
    const unsigned char* v_tile = k_tile + kTileBytes;
    floatx16 s = zero16(), dp = zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s = mfma32(row_operand(k_tile, at.row_read[ks]), qf[ks], s);
      const bf16x8 vf = row_operand(v_tile, at.row_read[ks]);
#pragma unroll
      for (int part = 2; part >= 0; --part) dp = mfma32(vf, gf[part][ks], dp);
    }
    const int limit = query_load - k0 - 4 * h;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p =
          __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.scale, -maximum) * kLog2e) * inverse;
      s[i] = 8 * (i / 4) + (i % 4) > limit ? 0.0f : p * (dp[i] - delta);
    }
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const Pieces ds = split_accumulator(s, s2);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const bf16x8 kt = tile_transposed_operand<D>(k_tile, at.tr_read[db], s2);
#pragma unroll
        for (int part = 2; part >= 0; --part) dq[db] = mfma32(kt, ds.part[part], dq[db]);
      }
    }
  }
  if (query >= T) return;
  float* out = a.dq + query * q_row + head * D + 4 * h;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<float4*>(out + 32 * db + 8 * j) =
          make_float4(dq[db][4 * j] * a.scale, dq[db][4 * j + 1] * a.scale,
                      dq[db][4 * j + 2] * a.scale, dq[db][4 * j + 3] * a.scale);
}

// Stage: Q tile, the three tiles of dC, and 64 floats each of the rows' maxima,
// inverse normalizers and deltas.
constexpr int kDkvStageBytes = 4 * kTileBytes + 1024;

__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
split_dkv_kernel(SplitArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kDkvStageBytes];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const int T = a.length, head = blockIdx.x % a.heads;
  const int k0 = static_cast<int>(blockIdx.x) / a.heads * kOwned;
  const long long q_row = 1LL * a.heads * D, kv_row = 1LL * (a.heads / a.group) * D;
  const int first_key = k0 + 32 * wave, key = first_key + n, key_load = min(key, T - 1);
  const TileAccess at(wave, lane, q_row);
  const int first_tile = k0 / kRows, tiles = (T + kRows - 1) / kRows;
  auto fill = [&](int tile) {
    unsigned char* stage = lds + (tile & 1) * kDkvStageBytes;
    const int q0 = tile * kRows;
    tile_fill<D, kLoads>(stage, wave, a.q + head * D + q0 * q_row, q_row, q0, T, at.fill);
#pragma unroll
    for (int part = 0; part < 3; ++part)
      tile_fill<D, kLoads>(stage + (1 + part) * kTileBytes, wave,
                           a.d_core + part * a.piece + head * D + q0 * q_row, q_row, q0, T, at.fill);
    if (wave < 3) {
      const float* source = wave == 0 ? a.maxima : wave == 1 ? a.inverses : a.deltas;
      const int32x4 rsrc = make_rsrc(source + 1LL * head * T + q0, static_cast<uint32_t>(T - q0) * 4u);
      lds_fill<4>(rsrc, stage + 4 * kTileBytes + wave * 256, lane * 4);
    }
  };
  fill(first_tile);
  bf16x8 kf[KS], vf[KS];
  load_row_operand(a.k + key_load * kv_row + head / a.group * D, h, kf);
  load_row_operand(a.v + key_load * kv_row + head / a.group * D, h, vf);
  floatx16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dk[db] = dv[db] = zero16();
  for (int tile = first_tile; tile < tiles; ++tile) {
    const int q0 = tile * kRows;
    stage_ready();
    if (tile + 1 < tiles) fill(tile + 1);
    if (q0 + 31 < first_key) continue;  // every query precedes my keys
    const unsigned char* q_tile = lds + (tile & 1) * kDkvStageBytes;
    const unsigned char* g_tile = q_tile + kTileBytes;
    const float* stats = reinterpret_cast<const float*>(q_tile + 4 * kTileBytes);
    floatx16 s = zero16(), dp = zero16();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      s = mfma32(row_operand(q_tile, at.row_read[ks]), kf[ks], s);
#pragma unroll
      for (int part = 2; part >= 0; --part)
        dp = mfma32(row_operand(g_tile + part * kTileBytes, at.row_read[ks]), vf[ks], dp);
    }
    // register i = (query q0 + 8(i/4) + 4h + i%4, key n)
    const int first = key - q0 - 4 * h, last = T - 1 - q0 - 4 * h;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 maximum = *reinterpret_cast<const float4*>(stats + 8 * j + 4 * h);
      const float4 inverse = *reinterpret_cast<const float4*>(stats + 64 + 8 * j + 4 * h);
      const float4 delta = *reinterpret_cast<const float4*>(stats + 128 + 8 * j + 4 * h);
      const float m[4] = {maximum.x, maximum.y, maximum.z, maximum.w};
      const float r[4] = {inverse.x, inverse.y, inverse.z, inverse.w};
      const float dl[4] = {delta.x, delta.y, delta.z, delta.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * j + e, local = 8 * j + e;
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.scale, -m[e]) * kLog2e) * r[e];
        const bool hidden = (local < first) | (local > last);
        s[i] = hidden ? 0.0f : p;
        dp[i] = hidden ? 0.0f : p * (dp[i] - dl[e]);
      }
    }
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const Pieces p = split_accumulator(s, s2), ds = split_accumulator(dp, s2);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const bf16x8 qt = tile_transposed_operand<D>(q_tile, at.tr_read[db], s2);
#pragma unroll
        for (int part = 2; part >= 0; --part) dk[db] = mfma32(qt, ds.part[part], dk[db]);
#pragma unroll
        for (int gp = 2; gp >= 0; --gp) {
          const bf16x8 gt = tile_transposed_operand<D>(g_tile + gp * kTileBytes, at.tr_read[db], s2);
#pragma unroll
          for (int part = 2 - gp; part >= 0; --part) dv[db] = mfma32(gt, p.part[part], dv[db]);
        }
      }
    }
  }
  if (key >= T) return;
  const long long out = key * q_row + head * D + 4 * h;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      *reinterpret_cast<float4*>(a.dk + out + 32 * db + 8 * j) =
          make_float4(dk[db][4 * j] * a.scale, dk[db][4 * j + 1] * a.scale,
                      dk[db][4 * j + 2] * a.scale, dk[db][4 * j + 3] * a.scale);
      *reinterpret_cast<float4*>(a.dv + out + 32 * db + 8 * j) =
          make_float4(dv[db][4 * j], dv[db][4 * j + 1], dv[db][4 * j + 2], dv[db][4 * j + 3]);
    }
}

unsigned tile_grid(const SplitArgs& a) {
  return static_cast<unsigned>((a.length + kOwned - 1) / kOwned) * a.heads;
}

}  // namespace

bool split_attention_supported(int length, int heads, int head_dim) {
  // a tensor's rows are addressed through 32-bit buffer offsets
  return head_dim == D && 1LL * length * heads * D * 2 < (1LL << 31) && heads <= 65535;
}

int launch_split_forward(hipStream_t stream, const SplitArgs& a) {
  split_forward_kernel<<<tile_grid(a), kThreads, 0, stream>>>(a);
  return launch_status();
}

int launch_split_gate(hipStream_t stream, const SplitArgs& a, const void* qg, const float* dy,
                      float* dqg) {
  const dim3 grid((a.length + 63) / 64, a.heads);
  const auto* gates = static_cast<const uint16_t*>(qg);
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  if (aligned(qg) && aligned(dy) && aligned(dqg))
    split_gate_kernel<true><<<grid, 256, 0, stream>>>(a, gates, dy, dqg);
  else
    split_gate_kernel<false><<<grid, 256, 0, stream>>>(a, gates, dy, dqg);
  return launch_status();
}

int launch_split_backward(hipStream_t stream, const SplitArgs& a) {
  if (kernel_enabled(kQueryKernel)) split_dq_kernel<<<tile_grid(a), kThreads, 0, stream>>>(a);
  const int status = launch_status();
  if (status != 0) return status;
  if (kernel_enabled(kMainKernel)) split_dkv_kernel<<<tile_grid(a), kThreads, 0, stream>>>(a);
  return launch_status();
}

}  // namespace pluto_hip
