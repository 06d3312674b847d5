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
// instruction that is a third of its time.  T = 1024, 24/4 heads: 0.05, 0.07
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
constexpr int kThreads = 256, kRows = 32;
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

// Where a wave's lanes read a tile, and what they fetch of one.  The swizzle
// permutes pieces within groups of eight, so operand addresses repeat every 128
// bytes of a row and four (two) registers serve all of them.
struct TileAccess {
  uint32_t fill[kLoads];
  int row_read[4], tr_read[2];
  __device__ TileAccess(int wave, int lane, long long row_stride) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
      fill[i] = tile_fill_offset<D>((wave * kLoads + i) * 64 + lane, row_stride);
#pragma unroll
    for (int i = 0; i < 4; ++i) row_read[i] = tile_row_read<D>(lane % 32, 2 * i + lane / 32);
#pragma unroll
    for (int i = 0; i < 2; ++i) tr_read[i] = tile_transpose_read<D>(lane, i);
  }
  // A operand: row n of the tile, contraction step ks
  __device__ bf16x8 row(const unsigned char* tile, int ks) const {
    return as_bf16x8(*reinterpret_cast<const uint4*>(tile + row_read[ks % 4] + ks / 4 * 128));
  }
  // A operand: channels 32 db + n of rows 16 s2 ..
  __device__ bf16x8 transposed(const unsigned char* tile, int db, int s2) const {
    return tile_transposed_operand<D>(tile + db / 2 * 128, tr_read[db % 2], s2);
  }
};

// Nothing moves across: the operands of a step are requested before the matrix
// instructions of the step before it, one step ahead of their use.  (Left to
// itself the compiler requests an operand and waits for it before every one to
// three matrix instructions: 282 us for dK/dV at T = 1024, 24 heads.)
__device__ inline void fence_schedule() { __builtin_amdgcn_sched_barrier(0); }

__device__ inline void stage_ready() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// The two query-owned kernels: a workgroup owns 64 queries, waves 0 and 1 the two
// halves at even key tiles, waves 2 and 3 the same at odd ones, and the upper
// waves' results are added in at the end.  One wave a SIMD has nothing to cover
// the chain scores -> softmax -> products of a tile; at T = 1024 the longest chain
// is what the kernel takes, and this halves it (forward 79 -> 52 us, dQ 103 -> 70).
constexpr int kQueries = 64;
constexpr int kQueryStageBytes = 4 * kTileBytes;  // K and V of two tiles
struct QueryWave {
  int head, half, parity, steps, first_query, query, query_load;
  __device__ QueryWave(const SplitArgs& a, int wave, int n) {
    head = blockIdx.x % a.heads;
    const int q0 = ((a.length + kQueries - 1) / kQueries - 1 - static_cast<int>(blockIdx.x) / a.heads) * kQueries;
    half = wave % 2;
    parity = wave / 2;
    steps = ((min(q0 + kQueries, a.length) - 1) / kRows) / 2 + 1;  // two tiles each
    first_query = q0 + 32 * half;
    query = first_query + n;
    query_load = min(query, a.length - 1);
  }
};
// Queues the fill of step's two tiles: K, V of the even one, K, V of the odd one.
__device__ inline void fill_query_stage(const SplitArgs& a, unsigned char* lds, int step, int wave,
                                        int head, const uint32_t* offsets) {
  const long long kv_row = 1LL * (a.heads / a.group) * D;
  const long long column = head / a.group * D;
  unsigned char* stage = lds + (step & 1) * kQueryStageBytes;
#pragma unroll
  for (int tile = 0; tile < 2; ++tile) {
    const int k0 = (2 * step + tile) * kRows;
    tile_fill<D, kLoads>(stage + 2 * tile * kTileBytes, wave, a.k + column + k0 * kv_row, kv_row, k0,
                         a.length, offsets);
    tile_fill<D, kLoads>(stage + (2 * tile + 1) * kTileBytes, wave, a.v + column + k0 * kv_row,
                         kv_row, k0, a.length, offsets);
  }
}
// The accumulators of the upper waves into LDS, 32 KiB each.
__device__ inline void store_upper(unsigned char* lds, int half, int lane, const floatx16 (&acc)[DB]) {
  float4* area = reinterpret_cast<float4*>(lds + half * 2 * kTileBytes);
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      area[(4 * db + j) * 64 + lane] =
          make_float4(acc[db][4 * j], acc[db][4 * j + 1], acc[db][4 * j + 2], acc[db][4 * j + 3]);
}
__device__ inline float4 load_upper(const unsigned char* lds, int half, int lane, int piece) {
  return reinterpret_cast<const float4*>(lds + half * 2 * kTileBytes)[piece * 64 + lane];
}

__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
split_forward_kernel(SplitArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kQueryStageBytes];
  __shared__ float upper_stats[2][2][64];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const QueryWave w(a, wave, n);
  const int T = a.length, query = w.query, query_load = w.query_load, head = w.head;
  const long long q_row = 1LL * a.heads * D;
  const TileAccess at(wave, lane, 1LL * (a.heads / a.group) * D);
  fill_query_stage(a, lds, 0, wave, head, at.fill);
  bf16x8 qf[KS];
  load_row_operand(a.q + query_load * q_row + head * D, h, qf);
  floatx16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = zero16();
  float running_max = kMasked, running_sum = 0.0f;  // of the scaled scores
  for (int step = 0; step < w.steps; ++step) {
    const int k0 = (2 * step + w.parity) * kRows;
    stage_ready();
    if (step + 1 < w.steps) fill_query_stage(a, lds, step + 1, wave, head, at.fill);
    if (k0 > w.first_query + 31) continue;  // every key follows my queries
    const unsigned char* k_tile = lds + (step & 1) * kQueryStageBytes + w.parity * 2 * kTileBytes;
    const unsigned char* v_tile = k_tile + kTileBytes;
    floatx16 s = zero16();
    {
      bf16x8 kf[2][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) kf[0][i] = at.row(k_tile, i);
#pragma unroll
      for (int g = 0; g < KS / 4; ++g) {
        if (g + 1 < KS / 4)
#pragma unroll
          for (int i = 0; i < 4; ++i) kf[(g + 1) % 2][i] = at.row(k_tile, 4 * (g + 1) + i);
        fence_schedule();
#pragma unroll
        for (int i = 0; i < 4; ++i) s = mfma32(kf[g % 2][i], qf[4 * g + i], s);
        fence_schedule();
      }
    }
    bf16x8 vt[3];
    vt[0] = at.transposed(v_tile, 0, 0);
    vt[1] = at.transposed(v_tile, 1, 0);
    fence_schedule();
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
        const int at_step = s2 * DB + db;
        if (at_step + 2 < 2 * DB)
          vt[(at_step + 2) % 3] = at.transposed(v_tile, (at_step + 2) % DB, (at_step + 2) / DB);
        fence_schedule();
#pragma unroll
        for (int part = 2; part >= 0; --part) o[db] = mfma32(vt[at_step % 3], p.part[part], o[db]);
        fence_schedule();
      }
    }
  }
  __syncthreads();  // nobody reads the stages any more
  if (w.parity == 1) {
    store_upper(lds, w.half, lane, o);
    upper_stats[w.half][0][lane] = running_max;
    upper_stats[w.half][1][lane] = running_sum;
  }
  __syncthreads();
  if (w.parity == 1 || query >= T) return;
  // a wave without tiles contributes weight 2^(kMasked - maximum) = 0
  const float upper_max = upper_stats[w.half][0][lane];
  const float maximum = fmaxf(running_max, upper_max);
  const float own = __builtin_amdgcn_exp2f((running_max - maximum) * kLog2e);
  const float other = __builtin_amdgcn_exp2f((upper_max - maximum) * kLog2e);
  const float sum = running_sum * own + upper_stats[w.half][1][lane] * other;
  const float inverse = 1.0f / (sum > 0.0f ? sum : 1.0f);
  float* out = a.core + query * q_row + head * D + 4 * h;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 u = load_upper(lds, w.half, lane, 4 * db + j);
      *reinterpret_cast<float4*>(out + 32 * db + 8 * j) =
          make_float4((o[db][4 * j] * own + u.x * other) * inverse,
                      (o[db][4 * j + 1] * own + u.y * other) * inverse,
                      (o[db][4 * j + 2] * own + u.z * other) * inverse,
                      (o[db][4 * j + 3] * own + u.w * other) * inverse);
    }
  if (h == 0) {
    a.maxima[1LL * head * T + query] = maximum;
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
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kQueryStageBytes];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const QueryWave w(a, wave, n);
  const int T = a.length, query = w.query, query_load = w.query_load, head = w.head;
  const long long q_row = 1LL * a.heads * D;
  const TileAccess at(wave, lane, 1LL * (a.heads / a.group) * D);
  fill_query_stage(a, lds, 0, wave, head, at.fill);
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
  for (int step = 0; step < w.steps; ++step) {
    const int k0 = (2 * step + w.parity) * kRows;
    stage_ready();
    if (step + 1 < w.steps) fill_query_stage(a, lds, step + 1, wave, head, at.fill);
    if (k0 > w.first_query + 31) continue;  // every key follows my queries
    const unsigned char* k_tile = lds + (step & 1) * kQueryStageBytes + w.parity * 2 * kTileBytes;
    const unsigned char* v_tile = k_tile + kTileBytes;
    floatx16 s = zero16(), dp = zero16();
    bf16x8 kf[3], vf[3];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      kf[i] = at.row(k_tile, i);
      vf[i] = at.row(v_tile, i);
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      if (ks + 2 < KS) {
        kf[(ks + 2) % 3] = at.row(k_tile, ks + 2);
        vf[(ks + 2) % 3] = at.row(v_tile, ks + 2);
      }
      fence_schedule();
      s = mfma32(kf[ks % 3], qf[ks], s);
#pragma unroll
      for (int part = 2; part >= 0; --part) dp = mfma32(vf[ks % 3], gf[part][ks], dp);
      fence_schedule();
    }
    bf16x8 kt[3];
    kt[0] = at.transposed(k_tile, 0, 0);
    kt[1] = at.transposed(k_tile, 1, 0);
    fence_schedule();
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
        const int at_step = s2 * DB + db;
        if (at_step + 2 < 2 * DB)
          kt[(at_step + 2) % 3] = at.transposed(k_tile, (at_step + 2) % DB, (at_step + 2) / DB);
        fence_schedule();
#pragma unroll
        for (int part = 2; part >= 0; --part) dq[db] = mfma32(kt[at_step % 3], ds.part[part], dq[db]);
        fence_schedule();
      }
    }
  }
  __syncthreads();  // nobody reads the stages any more
  if (w.parity == 1) store_upper(lds, w.half, lane, dq);
  __syncthreads();
  if (w.parity == 1 || query >= T) return;
  float* out = a.dq + query * q_row + head * D + 4 * h;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 u = load_upper(lds, w.half, lane, 4 * db + j);
      *reinterpret_cast<float4*>(out + 32 * db + 8 * j) =
          make_float4((dq[db][4 * j] + u.x) * a.scale, (dq[db][4 * j + 1] + u.y) * a.scale,
                      (dq[db][4 * j + 2] + u.z) * a.scale, (dq[db][4 * j + 3] + u.w) * a.scale);
    }
}

constexpr int kKeys = 128;  // of a workgroup of the key-owned kernel
// Stage: Q tile, the three tiles of dC, and 64 floats each of the rows' maxima,
// inverse normalizers and deltas.
constexpr int kDkvStageBytes = 4 * kTileBytes + 1024;

// dK or dV of 128 keys: both in one workgroup need 256 accumulator registers a
// lane and leave none for requests ahead of their use.  Apart they repeat the
// 16 of 112 products that make the scores, and there are twice as many
// workgroups, of equal length, which short sequences need.
template <bool VALUES>
__device__ __forceinline__ void split_key_owned(const SplitArgs& a, unsigned char* lds, int head,
                                                int k0) {
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const int T = a.length;
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
  bf16x8 kf[KS], vf[VALUES ? 1 : KS];
  load_row_operand(a.k + key_load * kv_row + head / a.group * D, h, kf);
  if constexpr (!VALUES) load_row_operand(a.v + key_load * kv_row + head / a.group * D, h, vf);
  floatx16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = zero16();
  for (int tile = first_tile; tile < tiles; ++tile) {
    const int q0 = tile * kRows;
    stage_ready();
    if (tile + 1 < tiles) fill(tile + 1);
    if (q0 + 31 < first_key) continue;  // every query precedes my keys
    const unsigned char* q_tile = lds + (tile & 1) * kDkvStageBytes;
    const unsigned char* g_tile = q_tile + kTileBytes;
    const float* stats = reinterpret_cast<const float*>(q_tile + 4 * kTileBytes);
    floatx16 s = zero16(), dp = zero16();
    if constexpr (VALUES) {
      bf16x8 qa[2][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) qa[0][i] = at.row(q_tile, i);
#pragma unroll
      for (int g = 0; g < KS / 4; ++g) {
        if (g + 1 < KS / 4)
#pragma unroll
          for (int i = 0; i < 4; ++i) qa[(g + 1) % 2][i] = at.row(q_tile, 4 * (g + 1) + i);
        fence_schedule();
#pragma unroll
        for (int i = 0; i < 4; ++i) s = mfma32(qa[g % 2][i], kf[4 * g + i], s);
        fence_schedule();
      }
    } else {
      bf16x8 qa[3], ga[3][3];
      auto request = [&](int ks) {
        qa[ks % 3] = at.row(q_tile, ks);
#pragma unroll
        for (int part = 0; part < 3; ++part)
          ga[ks % 3][part] = at.row(g_tile + part * kTileBytes, ks);
      };
      request(0);
      request(1);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (ks + 2 < KS) request(ks + 2);
        fence_schedule();
        s = mfma32(qa[ks % 3], kf[ks], s);
#pragma unroll
        for (int part = 2; part >= 0; --part) dp = mfma32(ga[ks % 3][part], vf[ks], dp);
        fence_schedule();
      }
    }
    // transposed operands of step (s2, db): dC's pieces for dV, Q for dK
    constexpr int kAhead = VALUES ? 1 : 2, kParts = VALUES ? 3 : 1;
    bf16x8 t[kAhead + 1][kParts];
    auto request_transposed = [&](int step) {
#pragma unroll
      for (int part = 0; part < kParts; ++part)
        t[step % (kAhead + 1)][part] = at.transposed(VALUES ? g_tile + part * kTileBytes : q_tile,
                                                     step % DB, step / DB);
    };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) request_transposed(i);
    fence_schedule();
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
        float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.scale, -m[e]) * kLog2e) * r[e];
        if constexpr (!VALUES) p *= dp[i] - dl[e];
        s[i] = ((local < first) | (local > last)) ? 0.0f : p;
      }
    }
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const Pieces p = split_accumulator(s, s2);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const int step = s2 * DB + db;
        if (step + kAhead < 2 * DB) request_transposed(step + kAhead);
        fence_schedule();
#pragma unroll
        for (int gp = kParts - 1; gp >= 0; --gp)
#pragma unroll
          for (int part = 2 - gp; part >= 0; --part)
            acc[db] = mfma32(t[step % (kAhead + 1)][gp], p.part[part], acc[db]);
        fence_schedule();
      }
    }
  }
  if (key >= T) return;
  const float factor = VALUES ? 1.0f : a.scale;
  float* out = (VALUES ? a.dv : a.dk) + key * q_row + head * D + 4 * h;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<float4*>(out + 32 * db + 8 * j) =
          make_float4(acc[db][4 * j] * factor, acc[db][4 * j + 1] * factor,
                      acc[db][4 * j + 2] * factor, acc[db][4 * j + 3] * factor);
}

__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
split_dkv_kernel(SplitArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kDkvStageBytes];
  const int unit = blockIdx.x % (2 * a.heads), k0 = static_cast<int>(blockIdx.x) / (2 * a.heads) * kKeys;
  if (unit < a.heads)
    split_key_owned<true>(a, lds, unit, k0);
  else
    split_key_owned<false>(a, lds, unit - a.heads, k0);
}

unsigned tile_grid(const SplitArgs& a, int owned) {
  return static_cast<unsigned>((a.length + owned - 1) / owned) * a.heads;
}

}  // namespace

bool split_attention_supported(int length, int heads, int head_dim) {
  // a tensor's rows are addressed through 32-bit buffer offsets
  return head_dim == D && 1LL * length * heads * D * 2 < (1LL << 31) && heads <= 65535;
}

int launch_split_forward(hipStream_t stream, const SplitArgs& a) {
  split_forward_kernel<<<tile_grid(a, kQueries), kThreads, 0, stream>>>(a);
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
  if (kernel_enabled(kQueryKernel)) split_dq_kernel<<<tile_grid(a, kQueries), kThreads, 0, stream>>>(a);
  const int status = launch_status();
  if (status != 0) return status;
  if (kernel_enabled(kMainKernel)) split_dkv_kernel<<<2 * tile_grid(a, kKeys), kThreads, 0, stream>>>(a);
  return launch_status();
}

}  // namespace pluto_hip
