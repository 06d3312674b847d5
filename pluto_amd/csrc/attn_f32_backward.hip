// Causal attention backward with FP32 storage: the two backward kernels of the
// reference's FP32 mode (src/llm/layers/attention.cc:235-396), every factor in three bf16
// pieces and every sum in FP32 (attn_f32_split.h).
//
//   dq    a workgroup owns 32 query rows of one (sequence, head); also does the
//         reference's delta pass (attention.cc:283-291) for them
//   dkv   a workgroup owns 32 keys
// In both, the four waves take every fourth tile of the other side (32 rows
// each) and their results are added in wave order through LDS: a sequence of 256 rows has
// 8 tiles a head, and splitting the streamed side is what fills the machine there.  A
// wave's area holds one tile at a time and takes them in turn (dq: V, K; dkv: Q, dO, Q),
// so that two workgroups share a compute unit.  The orientation is the one of
// attn_f32_mfma.hip: dq works on S^T (lane = query), dkv on S (lane = key), so the score
// tile's accumulator is the B operand of the gradient product.
//
// Of a call, us, on the FP32 matrix instructions and now: 4 sequences x 12 heads x 256 x 64
// 37.7, 25.0 (dq 11.6, dkv 15.2); 16 x 12 x 512 x 64 285, 194 (88, 117); 4 x 12 x 256 x 32
// 21.9, 17.0; 8 x 12 x 512 x 32 74, 62; 4 x 6 x 256 x 128 53.4, 33.6; 8 x 6 x 512 x 128 191,
// 143 (63, 83).  D = 128 leaves room for one workgroup a compute unit and takes 1.4 times
// what D = 64 does for as much work.  Having the other arithmetic at hand (attn_f32_split.h)
// costs 0.1 to 0.2 us of a small call.  Small calls are bound by the
// chain of a wave (its first tile's way from memory, the pieces, two products after each
// other, the merge: 7 us with one tile), large ones by streaming every tile once for 32
// rows.  Against 64-bit arithmetic the gradients are 2.4e-7 off for standard normal
// inputs of 256 rows, 3.0e-7 with the FP32 matrix instructions.
#include "attn_f32_split.h"
#include "attn_generic.h"

#include <type_traits>

namespace pluto_hip {
namespace {

constexpr int kWaves = 4;  // per workgroup, each taking every fourth streamed tile

struct F32Unit {
  int tile, head, seq;
};
// Tiles are numbered heaviest first over the whole grid.
__device__ inline F32Unit f32_unit(const GenericBackwardArgs& a, int block) {
  const int sequences = a.rows / a.context_length;
  const int units = sequences * a.num_heads;
  F32Unit u;
  u.tile = block / units;
  u.head = (block % units) % a.num_heads;
  u.seq = (block % units) / a.num_heads;
  return u;
}

// LDS of a workgroup: its own rows of two tensors, the waves' areas, the statistics of a
// streamed tile's rows; at the end the waves' results, `groups` KiB each.
constexpr int kOwnDeltaRows = 512;
template <int D, int GROUPS>
struct F32BackwardLds {
  static constexpr int kTiles = 2 * F32Rows<D>::kOwnBytes + kWaves * F32Rows<D>::kAreaBytes;
  static constexpr int kMerge = kWaves * GROUPS * 1024;
  __attribute__((aligned(1024))) unsigned char bytes[kTiles > kMerge ? kTiles : kMerge];
  __attribute__((aligned(16))) float row_stats[kWaves][3][32];
  float part_deltas[kWaves][64];
  __device__ unsigned char* own(int tensor) { return bytes + tensor * F32Rows<D>::kOwnBytes; }
  __device__ unsigned char* area(int wave) {
    return bytes + 2 * F32Rows<D>::kOwnBytes + wave * F32Rows<D>::kAreaBytes;
  }
};
template <int D>
using DqLds = F32BackwardLds<D, D / 8>;
template <int D>
using DkvLds = F32BackwardLds<D, D / 4>;

__device__ inline float dot4(float4 a, float4 b) { return (a.x * b.x + a.y * b.y) + (a.z * b.z + a.w * b.w); }

// Adds the waves' accumulators (COUNT groups of four registers a lane) in wave
// order.  The waves take turns at the groups; `store(group, sum)` gets each total once.
template <int COUNT, typename Store>
__device__ inline void merge_waves(unsigned char* lds, int wave, int lane, const float4 (&own)[COUNT], Store store) {
  __syncthreads();  // nobody reads tiles any more
  float4* mine = reinterpret_cast<float4*>(lds + wave * COUNT * 1024);
#pragma unroll
  for (int g = 0; g < COUNT; ++g) mine[g * 64 + lane] = own[g];
  __syncthreads();
  static_assert(COUNT % kWaves == 0, "the groups divide over the waves");
#pragma unroll
  for (int k = 0; k < COUNT / kWaves; ++k) {
    const int g = k * kWaves + wave;
    float4 sum = reinterpret_cast<const float4*>(lds)[g * 64 + lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) {
      const float4 v = reinterpret_cast<const float4*>(lds + w * COUNT * 1024)[g * 64 + lane];
      sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
    }
    store(g, sum);
  }
}

template <int D, class Lds>
__device__ __forceinline__ void f32_dq(const GenericBackwardArgs& a, const F32Unit& unit, Lds& sm) {
  using Rows = F32Rows<D>;
  constexpr int KS = Rows::KS, DB = Rows::DB;
  const int lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int T = a.context_length, E = a.embedding_dim;
  const int q0 = ((T + 31) / 32 - 1 - unit.tile) * 32;
  const long long row0 = static_cast<long long>(unit.seq) * T;
  const long long stats = (static_cast<long long>(unit.seq) * a.num_heads + unit.head) * T;
  const float* q_base = static_cast<const float*>(a.qkv) + row0 * 3 * E + unit.head * D;
  const int query = q0 + n, query_load = min(query, T - 1);
  const int key_tiles = q0 / 32 + 1;

  // a tile is requested as soon as the one before has been split
  unsigned char* area = sm.area(wave);
  typename Rows::Raw k_raw, v_raw;
  auto request = [&](typename Rows::Raw& raw, int tensor, int kt) {
    Rows::request(raw, q_base + tensor * E + (kt < key_tiles ? kt * 32 * 3LL * E : 0), 3LL * E,
                  kt < key_tiles ? T - kt * 32 : 0, lane);
  };
  request(k_raw, 1, wave);
  request(v_raw, 2, wave);
  const float maximum = a.maxima[stats + query_load];
  const float normalizer = a.normalizers[stats + query_load];
  const float inverse = 1.0f / (normalizer > 0.0f ? normalizer : 1.0f);
  float part_delta = 0.0f;
  for (int ks = wave; ks < KS; ks += kWaves) {
    const int c = 16 * ks + 8 * h;
    const long long at = (row0 + query_load) * E + unit.head * D + c;
    const float4* q = reinterpret_cast<const float4*>(q_base + query_load * 3LL * E + c);
    const float4* g = reinterpret_cast<const float4*>(a.d_out + at);
    const float4* o = reinterpret_cast<const float4*>(static_cast<const float*>(a.out) + at);
    const float4 g0 = g[0], g1 = g[1];
    Rows::keep_own(sm.own(0), ks, lane, split_eight(q[0], q[1]));
    Rows::keep_own(sm.own(1), ks, lane, split_eight(g0, g1));
    part_delta += dot4(g0, o[0]) + dot4(g1, o[1]);
  }
  sm.part_deltas[wave][lane] = part_delta;
  floatx16 acc[DB];
  auto clear = [&]() {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[db][i] = 0.0f;
  };
  clear();
  __syncthreads();
  float delta = 0.0f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) delta += sm.part_deltas[w][lane];
  delta = half_swap_sum(delta);
  if (wave == 0 && h == 0 && query < T) a.deltas[stats + query] = delta;

  auto walk = [&](auto pieces) {
    constexpr bool PIECES = decltype(pieces)::value;
    const int lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;  // ranges the addresses need to share bases
    for (int kt = wave; kt < key_tiles; kt += kWaves) {
      const int k0 = kt * 32;
      floatx16 s, dp;
      const float* k_tile = q_base + E + k0 * 3LL * E;
      if constexpr (PIECES) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = dp[i] = 0.0f;
        Rows::keep(area, v_raw, lane);
        request(v_raw, 2, kt + kWaves);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          dp = mma_pieces(Rows::read_rows(area, ks, lane), Rows::read_own(sm.own(1), ks, lane), dp);
        Rows::keep(area, k_raw, lane);  // in V's place
        request(k_raw, 1, kt + kWaves);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          s = mma_pieces(Rows::read_rows(area, ks, lane), Rows::read_own(sm.own(0), ks, lane), s);
      } else {
        dp = Rows::exact_rows(k_tile + E, 3LL * E, T - k0, a.d_out + (row0 + query_load) * E + unit.head * D, lane);
        s = Rows::exact_rows(k_tile, 3LL * E, T - k0, q_base + query_load * 3LL * E, lane);
      }
      // register i = (key k0 + 8(i/4) + 4h + i%4, query n)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = k0 + 8 * (i / 4) + 4 * h + (i % 4);
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.scale, -maximum) * kLog2e) * inverse;
        float ds = p * (dp[i] - delta) * a.scale;
        asm("" : "+v"(ds));  // in every lane: no branch around it
        s[i] = key <= query_load ? ds : 0.0f;
      }
      if constexpr (PIECES) {
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const Pieces ds = split_accumulator(s, s2);
#pragma unroll
          for (int db = 0; db < DB; ++db) acc[db] = mma_pieces(Rows::read_transposed(area, db, s2, lane), ds, acc[db]);
        }
      } else {
        Rows::exact_transposed(acc, k_tile, 3LL * E, T - k0, s, lane);
      }
    }
  };
  walk(std::true_type());
  if (__any(!all_finite(acc))) [[unlikely]] {
    clear();
    walk(std::false_type());
  }
  float4 own[4 * DB];
#pragma unroll
  for (int g = 0; g < 4 * DB; ++g)
    own[g] = make_float4(acc[g / 4][4 * (g % 4)], acc[g / 4][4 * (g % 4) + 1],
                         acc[g / 4][4 * (g % 4) + 2], acc[g / 4][4 * (g % 4) + 3]);
  float* out = a.d_qkv + (row0 + query_load) * 3 * E + unit.head * D + 4 * h;
  // group g = channels 32 (g / 4) + 8 (g % 4) + 4 h .. + 3 of query n
  merge_waves(sm.bytes, wave, lane, own, [&](int g, float4 sum) {
    if (query < T) *reinterpret_cast<float4*>(out + 8 * g) = sum;
  });
}

// own_deltas: [kOwnDeltaRows] in LDS, or null where the dq kernel has left the row sums.
template <int D, bool OWN_DELTAS, class Lds>
__device__ __forceinline__ void f32_dkv(const GenericBackwardArgs& a, const F32Unit& unit, Lds& sm, float* own_deltas) {
  using Rows = F32Rows<D>;
  constexpr int KS = Rows::KS, DB = Rows::DB;
  auto& row_stats = sm.row_stats;
  const int lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int T = a.context_length, E = a.embedding_dim;
  const int k0 = unit.tile * 32;
  const long long row0 = static_cast<long long>(unit.seq) * T;
  const long long stats = (static_cast<long long>(unit.seq) * a.num_heads + unit.head) * T;
  const float* q_base = static_cast<const float*>(a.qkv) + row0 * 3 * E + unit.head * D;
  const float* g_base = a.d_out + row0 * E + unit.head * D;
  const int key = k0 + n, key_load = min(key, T - 1);
  const int query_tiles = (T + 31) / 32;

  unsigned char* area = sm.area(wave);
  typename Rows::Raw q_raw, g_raw;
  auto request_q = [&](int qt) {
    const bool exists = qt < query_tiles;
    Rows::request(q_raw, q_base + (exists ? qt * 32 * 3LL * E : 0), 3LL * E, exists ? T - qt * 32 : 0, lane);
  };
  auto request_g = [&](int qt) {
    const bool exists = qt < query_tiles;
    Rows::request(g_raw, g_base + (exists ? qt * 32 * 1LL * E : 0), E, exists ? T - qt * 32 : 0, lane);
  };
  request_q(k0 / 32 + wave);
  request_g(k0 / 32 + wave);
  for (int ks = wave; ks < KS; ks += kWaves) {
    const float4* k = reinterpret_cast<const float4*>(q_base + E + key_load * 3LL * E + 16 * ks + 8 * h);
    const float4* v = reinterpret_cast<const float4*>(q_base + 2 * E + key_load * 3LL * E + 16 * ks + 8 * h);
    Rows::keep_own(sm.own(0), ks, lane, split_eight(k[0], k[1]));
    Rows::keep_own(sm.own(1), ks, lane, split_eight(v[0], v[1]));
  }
  if constexpr (OWN_DELTAS) {
    // those of the wave's own tiles: nobody else reads them
    for (int qt = k0 / 32 + wave; qt < query_tiles; qt += kWaves) {
      const int row = min(qt * 32 + n, T - 1);
      const float4* g = reinterpret_cast<const float4*>(g_base + row * 1LL * E + 8 * h);
      const float4* o = reinterpret_cast<const float4*>(static_cast<const float*>(a.out) + (row0 + row) * E +
                                                        unit.head * D + 8 * h);
      float delta = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) delta += dot4(g[4 * ks], o[4 * ks]) + dot4(g[4 * ks + 1], o[4 * ks + 1]);
      delta = half_swap_sum(delta);
      if (h == 0) own_deltas[qt * 32 + n] = delta;
    }
  }
  floatx16 dk[DB], dv[DB];
  auto clear = [&]() {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) dk[db][i] = dv[db][i] = 0.0f;
  };
  clear();
  __syncthreads();
  auto walk = [&](auto pieces) {
    constexpr bool PIECES = decltype(pieces)::value;
    const int lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;  // ranges the addresses need to share bases
    for (int qt = k0 / 32 + wave; qt < query_tiles; qt += kWaves) {
      const int q0 = qt * 32;
      if (h == 0) {
        const int row = min(q0 + n, T - 1);
        const float normalizer = a.normalizers[stats + row];
        row_stats[wave][0][n] = a.maxima[stats + row];
        row_stats[wave][1][n] = 1.0f / (normalizer > 0.0f ? normalizer : 1.0f);
        row_stats[wave][2][n] = OWN_DELTAS ? own_deltas[q0 + n] : a.deltas[stats + row];
      }
      floatx16 s, dp;
      const float* q_tile = q_base + q0 * 3LL * E;
      const float* g_tile = g_base + q0 * 1LL * E;
      if constexpr (PIECES) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = dp[i] = 0.0f;
        // one area for Q, dO and Q again: two would leave room for one workgroup a compute unit
        Rows::keep(area, q_raw, lane);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          s = mma_pieces(Rows::read_rows(area, ks, lane), Rows::read_own(sm.own(0), ks, lane), s);
        Rows::keep(area, g_raw, lane);
        request_g(qt + kWaves);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          dp = mma_pieces(Rows::read_rows(area, ks, lane), Rows::read_own(sm.own(1), ks, lane), dp);
      } else {
        const float* own_key = q_base + E + key_load * 3LL * E;
        s = Rows::exact_rows(q_tile, 3LL * E, T - q0, own_key, lane);
        dp = Rows::exact_rows(g_tile, E, T - q0, own_key + E, lane);
      }
      __builtin_amdgcn_sched_barrier(0);  // (the products spread over what follows: 24.7 -> 25.7 us above)
      // register i = (query q0 + 8(i/4) + 4h + i%4, key n)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int at = 8 * j + 4 * h;
        const float4 maximum = *reinterpret_cast<const float4*>(&row_stats[wave][0][at]);
        const float4 inverse = *reinterpret_cast<const float4*>(&row_stats[wave][1][at]);
        const float4 delta = *reinterpret_cast<const float4*>(&row_stats[wave][2][at]);
        const float m[4] = {maximum.x, maximum.y, maximum.z, maximum.w};
        const float r[4] = {inverse.x, inverse.y, inverse.z, inverse.w};
        const float dl[4] = {delta.x, delta.y, delta.z, delta.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 4 * j + e, query = q0 + at + e;
          float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.scale, -m[e]) * kLog2e) * r[e];
          float ds = p * (dp[i] - dl[e]) * a.scale;
          asm("" : "+v"(p), "+v"(ds));  // in every lane: no branch around them
          const bool visible = key <= query && query < T;
          s[i] = visible ? p : 0.0f;
          dp[i] = visible ? ds : 0.0f;
        }
      }
      if constexpr (PIECES) {
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const Pieces p = split_accumulator(s, s2);
#pragma unroll
          for (int db = 0; db < DB; ++db) dv[db] = mma_pieces(Rows::read_transposed(area, db, s2, lane), p, dv[db]);
        }
        Rows::keep(area, q_raw, lane);
        request_q(qt + kWaves);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const Pieces ds = split_accumulator(dp, s2);
#pragma unroll
          for (int db = 0; db < DB; ++db) dk[db] = mma_pieces(Rows::read_transposed(area, db, s2, lane), ds, dk[db]);
        }
      } else {
        Rows::exact_transposed(dv, g_tile, E, T - q0, s, lane);
        Rows::exact_transposed(dk, q_tile, 3LL * E, T - q0, dp, lane);
      }
    }
  };
  walk(std::true_type());
  if (__any(!all_finite(dk) || !all_finite(dv))) [[unlikely]] {
    clear();
    walk(std::false_type());
  }
  float4 own[8 * DB];
#pragma unroll
  for (int g = 0; g < 4 * DB; ++g) {
    own[g] = make_float4(dk[g / 4][4 * (g % 4)], dk[g / 4][4 * (g % 4) + 1],
                         dk[g / 4][4 * (g % 4) + 2], dk[g / 4][4 * (g % 4) + 3]);
    own[4 * DB + g] = make_float4(dv[g / 4][4 * (g % 4)], dv[g / 4][4 * (g % 4) + 1],
                                  dv[g / 4][4 * (g % 4) + 2], dv[g / 4][4 * (g % 4) + 3]);
  }
  float* out = a.d_qkv + (row0 + key_load) * 3 * E + E + unit.head * D + 4 * h;
  merge_waves(sm.bytes, wave, lane, own, [&](int g, float4 sum) {
    const int tensor = g / (4 * DB);
    if (key < T) *reinterpret_cast<float4*>(out + tensor * E + 8 * (g % (4 * DB))) = sum;
  });
}

template <int D>
__global__ void __launch_bounds__(64 * kWaves, D == 128 ? 1 : 2)
f32_dq_kernel(GenericBackwardArgs a) {
  __shared__ DqLds<D> sm;
  f32_dq<D>(a, f32_unit(a, blockIdx.x), sm);
}

template <int D>
__global__ void __launch_bounds__(64 * kWaves, D == 128 ? 1 : 2)
f32_dkv_kernel(GenericBackwardArgs a) {
  __shared__ DkvLds<D> sm;
  f32_dkv<D, false>(a, f32_unit(a, blockIdx.x), sm, nullptr);
}

// Both in one launch: every dkv workgroup makes the row sums of the queries it streams.
// The halves of a level (tiles of equal length) follow each other.
template <int D>
__global__ void __launch_bounds__(64 * kWaves, D == 128 ? 1 : 2)
f32_pair_kernel(GenericBackwardArgs a) {
  __shared__ DkvLds<D> sm;
  __shared__ float own_deltas[kOwnDeltaRows];
  const int units = a.rows / a.context_length * a.num_heads;
  const int level = blockIdx.x / units, block = level / 2 * units + blockIdx.x % units;
  if (level % 2 == 0)
    f32_dkv<D, true>(a, f32_unit(a, block), sm, own_deltas);
  else
    f32_dq<D>(a, f32_unit(a, block), sm);
}

// One launch where the workgroups of both kernels fit on the chip together, or nearly so
// (two a compute unit, one at D = 128), and for short sequences, of which a workgroup sees
// little, to several times that.  Beyond, the row sums made more than once cost more than
// the launch.  Two launches against one, us: 1 x 12 x 48 x 64 14.8, 8.9; 4 x 12 x 200 24.2,
// 20.6; 16 x 12 x 100 32.5, 29.9; 4 x 12 x 256 (384 workgroups each) 25.1, 26.7; 8 x 12 x
// 512 104, 120; 4 x 6 x 256 x 128 41.7, 34.3; 8 x 6 x 512 x 128 145, 179.
template <int D>
bool one_launch(const GenericBackwardArgs& a, unsigned grid) {
  constexpr unsigned kResident = D == 128 ? 192 : 352, kShort = D == 128 ? 576 : 1152;
  return a.context_length <= kOwnDeltaRows && (grid <= kResident || (a.context_length <= 128 && grid <= kShort));
}

template <int D>
int launch(hipStream_t stream, const GenericBackwardArgs& a, unsigned grid) {
  if (one_launch<D>(a, grid) && kernel_enabled(kQueryKernel) && kernel_enabled(kMainKernel)) {
    f32_pair_kernel<D><<<2 * grid, 64 * kWaves, 0, stream>>>(a);
    return launch_status();
  }
  if (kernel_enabled(kQueryKernel)) f32_dq_kernel<D><<<grid, 64 * kWaves, 0, stream>>>(a);
  int status = launch_status();
  if (status != 0) return status;
  if (kernel_enabled(kMainKernel)) f32_dkv_kernel<D><<<grid, 64 * kWaves, 0, stream>>>(a);
  return launch_status();
}

}  // namespace

bool f32_backward_supported(const GenericBackwardArgs& a) {
  const int dim = a.embedding_dim / a.num_heads;
  if (a.dtype != PLUTO_HIP_F32 || (dim != 32 && dim != 64 && dim != 128)) return false;
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  // a tile's rows are addressed through 32-bit buffer offsets
  if (32LL * 3 * a.embedding_dim * 4 >= (1LL << 31)) return false;
  const long long units = static_cast<long long>(a.rows / a.context_length) * a.num_heads;
  if ((a.context_length + 31LL) / 32 * units > 0x7fffffffLL) return false;
  return aligned(a.qkv) && aligned(a.out) && aligned(a.d_out) && aligned(a.d_qkv);
}

int launch_f32_backward(hipStream_t stream, const GenericBackwardArgs& a) {
  const unsigned grid = static_cast<unsigned>((a.context_length + 31LL) / 32 *
                                              (a.rows / a.context_length) * a.num_heads);
  switch (a.embedding_dim / a.num_heads) {
    case 32: return launch<32>(stream, a, grid);
    case 64: return launch<64>(stream, a, grid);
    case 128: return launch<128>(stream, a, grid);
    default: return PLUTO_HIP_EUNSUPPORTED;
  }
}

}  // namespace pluto_hip
