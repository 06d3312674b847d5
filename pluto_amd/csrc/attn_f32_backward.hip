// Causal attention backward with FP32 storage on the FP32 matrix cores
// (v_mfma_f32_32x32x2_f32): the two backward kernels of the reference's FP32
// mode (src/llm/layers/attention.cc:235-396), every product and sum in FP32.
//
//   dq    a workgroup owns 32 query rows of one (sequence, head); also does the
//         reference's delta pass (attention.cc:283-291) for them
//   dkv   a workgroup owns 32 keys
// In both, the four waves take every fourth tile of the other side (32 rows
// each) and their results are added in wave order through LDS: the matrix
// instruction is slow (64 cycles), a sequence of 256 rows has 8 tiles a head, and
// splitting the streamed side is what fills the machine there.  A tile is filled
// by direct-to-LDS loads into the wave's own area (no barrier in the loop) and
// read both ways: 16-byte pieces of a lane's row for the score products, one
// float a lane along a row for the gradient products.  The orientation is the
// one of attn_f32_mfma.hip: dq works on S^T (lane = query), dkv on S (lane = key),
// so the score tile's accumulator is the B operand of the gradient product.
// 4 sequences x 12 heads x 256 x 64: 40 us for the pair, where the kernels that
// multiply one element at a time took 653 us.
#include "attn_f32_tile.h"
#include "attn_generic.h"
#include "mfma_tile.h"

namespace pluto_hip {
namespace {

constexpr int kWaves = 4;  // per workgroup, each taking every fourth streamed tile

struct F32Unit {
  int tile, head, seq;
};
// Tiles are numbered heaviest first over the whole grid.
__device__ inline F32Unit f32_unit(const GenericBackwardArgs& a) {
  const int sequences = a.rows / a.context_length;
  const int units = sequences * a.num_heads;
  F32Unit u;
  u.tile = blockIdx.x / units;
  u.head = (blockIdx.x % units) % a.num_heads;
  u.seq = (blockIdx.x % units) / a.num_heads;
  return u;
}

// Adds the waves' accumulators (COUNT groups of four registers a lane) in wave
// order.  The waves take turns at the groups; `store(group, lane, sum)` gets each
// total once.  Every wave's area holds its COUNT * 1 KiB.
template <int COUNT, typename Store>
__device__ inline void merge_waves(unsigned char* areas, int area_bytes, int wave, int lane,
                                   const float4 (&own)[COUNT], Store store) {
  float4* mine = reinterpret_cast<float4*>(areas + wave * area_bytes);
#pragma unroll
  for (int g = 0; g < COUNT; ++g) mine[g * 64 + lane] = own[g];
  __syncthreads();
  static_assert(COUNT % kWaves == 0, "the groups divide over the waves");
#pragma unroll
  for (int k = 0; k < COUNT / kWaves; ++k) {
    const int g = k * kWaves + wave;
    float4 sum = reinterpret_cast<const float4*>(areas)[g * 64 + lane];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) {
      const float4 v = reinterpret_cast<const float4*>(areas + w * area_bytes)[g * 64 + lane];
      sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
    }
    store(g, sum);
  }
}

template <int D>
__global__ void __launch_bounds__(64 * kWaves, D == 128 ? 1 : 2)
f32_dq_kernel(GenericBackwardArgs a) {
  using Tile = F32Tile<D>;
  constexpr int HALF = D / 2, DB = D / 32, kArea = 2 * Tile::kBytes;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kWaves * kArea];
  const int lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int T = a.context_length, E = a.embedding_dim;
  const F32Unit unit = f32_unit(a);
  const int q0 = ((T + 31) / 32 - 1 - unit.tile) * 32;
  const long long row0 = static_cast<long long>(unit.seq) * T;
  const long long stats = (static_cast<long long>(unit.seq) * a.num_heads + unit.head) * T;
  const float* q_base = static_cast<const float*>(a.qkv) + row0 * 3 * E + unit.head * D;
  const int query = q0 + n, query_load = min(query, T - 1);

  // A wave's first tile is on its way while it reads its own rows, the others while the
  // one before is worked on: V in place as soon as it has been read, K, which is
  // needed to the end, through registers.
  unsigned char* k_tile = lds + wave * kArea;
  unsigned char* v_tile = k_tile + Tile::kBytes;
  typename Tile::Held k_held;
  auto rows_of = [&](int kt) { return kt <= q0 / 32 ? T - kt * 32 : 0; };
  auto request_k = [&](int kt) {
    Tile::request(k_held, q_base + E + kt * 32 * 3LL * E, 3LL * E, rows_of(kt), lane);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto request_v = [&](int kt) {
    Tile::fill(v_tile, q_base + 2 * E + kt * 32 * 3LL * E, 3LL * E, rows_of(kt), lane);
  };
  request_k(wave);
  request_v(wave);
  float qf[HALF], gf[HALF];
  load_half_row<HALF>(q_base + query_load * 3LL * E + h * HALF, qf);
  const long long out_at = (row0 + query_load) * E + unit.head * D + h * HALF;
  load_half_row<HALF>(a.d_out + out_at, gf);
  float delta = 0.0f;
#pragma unroll
  for (int j = 0; j < HALF / 4; ++j) {
    const float4 o = reinterpret_cast<const float4*>(static_cast<const float*>(a.out) + out_at)[j];
    delta += gf[4 * j] * o.x + gf[4 * j + 1] * o.y + gf[4 * j + 2] * o.z + gf[4 * j + 3] * o.w;
  }
  delta = half_swap_sum(delta);
  if (wave == 0 && h == 0 && query < T) a.deltas[stats + query] = delta;
  const float maximum = a.maxima[stats + query_load];
  const float normalizer = a.normalizers[stats + query_load];
  const float inverse = 1.0f / (normalizer > 0.0f ? normalizer : 1.0f);

  floatx16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[db][i] = 0.0f;
  const int key_tiles = q0 / 32 + 1;
  for (int kt = wave; kt < key_tiles; kt += kWaves) {
    const int k0 = kt * 32;
    Tile::place(k_tile, k_held, lane);
    wait_fills();
    request_k(kt + kWaves);
    floatx16 s, dp;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = dp[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < HALF / 4; ++j) {
      const float4 k4 = Tile::row_piece(k_tile, n, h * (HALF / 4) + j);
      const float4 v4 = Tile::row_piece(v_tile, n, h * (HALF / 4) + j);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.x, qf[4 * j], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(v4.x, gf[4 * j], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.y, qf[4 * j + 1], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(v4.y, gf[4 * j + 1], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.z, qf[4 * j + 2], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(v4.z, gf[4 * j + 2], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.w, qf[4 * j + 3], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(v4.w, gf[4 * j + 3], dp, 0, 0, 0);
    }
    wait_reads();
    request_v(kt + kWaves);
    // register i = (key k0 + 8(i/4) + 4h + i%4, query n)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = k0 + 8 * (i / 4) + 4 * h + (i % 4);
      const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.scale, -maximum) * kLog2e) * inverse;
      s[i] = key <= query_load ? p * (dp[i] - delta) * a.scale : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int db = 0; db < DB; ++db)
        acc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(
            Tile::element(k_tile, 8 * (i / 4) + 4 * h + (i % 4), 32 * db + n), s[i], acc[db], 0, 0, 0);
  }
  wait_fills();
  float4 own[4 * DB];
#pragma unroll
  for (int g = 0; g < 4 * DB; ++g)
    own[g] = make_float4(acc[g / 4][4 * (g % 4)], acc[g / 4][4 * (g % 4) + 1],
                         acc[g / 4][4 * (g % 4) + 2], acc[g / 4][4 * (g % 4) + 3]);
  float* out = a.d_qkv + (row0 + query_load) * 3 * E + unit.head * D + 4 * h;
  // group g = channels 32 (g / 4) + 8 (g % 4) + 4 h .. + 3 of query n
  merge_waves(lds, kArea, wave, lane, own, [&](int g, float4 sum) {
    if (query < T) *reinterpret_cast<float4*>(out + 8 * g) = sum;
  });
}

template <int D>
__global__ void __launch_bounds__(64 * kWaves, D == 128 ? 1 : 2)
f32_dkv_kernel(GenericBackwardArgs a) {
  using Tile = F32Tile<D>;
  constexpr int HALF = D / 2, DB = D / 32, kArea = 2 * Tile::kBytes;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kWaves * kArea];
  __shared__ __attribute__((aligned(16))) float row_stats[kWaves][3][32];
  const int lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int T = a.context_length, E = a.embedding_dim;
  const F32Unit unit = f32_unit(a);
  const int k0 = unit.tile * 32;
  const long long row0 = static_cast<long long>(unit.seq) * T;
  const long long stats = (static_cast<long long>(unit.seq) * a.num_heads + unit.head) * T;
  const float* q_base = static_cast<const float*>(a.qkv) + row0 * 3 * E + unit.head * D;
  const float* g_base = a.d_out + row0 * E + unit.head * D;
  const int key = k0 + n, key_load = min(key, T - 1);

  // the first tile is on its way before the wave's own rows; registers to hold
  // another are not left (21.5 us at 256 rows, 23.8 with the request in the loop)
  unsigned char* q_tile = lds + wave * kArea;
  unsigned char* g_tile = q_tile + Tile::kBytes;
  auto request = [&](int qt) {
    const int q0 = qt * 32;
    Tile::fill(q_tile, q_base + q0 * 3LL * E, 3LL * E, T - q0, lane);
    Tile::fill(g_tile, g_base + q0 * 1LL * E, E, T - q0, lane);
  };
  request(k0 / 32 + wave);
  float kf[HALF], vf[HALF];
  load_half_row<HALF>(q_base + E + key_load * 3LL * E + h * HALF, kf);
  load_half_row<HALF>(q_base + 2 * E + key_load * 3LL * E + h * HALF, vf);
  floatx16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[db][i] = dv[db][i] = 0.0f;
  const int query_tiles = (T + 31) / 32;
  for (int qt = k0 / 32 + wave; qt < query_tiles; qt += kWaves) {
    const int q0 = qt * 32;
    if (h == 0) {
      const int row = min(q0 + n, T - 1);
      const float normalizer = a.normalizers[stats + row];
      row_stats[wave][0][n] = a.maxima[stats + row];
      row_stats[wave][1][n] = 1.0f / (normalizer > 0.0f ? normalizer : 1.0f);
      row_stats[wave][2][n] = a.deltas[stats + row];
    }
    wait_fills();
    floatx16 s, dp;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = dp[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < HALF / 4; ++j) {
      const float4 q4 = Tile::row_piece(q_tile, n, h * (HALF / 4) + j);
      const float4 g4 = Tile::row_piece(g_tile, n, h * (HALF / 4) + j);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(q4.x, kf[4 * j], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(g4.x, vf[4 * j], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(q4.y, kf[4 * j + 1], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(g4.y, vf[4 * j + 1], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(q4.z, kf[4 * j + 2], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(g4.z, vf[4 * j + 2], dp, 0, 0, 0);
      s = __builtin_amdgcn_mfma_f32_32x32x2f32(q4.w, kf[4 * j + 3], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x2f32(g4.w, vf[4 * j + 3], dp, 0, 0, 0);
    }
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
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], a.scale, -m[e]) * kLog2e) * r[e];
        const bool visible = key <= query && query < T;
        s[i] = visible ? p : 0.0f;
        dp[i] = visible ? p * (dp[i] - dl[e]) * a.scale : 0.0f;
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const int row = 8 * (i / 4) + 4 * h + (i % 4);
        dv[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(Tile::element(g_tile, row, 32 * db + n), s[i],
                                                      dv[db], 0, 0, 0);
        dk[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(Tile::element(q_tile, row, 32 * db + n), dp[i],
                                                      dk[db], 0, 0, 0);
      }
    wait_reads();
    if (qt + kWaves < query_tiles) request(qt + kWaves);
  }
  wait_fills();
  float4 own[8 * DB];
#pragma unroll
  for (int g = 0; g < 4 * DB; ++g) {
    own[g] = make_float4(dk[g / 4][4 * (g % 4)], dk[g / 4][4 * (g % 4) + 1],
                         dk[g / 4][4 * (g % 4) + 2], dk[g / 4][4 * (g % 4) + 3]);
    own[4 * DB + g] = make_float4(dv[g / 4][4 * (g % 4)], dv[g / 4][4 * (g % 4) + 1],
                                  dv[g / 4][4 * (g % 4) + 2], dv[g / 4][4 * (g % 4) + 3]);
  }
  float* out = a.d_qkv + (row0 + key_load) * 3 * E + E + unit.head * D + 4 * h;
  merge_waves(lds, kArea, wave, lane, own, [&](int g, float4 sum) {
    const int tensor = g / (4 * DB);
    if (key < T) *reinterpret_cast<float4*>(out + tensor * E + 8 * (g % (4 * DB))) = sum;
  });
}

template <int D>
int launch(hipStream_t stream, const GenericBackwardArgs& a, unsigned grid) {
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
