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
// instruction that is a third of its time.  T = 1024, 24/4 heads: 0.044 ms for the
// forward with the gated output and 0.147 for the gradients (0.046 and 0.157 before the
// clock has settled), where the kernels that multiply one element at a time took 3.9 and
// 12.4 ms.  What bounds them: one wave a SIMD in a workgroup's chain of tiles (a step is 112
// matrix instructions in the gradients, half of whose time is softmax arithmetic, splits and
// waits beside an idle matrix pipe), about 8 us before the first and after the last tile of
// each of 768 workgroups, and for the forward 384 workgroups of lengths 1 to 16 on 256 compute
// units.
//
// Shape of the kernels as in flash_bwd_mfma.hip: four waves of 32 queries (keys)
// each, tiles of 32 rows of the other side through two LDS stages filled by
// direct-to-LDS loads, one barrier a tile, score tiles oriented so that their
// accumulator is the B operand of the product that follows.
#include "attn_split_mfma.h"

#include "attn_f32_split.h"
#include "mfma_tile.h"

#include <type_traits>

namespace pluto_hip {
namespace {

constexpr int D = kSplitHeadDim;
constexpr int kThreads = 256, kRows = 32;
constexpr int KCH = D / 8, KS = D / 16, DB = D / 32;
constexpr int kLoads = kRows * KCH / kThreads;
constexpr int kTileBytes = kRows * D * 2;

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

// A wave's own rows of a tensor as operands, sixteen bytes of one row a lane, cost the compute
// unit's address path 64 cycles a load instruction: 7 of the 8.9 us before a query-owned
// gradient workgroup's first tile at T = 1024.  Brought to LDS as tiles of 32 rows, 1 KiB a
// request, they cost a quarter.  Rows beyond the sequence repeat the last one.
__device__ inline void request_own_tile(const uint16_t* tensor, long long row_stride, int length, int row0,
                                        unsigned char* tile, int wave, int lane) {
  const int32x4 rsrc = make_rsrc(tensor, tile_bytes<D>(0, length, row_stride));
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int position = (wave * kLoads + i) * 64 + lane, row = position / KCH, slot = position % KCH;
    const uint32_t at = static_cast<uint32_t>(min(row0 + row, length - 1) * row_stride * 2) + (slot ^ tile_swizzle(row)) * 16;
    lds_fill<16>(rsrc, tile + (wave * kLoads + i) * 1024, at);
  }
}
// The other way round: sixteen-byte pieces of 32 rows, a row a lane, through `area`, which no
// other wave touches, to whole rows of CHUNKS pieces.  piece(c) is the lane's piece c of its
// row n (c's parity is the lane's half); use(round, row, c, piece) has pieces of neighbouring
// lanes next to each other.
template <int CHUNKS, typename Piece, typename Use>
__device__ inline void by_rows(unsigned char* area, int lane, Piece&& piece, Use&& use) {
  const int h = lane / 32, n = lane % 32;
  float4* pieces = reinterpret_cast<float4*>(area);
#pragma unroll
  for (int c = 0; c < CHUNKS; c += 2) pieces[n * CHUNKS + ((c + h) ^ (n & 15))] = piece(c);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int kRowsAtOnce = 64 / CHUNKS;
#pragma unroll
  for (int r = 0; r < 32; r += kRowsAtOnce) {
    const int row = r + lane / CHUNKS, c = lane % CHUNKS;
    use(r / kRowsAtOnce, row, c, pieces[row * CHUNKS + (c ^ (row & 15))]);
  }
}

// Nothing moves across.  Operands are requested two or three steps ahead of their use
// and what a step requests stands between its matrix instructions: one wave a SIMD
// issues in order, so whatever stands before them in a burst runs beside none.  (Left to
// itself the compiler requests an operand and waits for it before every one to three
// matrix instructions: 282 us for dK/dV at T = 1024, 24 heads.)
__device__ inline void fence_schedule() { __builtin_amdgcn_sched_barrier(0); }

// Barrier for data exchanged through LDS: requests from memory stay under way.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ inline void stage_ready() {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// The two query-owned kernels: a workgroup owns 64 queries, waves 0 and 1 the two
// halves at even key tiles, waves 2 and 3 the same at odd ones, and the waves of a
// half add up what they have at the end.  One wave a SIMD has nothing to cover
// the chain scores -> softmax -> products of a tile; at T = 1024 the longest chain
// is what the kernel takes, and this halves it (forward 79 -> 52 us, dQ 103 -> 70
// when it was made).
constexpr int kQueries = 64;
constexpr int kQueryStageBytes = 4 * kTileBytes;  // K and V of two tiles
struct QueryWave {
  int head, half, parity, steps, first_query, query, query_load;
  __device__ QueryWave(const SplitArgs& a, int wave, int n, int head_, int q0) : head(head_) {
    half = wave % 2;
    parity = wave / 2;
    steps = ((min(q0 + kQueries, a.length) - 1) / kRows) / 2 + 1;  // two tiles each
    first_query = q0 + 32 * half;
    query = first_query + n;
    query_load = min(query, a.length - 1);
  }
};
// The fill of a step's two tiles, K, V of the even one, then of the odd one: sixteen
// requests a wave, dealt out between its products.  Issued together behind the barrier
// they queue at the compute unit's one address path (16 cycles each, four waves) while no
// wave computes (T = 1024, 24 heads: forward 50, dQ 67, dK/dV 118 us that way).  The
// descriptors stay, the lanes' offsets move from step to step; rows beyond the tensor read
// zero.
struct QueryFill {
  int32x4 rsrc[4];
  uint32_t stage, advance, offsets[kLoads];
  __device__ QueryFill(const SplitArgs& a, unsigned char* lds, int wave, int head, const TileAccess& at) {
    const long long kv_row = 1LL * (a.heads / a.group) * D;
    const long long column = head / a.group * D;
    stage = lds_address(lds + wave * kLoads * 1024);
#pragma unroll
    for (int tile = 0; tile < 2; ++tile) {
      const uint32_t bytes = tile_bytes<D>(tile * kRows, a.length, kv_row);
      rsrc[2 * tile] = make_rsrc(a.k + column + tile * kRows * kv_row, bytes);
      rsrc[2 * tile + 1] = make_rsrc(a.v + column + tile * kRows * kv_row, bytes);
    }
    advance = static_cast<uint32_t>(2 * kRows * kv_row * 2);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) offsets[i] = at.fill[i];
  }
  __device__ void next_step() {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) offsets[i] += advance;
  }
  __device__ void request(int step, int i) const {
    const uint32_t at = __builtin_amdgcn_readfirstlane(stage + (step & 1) * kQueryStageBytes);
    lds_fill_at<16>(rsrc[i / kLoads], at + i / kLoads * kTileBytes + i % kLoads * 1024, offsets[i % kLoads]);
  }
  __device__ void request_all(int step) const {
#pragma unroll
    for (int i = 0; i < 4 * kLoads; ++i) request(step, i);
  }
};
// The end of the query-owned kernels: of the two waves of a half, which hold sums of the
// even and of the odd key tiles, the lower finishes channels 0..127 and the upper the
// others (with one wave finishing all of them the gated forward took 61 us instead of
// 50-55).
constexpr int kHalfBlocks = DB / 2;
template <int FIRST>
__device__ inline void hand_over(unsigned char* lds, int half, int lane, const floatx16 (&acc)[DB]) {
  float4* area = reinterpret_cast<float4*>(lds + (2 * half + FIRST / kHalfBlocks) * kTileBytes);
#pragma unroll
  for (int i = 0; i < kHalfBlocks; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const floatx16& from = acc[FIRST + i];
      area[(4 * i + j) * 64 + lane] = make_float4(from[4 * j], from[4 * j + 1], from[4 * j + 2], from[4 * j + 3]);
    }
}
// Four channels of block FIRST + i, registers 4 j .. 4 j + 3, of the other wave.
template <int FIRST>
__device__ inline float4 handed_over(const unsigned char* lds, int half, int lane, int i, int j) {
  return reinterpret_cast<const float4*>(lds + (2 * half + FIRST / kHalfBlocks) * kTileBytes)[(4 * i + j) * 64 + lane];
}

// What the forward leaves beside core and its statistics: the backward's own forward
// nothing, a layer's forward the gated output, stored eight bytes at a time where the
// caller's tensors allow that.
enum class Gated { kNone, kWide, kNarrow };

template <Gated OUTPUT>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
split_forward_kernel(SplitArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[2 * kQueryStageBytes];
  __shared__ float wave_stats[2][2][2][64];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const QueryWave w(a, wave, n, blockIdx.x % a.heads,
                    ((a.length + kQueries - 1) / kQueries - 1 - static_cast<int>(blockIdx.x) / a.heads) * kQueries);
  const int T = a.length, query = w.query, query_load = w.query_load, head = w.head;
  const long long q_row = 1LL * a.heads * D;
  const TileAccess at(wave, lane, 1LL * (a.heads / a.group) * D);
  QueryFill fill(a, lds, wave, head, at);
  fill.request_all(0);
  bf16x8 qf[KS];
  {
    // the queries in the stage that is filled second
    unsigned char* own = lds + kQueryStageBytes;
#pragma unroll
    for (int half = 0; half < 2; ++half)
      request_own_tile(a.q + head * D, q_row, T, w.first_query + 32 * (half - w.half), own + half * kTileBytes, wave, lane);
    stage_ready();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = at.row(own + w.half * kTileBytes, ks);
    lds_barrier();
  }
  floatx16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = zero16();
  float running_max = kMasked, running_sum = 0.0f;  // of the scaled scores
  // scores to weights; register i = (key k0 + 8(i/4) + 4h + i%4, query n)
  auto softmax = [&](floatx16& s, int k0) {
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
  };
  for (int step = 0; step < w.steps; ++step) {
    const int k0 = (2 * step + w.parity) * kRows;
    stage_ready();
    fill.next_step();
    if (k0 > w.first_query + 31) {  // every key follows my queries
      fill.request_all(step + 1);
      continue;
    }
    const unsigned char* k_tile = lds + (step & 1) * kQueryStageBytes + w.parity * 2 * kTileBytes;
    const unsigned char* v_tile = k_tile + kTileBytes;
    floatx16 s = zero16();
    {
      bf16x8 kf[4];
#pragma unroll
      for (int ks = 0; ks < 3; ++ks) kf[ks] = at.row(k_tile, ks);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        fence_schedule();
        s = mfma32(kf[ks % 4], qf[ks], s);
        fence_schedule();
        if (ks + 3 < KS) kf[(ks + 3) % 4] = at.row(k_tile, ks + 3);
        if (ks % 2 == 1) fill.request(step + 1, ks / 2);
      }
      fence_schedule();
    }
    bf16x8 vt[3];
    vt[0] = at.transposed(v_tile, 0, 0);
    vt[1] = at.transposed(v_tile, 1, 0);
    fence_schedule();
    softmax(s, k0);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const Pieces p = split_accumulator(s, s2);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const int at_step = s2 * DB + db;
#pragma unroll
        for (int part = 2; part >= 0; --part) {
          fence_schedule();
          o[db] = mfma32(vt[at_step % 3], p.part[part], o[db]);
          fence_schedule();
          if (part == 2 && at_step + 2 < 2 * DB)
            vt[(at_step + 2) % 3] = at.transposed(v_tile, (at_step + 2) % DB, (at_step + 2) / DB);
          if (part == 1 && at_step < 2 * kLoads) fill.request(step + 1, 2 * kLoads + at_step);
        }
      }
    }
  }
  if (__any(!all_finite(o) || running_sum != running_sum)) [[unlikely]] {
    // An infinity in V by a weight in pieces is NaN (a piece may be zero or negative), by the
    // weight it is the infinity: the wave's tiles again, straight from memory, the weights
    // as they are.  (The scores' factors are bf16: no pieces.)
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = zero16();
    running_max = kMasked, running_sum = 0.0f;
    const long long kv_row = 1LL * (a.heads / a.group) * D;
    for (int k0 = w.parity * kRows; k0 <= w.first_query + 31 && k0 < T; k0 += 2 * kRows) {
      const long long tile = k0 * kv_row + head / a.group * D;
      const int rows = T - k0;  // those beyond count as zero
      floatx16 s = zero16();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const uint4 key = *reinterpret_cast<const uint4*>(a.k + tile + (n < rows ? n : 0) * kv_row + 16 * ks + 8 * h);
        const uint4 q = *reinterpret_cast<const uint4*>(a.q + query_load * q_row + head * D + 16 * ks + 8 * h);
        s = mfma32(as_bf16x8(n < rows ? key : make_uint4(0, 0, 0, 0)), as_bf16x8(q), s);
      }
      softmax(s, k0);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = 8 * (i / 4) + 4 * h + i % 4;
        const uint16_t* values = a.v + tile + (row < rows ? row : 0) * kv_row + n;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const float value = bf16_bits_to_float(values[32 * db]);
          o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(row < rows ? value : 0.0f, s[i], o[db], 0, 0, 0);
        }
        fence_schedule();
      }
    }
  }
  stage_ready();  // nobody reads the stages any more, or fills one
  if (w.parity == 0)
    hand_over<kHalfBlocks>(lds, w.half, lane, o);
  else
    hand_over<0>(lds, w.half, lane, o);
  wave_stats[w.half][w.parity][0][lane] = running_max;
  wave_stats[w.half][w.parity][1][lane] = running_sum;
  // 128 channels a wave leave as whole rows: lane l of round r has four channels of row 2 r +
  // l / 32
  auto finish = [&](auto first) {
    constexpr int FIRST = decltype(first)::value;
    auto place = [&](int row) {  // of a query's channels among all
      return (1LL * min(w.first_query + row, T - 1) * a.heads + head) * D + 32 * FIRST + 4 * (lane % 32);
    };
    auto gate_place = [&](int row) { return 2 * place(row) + D - 32 * FIRST - 4 * (lane % 32); };
    // the gates travel while the waves meet
    [[maybe_unused]] uint2 gates[16];
    if constexpr (OUTPUT == Gated::kWide) {
#pragma unroll
      for (int r = 0; r < 16; ++r) gates[r] = *reinterpret_cast<const uint2*>(a.qg + gate_place(2 * r + h));
    }
    lds_barrier();
    // a wave without tiles has weight 2^(kMasked - maximum) = 0
    const float other_max = wave_stats[w.half][1 - w.parity][0][lane];
    const float maximum = fmaxf(running_max, other_max);
    const float own = __builtin_amdgcn_exp2f((running_max - maximum) * kLog2e);
    const float other = __builtin_amdgcn_exp2f((other_max - maximum) * kLog2e);
    const float own_sum = running_sum * own, other_sum = wave_stats[w.half][1 - w.parity][1][lane] * other;
    const float sum = own_sum + other_sum;
    const float inverse = 1.0f / (sum > 0.0f ? sum : 1.0f);
    if (FIRST == 0 && h == 0 && query < T) {
      a.maxima[1LL * head * T + query] = maximum;
      a.inverses[1LL * head * T + query] = inverse;
      if (OUTPUT != Gated::kNone && a.lse) a.lse[1LL * query * a.heads + head] = maximum + logf(sum > 0.0f ? sum : 1.0f);
    }
    by_rows<32>(lds + (4 + wave) * kTileBytes, lane,
                [&](int c) {
                  const int i = c / 8, j = c % 8 / 2;
                  const float4 u = handed_over<FIRST>(lds, w.half, lane, i, j);
                  const floatx16& from = o[FIRST + i];
                  return make_float4((from[4 * j] * own + u.x * other) * inverse,
                                     (from[4 * j + 1] * own + u.y * other) * inverse,
                                     (from[4 * j + 2] * own + u.z * other) * inverse,
                                     (from[4 * j + 3] * own + u.w * other) * inverse);
                },
                [&](int round, int row, int, float4 core) {
                  if (w.first_query + row >= T) return;
                  *reinterpret_cast<float4*>(a.core + place(row)) = core;
                  if constexpr (OUTPUT != Gated::kNone) {
                    // qwen_attention.cc:103-108
                    const float c[4] = {core.x, core.y, core.z, core.w};
                    uint16_t* gated = a.out + place(row);
                    float logits[4], g[4];
                    if constexpr (OUTPUT == Gated::kWide) {
                      const uint2 bits = gates[round];
                      logits[0] = __uint_as_float(bits.x << 16), logits[1] = __uint_as_float(bits.x & 0xffff0000u);
                      logits[2] = __uint_as_float(bits.y << 16), logits[3] = __uint_as_float(bits.y & 0xffff0000u);
                    } else {
#pragma unroll
                      for (int e = 0; e < 4; ++e) logits[e] = bf16_bits_to_float(a.qg[gate_place(row) + e]);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) g[e] = round_to_bf16(c[e]) * round_to_bf16(gate_sigmoid(logits[e]));
                    if constexpr (OUTPUT == Gated::kWide) {
                      *reinterpret_cast<uint2*>(gated) = make_uint2(pack_bf16(g[0], g[1]), pack_bf16(g[2], g[3]));
                    } else {
#pragma unroll
                      for (int e = 0; e < 4; ++e) gated[e] = float_to_bf16_bits(g[e]);
                    }
                  }
                });
  };
  if (w.parity == 0)
    finish(std::integral_constant<int, 0>());
  else
    finish(std::integral_constant<int, kHalfBlocks>());
}

// 32 lanes a row, eight channels a lane; a workgroup walks `rows` rows of one head.
// WIDE: the caller's tensors are 16-byte aligned.
template <bool WIDE>
__global__ void __launch_bounds__(256)
split_gate_kernel(SplitArgs a, const uint16_t* __restrict__ qg, const float* __restrict__ dy,
                  float* __restrict__ dqg, int rows) {
  const int c = 8 * (threadIdx.x % 32), head = blockIdx.y;
  for (int i = 0; i < rows; i += 8) {
    const int row = blockIdx.x * rows + i + threadIdx.x / 32;
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

// dQ of 64 queries.
__device__ __forceinline__ void split_query_owned(const SplitArgs& a, unsigned char* lds, int head, int q0) {
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const QueryWave w(a, wave, n, head, q0);
  const int T = a.length, query = w.query, query_load = w.query_load;
  const long long q_row = 1LL * a.heads * D;
  const TileAccess at(wave, lane, 1LL * (a.heads / a.group) * D);
  QueryFill fill(a, lds, wave, head, at);
  const long long stat = 1LL * head * T + query_load;
  const float maximum = a.maxima[stat], inverse = a.inverses[stat], delta = a.deltas[stat];
  bf16x8 qf[KS], gf[3][KS];
  // Q and the three pieces of dC of both halves take both stages
#pragma unroll
  for (int tensor = 0; tensor < 4; ++tensor)
#pragma unroll
    for (int half = 0; half < 2; ++half)
      request_own_tile((tensor == 0 ? a.q : a.d_core + (tensor - 1) * a.piece) + head * D, q_row, T, q0 + 32 * half,
                       lds + (2 * tensor + half) * kTileBytes, wave, lane);
  stage_ready();
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qf[ks] = at.row(lds + w.half * kTileBytes, ks);
#pragma unroll
    for (int part = 0; part < 3; ++part) gf[part][ks] = at.row(lds + (2 + 2 * part + w.half) * kTileBytes, ks);
  }
  lds_barrier();
  fill.request_all(0);
  floatx16 dq[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) dq[db] = zero16();
  for (int step = 0; step < w.steps; ++step) {
    const int k0 = (2 * step + w.parity) * kRows;
    stage_ready();
    fill.next_step();
    if (k0 > w.first_query + 31) {  // every key follows my queries
      fill.request_all(step + 1);
      continue;
    }
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
      fence_schedule();
      s = mfma32(kf[ks % 3], qf[ks], s);
#pragma unroll
      for (int part = 2; part >= 0; --part) {
        fence_schedule();
        if (part == 2 && ks + 2 < KS) kf[(ks + 2) % 3] = at.row(k_tile, ks + 2);
        if (part == 1 && ks + 2 < KS) vf[(ks + 2) % 3] = at.row(v_tile, ks + 2);
        if (part == 0) fill.request(step + 1, ks);
        fence_schedule();
        dp = mfma32(vf[ks % 3], gf[part][ks], dp);
      }
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
      float ds = p * (dp[i] - delta);
      asm("" : "+v"(ds));  // in every lane: no branch around it
      s[i] = 8 * (i / 4) + (i % 4) > limit ? 0.0f : ds;
    }
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const Pieces ds = split_accumulator(s, s2);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const int at_step = s2 * DB + db;
#pragma unroll
        for (int part = 2; part >= 0; --part) {
          fence_schedule();
          dq[db] = mfma32(kt[at_step % 3], ds.part[part], dq[db]);
          fence_schedule();
          if (part == 2 && at_step + 2 < 2 * DB)
            kt[(at_step + 2) % 3] = at.transposed(k_tile, (at_step + 2) % DB, (at_step + 2) / DB);
        }
      }
    }
  }
  stage_ready();  // nobody reads the stages any more, or fills one
  if (w.parity == 0)
    hand_over<kHalfBlocks>(lds, w.half, lane, dq);
  else
    hand_over<0>(lds, w.half, lane, dq);
  __syncthreads();
  // the sums of 128 channels a wave leave as whole rows
  auto finish = [&](auto first) {
    constexpr int FIRST = decltype(first)::value;
    float* out = a.dq + head * D + 32 * FIRST;
    by_rows<32>(lds + (4 + wave) * kTileBytes, lane,
                [&](int c) {
                  const int i = c / 8, j = c % 8 / 2;
                  const float4 u = handed_over<FIRST>(lds, w.half, lane, i, j);
                  const floatx16& from = dq[FIRST + i];
                  return make_float4((from[4 * j] + u.x) * a.scale, (from[4 * j + 1] + u.y) * a.scale,
                                     (from[4 * j + 2] + u.z) * a.scale, (from[4 * j + 3] + u.w) * a.scale);
                },
                [&](int, int row, int c, float4 v) {
                  if (w.first_query + row < T) *reinterpret_cast<float4*>(out + (w.first_query + row) * q_row + 4 * c) = v;
                });
  };
  if (w.parity == 0)
    finish(std::integral_constant<int, 0>());
  else
    finish(std::integral_constant<int, kHalfBlocks>());
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
  // A tile's requests, as in QueryFill; the first brings the rows' statistics as well.
  const uint32_t bytes = tile_bytes<D>(0, T, q_row);
  int32x4 rsrc[4];
  rsrc[0] = make_rsrc(a.q + head * D, bytes);
#pragma unroll
  for (int part = 0; part < 3; ++part) rsrc[1 + part] = make_rsrc(a.d_core + part * a.piece + head * D, bytes);
  const float* stats_of_wave = wave == 0 ? a.maxima : wave == 1 ? a.inverses : a.deltas;
  const int32x4 stats_rsrc = make_rsrc(stats_of_wave + 1LL * head * T, static_cast<uint32_t>(T) * 4u);
  const uint32_t tile_stage = lds_address(lds + wave * kLoads * 1024),
                 stats_stage = lds_address(lds + 4 * kTileBytes + wave * 256);
  const uint32_t advance = static_cast<uint32_t>(kRows * q_row * 2);
  uint32_t offsets[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) offsets[i] = at.fill[i] + first_tile * advance;
  auto request = [&](int tile, int i) {
    const uint32_t stage = __builtin_amdgcn_readfirstlane((tile & 1) * kDkvStageBytes);
    lds_fill_at<16>(rsrc[i / kLoads], tile_stage + stage + i / kLoads * kTileBytes + i % kLoads * 1024,
                    offsets[i % kLoads]);
    if (i == 0 && wave < 3) lds_fill_at<4>(stats_rsrc, stats_stage + stage, lane * 4 + tile * (kRows * 4));
  };
  auto request_all = [&](int tile) {
#pragma unroll
    for (int i = 0; i < 4 * kLoads; ++i) request(tile, i);
  };
  request_all(first_tile);
  bf16x8 kf[KS], vf[VALUES ? 1 : KS];
  {
    // the keys in the stage that is filled second (what V would save there it would wait)
    unsigned char* own = lds + ((first_tile + 1) & 1) * kDkvStageBytes;
#pragma unroll
    for (int tile = 0; tile < 4; ++tile)
      request_own_tile(a.k + head / a.group * D, kv_row, T, k0 + 32 * tile, own + tile * kTileBytes, wave, lane);
    if constexpr (!VALUES) load_row_operand(a.v + key_load * kv_row + head / a.group * D, h, vf);
    stage_ready();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kf[ks] = at.row(own + wave * kTileBytes, ks);
    lds_barrier();
  }
  floatx16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = zero16();
  for (int tile = first_tile; tile < tiles; ++tile) {
    const int q0 = tile * kRows;
    stage_ready();
#pragma unroll
    for (int i = 0; i < kLoads; ++i) offsets[i] += advance;
    if (q0 + 31 < first_key) {  // every query precedes my keys
      request_all(tile + 1);
      continue;
    }
    const unsigned char* q_tile = lds + (tile & 1) * kDkvStageBytes;
    const unsigned char* g_tile = q_tile + kTileBytes;
    const float* stats = reinterpret_cast<const float*>(q_tile + 4 * kTileBytes);
    floatx16 s = zero16(), dp = zero16();
    if constexpr (VALUES) {
      bf16x8 qa[4];
#pragma unroll
      for (int ks = 0; ks < 3; ++ks) qa[ks] = at.row(q_tile, ks);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        fence_schedule();
        s = mfma32(qa[ks % 4], kf[ks], s);
        fence_schedule();
        if (ks + 3 < KS) qa[(ks + 3) % 4] = at.row(q_tile, ks + 3);
        if (ks % 2 == 1) request(tile + 1, ks / 2);
      }
      fence_schedule();
    } else {
      bf16x8 qa[3], ga[3][3];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        qa[ks] = at.row(q_tile, ks);
#pragma unroll
        for (int part = 0; part < 3; ++part) ga[ks][part] = at.row(g_tile + part * kTileBytes, ks);
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        fence_schedule();
        s = mfma32(qa[ks % 3], kf[ks], s);
        fence_schedule();
        if (ks + 2 < KS) qa[(ks + 2) % 3] = at.row(q_tile, ks + 2);
        request(tile + 1, ks);
#pragma unroll
        for (int part = 2; part >= 0; --part) {
          fence_schedule();
          dp = mfma32(ga[ks % 3][part], vf[ks], dp);
          fence_schedule();
          if (ks + 2 < KS) ga[(ks + 2) % 3][part] = at.row(g_tile + part * kTileBytes, ks + 2);
        }
      }
      fence_schedule();
    }
    // transposed operands of step (s2, db): dC's pieces for dV, Q for dK
    constexpr int kAhead = VALUES ? 1 : 2, kParts = VALUES ? 3 : 1;
    bf16x8 t[kAhead + 1][kParts];
    auto read_transposed = [&](int step, int part) {
      t[step % (kAhead + 1)][part] =
          at.transposed(VALUES ? g_tile + part * kTileBytes : q_tile, step % DB, step / DB);
    };
#pragma unroll
    for (int i = 0; i < kAhead; ++i)
#pragma unroll
      for (int part = 0; part < kParts; ++part) read_transposed(i, part);
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
#pragma unroll
        for (int gp = kParts - 1; gp >= 0; --gp)
#pragma unroll
          for (int part = 2 - gp; part >= 0; --part) {
            fence_schedule();
            acc[db] = mfma32(t[step % (kAhead + 1)][gp], p.part[part], acc[db]);
            fence_schedule();
            if (part == 2 - gp && step + kAhead < 2 * DB) read_transposed(step + kAhead, gp);
            if (VALUES && gp == 0 && part == 1 && step < 2 * kLoads) request(tile + 1, 2 * kLoads + step);
          }
      }
    }
  }
  stage_ready();  // the requests beyond the last tile; nobody reads the stages any more
  const float factor = VALUES ? 1.0f : a.scale;
  float* out = (VALUES ? a.dv : a.dk) + head * D;
  by_rows<64>(lds + wave * 2 * kTileBytes, lane,
              [&](int c) {
                const int db = c / 8, j = c % 8 / 2;
                return make_float4(acc[db][4 * j] * factor, acc[db][4 * j + 1] * factor, acc[db][4 * j + 2] * factor,
                                   acc[db][4 * j + 3] * factor);
              },
              [&](int, int row, int c, float4 v) {
                if (first_key + row < T) *reinterpret_cast<float4*>(out + (first_key + row) * q_row + 4 * c) = v;
              });
}

// All gradients in one launch, longest workgroups first: a compute unit holds one, and those
// of the last queries' tiles and of the first keys' take many times what the others do, so
// that dQ and dK/dV in launches of their own each end with most compute units idle.  24
// heads, 59.3 + 98.4 us at 1024 tokens and 149 so, 900 52.8 + 87.7 and 127, 400 27.6 + 43.8 and
// 46, 70 15.5 + 16.1 and 17.7.
enum class Gradients { kQueries, kKeys, kBoth };  // which of them a launch makes
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
split_backward_kernel(SplitArgs a, Gradients which) {
  constexpr int kLds = 2 * (kQueryStageBytes > kDkvStageBytes ? kQueryStageBytes : kDkvStageBytes);
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kLds];
  const int query_tiles = which == Gradients::kKeys ? 0 : (a.length + kQueries - 1) / kQueries;
  const int key_tiles = which == Gradients::kQueries ? 0 : (a.length + kKeys - 1) / kKeys;
  const int rows = (a.length + kRows - 1) / kRows;
  int query = query_tiles - 1, key = 0, block = blockIdx.x;
  while (true) {
    // The longest tile that is left: of keys, once for each gradient, or of queries.  A step of
    // the one takes about as long as one of the other (2.4 us).
    const int query_steps = query < 0 ? 0 : (min((query + 1) * kQueries, a.length) - 1) / kRows / 2 + 1;
    const int key_steps = key >= key_tiles ? 0 : rows - key * (kKeys / kRows);
    if (key_steps > query_steps) {
      if (block < a.heads) return split_key_owned<true>(a, lds, block, key * kKeys);
      if (block < 2 * a.heads) return split_key_owned<false>(a, lds, block - a.heads, key * kKeys);
      block -= 2 * a.heads, ++key;
    } else {
      if (block < a.heads) return split_query_owned(a, lds, block, query * kQueries);
      block -= a.heads, --query;
    }
  }
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
  auto launch = [&](auto kernel) { kernel<<<tile_grid(a, kQueries), kThreads, 0, stream>>>(a); };
  const bool wide = ((reinterpret_cast<uintptr_t>(a.out) | reinterpret_cast<uintptr_t>(a.qg)) & 7u) == 0;
  if (!a.out)
    launch(split_forward_kernel<Gated::kNone>);
  else if (wide)
    launch(split_forward_kernel<Gated::kWide>);
  else
    launch(split_forward_kernel<Gated::kNarrow>);
  return launch_status();
}

int launch_split_gate(hipStream_t stream, const SplitArgs& a, const void* qg, const float* dy,
                      float* dqg) {
  const int rows = gate_group_rows(a.length, a.heads, D);
  const dim3 grid((a.length + rows - 1) / rows, a.heads);
  const auto* gates = static_cast<const uint16_t*>(qg);
  auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  if (aligned(qg) && aligned(dy) && aligned(dqg))
    split_gate_kernel<true><<<grid, 256, 0, stream>>>(a, gates, dy, dqg, rows);
  else
    split_gate_kernel<false><<<grid, 256, 0, stream>>>(a, gates, dy, dqg, rows);
  return launch_status();
}

int launch_split_backward(hipStream_t stream, const SplitArgs& a) {
  const bool queries = kernel_enabled(kQueryKernel), keys = kernel_enabled(kMainKernel);
  const unsigned grid = (queries ? tile_grid(a, kQueries) : 0) + (keys ? 2 * tile_grid(a, kKeys) : 0);
  if (grid == 0) return 0;
  split_backward_kernel<<<grid, kThreads, 0, stream>>>(
      a, queries && keys ? Gradients::kBoth : queries ? Gradients::kQueries : Gradients::kKeys);
  return launch_status();
}

}  // namespace pluto_hip
