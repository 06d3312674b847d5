// Causal attention forward with FP32 storage: the reference's FP32 mode of
// FlashAttentionForwardKernel (src/llm/layers/attention.cc:98-170), every factor in three
// bf16 pieces and every sum in FP32 (attn_f32_split.h).
//
// A workgroup of four waves owns 32 query rows of one (sequence, head); wave w
// walks the visible key tiles (32 keys each) w, w + 4, ... with its own running
// maximum, sum and output, and the waves merge the four partial results through
// LDS in wave order.  A row block near the end of a sequence has many tiles and there
// are few row blocks, so splitting the keys is what fills the machine; the row
// blocks are handed out heaviest first, and a wave's next tiles travel while it
// works on the ones it has.  Of a call, us, on the FP32 matrix instructions and now:
// 4 sequences x 12 heads x 256 x 64 12.1, 10.0; 16 x 12 x 512 x 64 86, 71-75; 4 x 12 x 256 x
// 32 8.3, 7.5; 8 x 12 x 512 x 32 25.6, 24.0; 4 x 6 x 256 x 128 17.5, 15.7; 8 x 6 x 512 x 128
// 57.7, 52.2 (looking at the results costs 0.2 us of a small call).  Outputs 1.7e-7 off
// 64-bit arithmetic for standard normal inputs, 2.2e-7 with those instructions.  As in
// the bf16 kernels the products are transposed,
// S^T = K Q^T and O^T = V^T P^T, so that a lane owns one query column: its row
// maximum and sum are lane-local up to one exchange between the two lane
// halves, and P^T leaves the accumulator in B-operand order.  K and V take turns in the
// wave's area: with one each a compute unit would hold one workgroup.
#include "attn_f32_split.h"
#include "attn_generic.h"

#include <type_traits>

namespace pluto_hip {
namespace {

constexpr int kKeySplit = 4;  // waves per workgroup, each taking every fourth key tile

template <int D>
__global__ void __launch_bounds__(64 * kKeySplit, D == 128 ? 1 : 2)
f32_forward_kernel(GenericForwardArgs a) {
  using Rows = F32Rows<D>;
  constexpr int KS = Rows::KS, DB = Rows::DB;
  constexpr int kMergeBytes = kKeySplit * 4 * DB * 1024, kTileBytes = Rows::kOwnBytes + kKeySplit * Rows::kAreaBytes;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kTileBytes > kMergeBytes ? kTileBytes : kMergeBytes];
  __shared__ float part_max[kKeySplit][64], part_sum[kKeySplit][64];
  const int lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  // the row blocks that see the most keys first, of every (sequence, head)
  const int q_tiles = (a.q_rows + 31) / 32, units = gridDim.x / q_tiles;
  const int q0 = (q_tiles - 1 - static_cast<int>(blockIdx.x / units)) * 32;
  const int head = (blockIdx.x % units) % a.query_heads, seq = (blockIdx.x % units) / a.query_heads;
  const int kv_head = head / a.group;
  const float* q_base = static_cast<const float*>(a.q.base) + seq * a.q.seq_stride +
                        head * a.q.head_stride;
  const float* k_base = static_cast<const float*>(a.k.base) + seq * a.k.seq_stride +
                        kv_head * a.k.head_stride;
  const float* v_base = static_cast<const float*>(a.v.base) + seq * a.v.seq_stride +
                        kv_head * a.v.head_stride;
  const int query = q0 + n;
  const int query_load = min(query, a.q_rows - 1);
  const float scale2 = a.scale * kLog2e;

  const int last_query = min(q0 + 32, a.q_rows) - 1;
  const int visible_keys = min(a.kv_rows, a.start_position + last_query + 1);
  const int key_tiles = (visible_keys + 31) / 32;
  unsigned char* own = lds;
  unsigned char* area = lds + Rows::kOwnBytes + wave * Rows::kAreaBytes;
  // a tile is requested as soon as the one before has been split
  typename Rows::Raw k_raw, v_raw;
  auto request = [&](typename Rows::Raw& raw, const float* base, long long row_stride, int kt) {
    const int k0 = kt < key_tiles ? kt * 32 : 0;
    Rows::request(raw, base + k0 * row_stride, row_stride, kt < key_tiles ? a.kv_rows - k0 : 0, lane);
  };
  request(k_raw, k_base, a.k.row_stride, wave);
  request(v_raw, v_base, a.v.row_stride, wave);
  for (int ks = wave; ks < KS; ks += kKeySplit) {
    const float4* row = reinterpret_cast<const float4*>(q_base + query_load * a.q.row_stride + 16 * ks + 8 * h);
    Rows::keep_own(own, ks, lane, split_eight(row[0], row[1]));
  }
  floatx16 o[DB];
  float running_max, running_sum;  // base-2 scaled scores
  auto clear = [&]() {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[db][i] = 0.0f;
    running_max = kMasked;
    running_sum = 0.0f;
  };
  clear();
  __syncthreads();

  const int last_key = min(a.start_position + query, a.kv_rows - 1);  // keys beyond it are masked
  auto walk = [&](auto pieces) {
    constexpr bool PIECES = decltype(pieces)::value;
    const int lane = threadIdx.x % 64, h = lane / 32;  // ranges the addresses need to share bases
    for (int kt = wave; kt < key_tiles; kt += kKeySplit) {
      const int k0 = kt * 32;
      floatx16 s;
      if constexpr (PIECES) {
        Rows::keep(area, k_raw, lane);
        request(k_raw, k_base, a.k.row_stride, kt + kKeySplit);
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          s = mma_pieces(Rows::read_rows(area, ks, lane), Rows::read_own(own, ks, lane), s);
        Rows::keep(area, v_raw, lane);  // in K's place
        request(v_raw, v_base, a.v.row_stride, kt + kKeySplit);
      } else {
        s = Rows::exact_rows(k_base + k0 * a.k.row_stride, a.k.row_stride, a.kv_rows - k0,
                             q_base + query_load * a.q.row_stride, lane);
      }
      // register i = (key k0 + 8(i/4) + 4h + i%4, query n)
      const int last = last_key - k0 - 4 * h;
      float tile_max = kMasked;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        s[i] = 8 * (i / 4) + i % 4 <= last ? s[i] * scale2 : kMasked;
        tile_max = fmaxf(tile_max, s[i]);
      }
      tile_max = half_swap_max(tile_max);
      const float new_max = fmaxf(running_max, tile_max);
      const float correction = __builtin_amdgcn_exp2f(running_max - new_max);
      running_max = new_max;
      float tile_sum = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = s[i] == kMasked ? 0.0f : __builtin_amdgcn_exp2f(s[i] - new_max);
        s[i] = p;
        tile_sum += p;
      }
      running_sum = running_sum * correction + half_swap_sum(tile_sum);
      if (__any(correction != 1.0f)) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[db][i] *= correction;
      }
      if constexpr (PIECES) {
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const Pieces p = split_accumulator(s, s2);
#pragma unroll
          for (int db = 0; db < DB; ++db) o[db] = mma_pieces(Rows::read_transposed(area, db, s2, lane), p, o[db]);
        }
      } else {
        Rows::exact_transposed(o, v_base + k0 * a.v.row_stride, a.v.row_stride, a.kv_rows - k0, s, lane);
      }
    }
  };
  walk(std::true_type());
  if (__any(!all_finite(o) || running_sum != running_sum)) [[unlikely]] {
    clear();
    walk(std::false_type());
  }
  // ---- merge: every wave's result is relative to its own maximum; the waves take turns at
  // the groups of four channels
  __syncthreads();  // nobody reads tiles any more
  constexpr int kGroups = 4 * DB;
  static_assert(kGroups % kKeySplit == 0, "the groups divide over the waves");
  float4* mine = reinterpret_cast<float4*>(lds + wave * kGroups * 1024);
#pragma unroll
  for (int g = 0; g < kGroups; ++g)
    mine[g * 64 + lane] = make_float4(o[g / 4][4 * (g % 4)], o[g / 4][4 * (g % 4) + 1], o[g / 4][4 * (g % 4) + 2],
                                      o[g / 4][4 * (g % 4) + 3]);
  part_max[wave][lane] = running_max;
  part_sum[wave][lane] = running_sum;
  __syncthreads();
  float maximum = part_max[0][lane];
#pragma unroll
  for (int w = 1; w < kKeySplit; ++w) maximum = fmaxf(maximum, part_max[w][lane]);
  // a wave without tiles has weight 2^(kMasked - maximum) = 0
  float weight[kKeySplit], sum = 0.0f;
#pragma unroll
  for (int w = 0; w < kKeySplit; ++w) {
    weight[w] = __builtin_amdgcn_exp2f(part_max[w][lane] - maximum);
    sum += part_sum[w][lane] * weight[w];
  }
  if (query >= a.q_rows) return;
  const float normalizer = sum > 0.0f ? sum : 1.0f;
  const float inverse = 1.0f / normalizer;
  float* out = static_cast<float*>(a.out) + seq * a.o_seq_stride + query * a.o_row_stride +
               head * a.o_head_stride + 4 * h;
  // group g = channels 8 g + 4 h .. + 3 of query n
#pragma unroll
  for (int k = 0; k < kGroups / kKeySplit; ++k) {
    const int g = k * kKeySplit + wave;
    float4 total = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int w = 0; w < kKeySplit; ++w) {
      const float4 v = reinterpret_cast<const float4*>(lds + w * kGroups * 1024)[g * 64 + lane];
      total.x += v.x * weight[w]; total.y += v.y * weight[w];
      total.z += v.z * weight[w]; total.w += v.w * weight[w];
    }
    *reinterpret_cast<float4*>(out + 8 * g) =
        make_float4(total.x * inverse, total.y * inverse, total.z * inverse, total.w * inverse);
  }
  if (wave == 0 && h == 0) {
    maximum *= 1.0f / kLog2e;
    const long long stat = (static_cast<long long>(seq) * a.query_heads + head) * a.q_rows + query;
    if (a.maxima) a.maxima[stat] = maximum;
    if (a.normalizers) a.normalizers[stat] = normalizer;
    if (a.lse)
      a.lse[(static_cast<long long>(seq) * a.q_rows + query) * a.query_heads + head] =
          maximum + logf(normalizer);
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

bool f32_forward_supported(const GenericForwardArgs& a) {
  if (a.head_dim != 32 && a.head_dim != 64 && a.head_dim != 128) return false;
  if (a.q.dtype != PLUTO_HIP_F32 || a.k.dtype != PLUTO_HIP_F32 || a.v.dtype != PLUTO_HIP_F32 ||
      a.o_dtype != PLUTO_HIP_F32 || a.gate.base != nullptr)
    return false;
  if (a.q_rows <= 0 || a.kv_rows <= 0) return false;
  // a tile's rows are addressed through 32-bit buffer offsets
  if (32 * a.k.row_stride * 4 >= (1LL << 31) || 32 * a.v.row_stride * 4 >= (1LL << 31)) return false;
  auto mult4 = [](long long s) { return (s % 4) == 0; };
  return aligned16(a.q.base) && aligned16(a.k.base) && aligned16(a.v.base) && aligned16(a.out) &&
         mult4(a.q.seq_stride) && mult4(a.q.row_stride) && mult4(a.q.head_stride) &&
         mult4(a.k.seq_stride) && mult4(a.k.row_stride) && mult4(a.k.head_stride) &&
         mult4(a.v.seq_stride) && mult4(a.v.row_stride) && mult4(a.v.head_stride) &&
         mult4(a.o_seq_stride) && mult4(a.o_row_stride) && mult4(a.o_head_stride);
}

int launch_f32_forward(hipStream_t stream, const GenericForwardArgs& a, int sequences) {
  const long long blocks = (a.q_rows + 31LL) / 32 * a.query_heads * sequences;
  if (blocks > 0x7fffffffLL) return PLUTO_HIP_EUNSUPPORTED;
  const unsigned grid = static_cast<unsigned>(blocks);
  if (!kernel_enabled(kMainKernel)) return 0;
  switch (a.head_dim) {
    case 32: f32_forward_kernel<32><<<grid, 64 * kKeySplit, 0, stream>>>(a); break;
    case 64: f32_forward_kernel<64><<<grid, 64 * kKeySplit, 0, stream>>>(a); break;
    case 128: f32_forward_kernel<128><<<grid, 64 * kKeySplit, 0, stream>>>(a); break;
    default: return PLUTO_HIP_EUNSUPPORTED;
  }
  return launch_status();
}

}  // namespace pluto_hip
