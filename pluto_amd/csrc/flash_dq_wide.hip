// Query-owned half of the causal attention backward for bf16 heads of 128
// channels: dQ^T[d, query] = sum_keys K^T[d, key] dS^T[key, query]
// (src/llm/layers/attention.cc:235-291), with the main loop as a hand-scheduled
// instruction stream (gen_flash_dq_loop128.py describes the schedule).  Where the
// upstream gradient arrives in FP32 the prologue also leaves delta, the row's
// log2-sum-exp and a bf16 copy of dO for the key-owned kernel.
//
// A workgroup of two waves owns 128 queries, a wave 64 of them as two halves of
// 32 (lane = query), one wave a SIMD.  The kernel before it, with 32 queries a wave and
// its operands straight from LDS, was bound by the LDS reads; this one keeps the matrix
// pipe busy 64 % of the time at the 1.84 GHz the card holds under it, with 2.8 other
// vector instructions to a matrix instruction: 24 heads of 8192 rows 601 -> 518 us
// (0.62 TFLOP, 1.2 PFLOP/s).
#include "flash_bwd_mfma.h"

#include "flash_dq_loop128.inc"
#include "mfma_tile.h"

namespace pluto_hip {
namespace {

constexpr int kThreads = 128, D = 128, KS = D / 16, KCH = D / 8;
constexpr int kRing = FLASH_DQ_D128_RING, kStageBytes = FLASH_DQ_D128_STAGE_BYTES;
constexpr int kTileBytes = FLASH_DQ_D128_TILE_BYTES;
static_assert(kTileBytes == 32 * D * 2);

// PREPARED: dO arrives as bf16 with its row statistics, else the prologue makes them.
template <bool PREPARED>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
flash_dq_wide_kernel(FlashBackwardArgs a) {
  __shared__ __attribute__((aligned(1024))) unsigned char lds[kRing * kStageBytes];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int lane = threadIdx.x % 64, h = lane / 32, n = lane % 32;
  const int T = a.context_length, H = a.num_heads, E = H * D;
  // one tile per workgroup, the tiles that see the most keys first; a (sequence,
  // head) unit keeps its XCD across tiles whenever the number of units is a
  // multiple of 8
  const int q_tiles = (T + 127) / 128;
  const int units = gridDim.x / q_tiles;
  const int q_tile = q_tiles - 1 - static_cast<int>(blockIdx.x / units);
  const int head = (blockIdx.x % units) % H, seq = (blockIdx.x % units) / H;
  const long long seq_row0 = static_cast<long long>(seq) * T;
  const long long stats_base = (static_cast<long long>(seq) * H + head) * T;
  const long long q_stride = a.q_row, kv_stride = a.kv_row;
  const uint16_t* q_base = a.q + seq_row0 * q_stride + head * D;
  const uint16_t* k_base = a.k + seq_row0 * kv_stride + head / a.group * D;
  const uint16_t* v_base = a.v + seq_row0 * kv_stride + head / a.group * D;
  uint16_t* gb_base = a.d_out_bf16 + seq_row0 * E + head * D;
  const float scale2 = a.scale * kLog2e;
  const int q0 = q_tile * 128, wave_first = q0 + 64 * wave;

  bf16x8 qf[2][KS], gf[2][KS];
  float lse[2], delta[2];  // both negated
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int first = wave_first + 32 * c, q_row = first + n;
    // rows beyond the sequence are clamped to its last row and never stored
    const int q_load = min(q_row, T - 1);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[c][ks] = as_bf16x8(*reinterpret_cast<const uint4*>(q_base + q_load * q_stride + 16 * ks + 8 * h));
    if constexpr (PREPARED) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        gf[c][ks] = as_bf16x8(*reinterpret_cast<const uint4*>(
            gb_base + static_cast<long long>(q_load) * E + 16 * ks + 8 * h));
      delta[c] = a.deltas[stats_base + q_load];
      lse[c] = a.lse2[stats_base + q_load] * scale2;
    } else {
      const long long row = seq_row0 * E + head * D + static_cast<long long>(q_load) * E;
      uint4* copy_area = reinterpret_cast<uint4*>(lds) + wave * 32 * KCH;
      float partial = 0.0f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int at = 16 * ks + 8 * h;
        const float4 g0 = *reinterpret_cast<const float4*>(a.d_out + row + at);
        const float4 g1 = *reinterpret_cast<const float4*>(a.d_out + row + at + 4);
        const uint4 o = *reinterpret_cast<const uint4*>(a.out + row + at);
        const float g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
        const uint32_t ow[4] = {o.x, o.y, o.z, o.w};
        uint32_t packed[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          partial += g[2 * i] * __uint_as_float(ow[i] << 16);
          partial += g[2 * i + 1] * __uint_as_float(ow[i] & 0xffff0000u);
          packed[i] = pack_bf16(g[2 * i], g[2 * i + 1]);
        }
        const uint4 bits = make_uint4(packed[0], packed[1], packed[2], packed[3]);
        gf[c][ks] = as_bf16x8(bits);
        copy_area[n * KCH + ((2 * ks + h) ^ (n & 7))] = bits;
      }
      // the bf16 copy of dO leaves through the wave's own LDS: whole rows a store
#pragma unroll
      for (int i = 0; i < 32 * KCH / 64; ++i) {
        const int at = i * 64 + lane, r = at / KCH, chunk = at % KCH;
        const uint4 bits = copy_area[r * KCH + (chunk ^ (r & 7))];
        if (first + r < T)
          *reinterpret_cast<uint4*>(gb_base + static_cast<long long>(first + r) * E + 8 * chunk) = bits;
      }
      // delta of attention.cc:283-291 (uses the stored, rounded output)
      delta[c] = -half_swap_sum(partial);
      const float normalizer = a.normalizers[stats_base + q_load];
      lse[c] = -(a.maxima[stats_base + q_load] * kLog2e + __log2f(normalizer > 0.0f ? normalizer : 1.0f));
      if (h == 0 && q_row < T) {
        // the key-owned kernel starts its accumulators from these
        a.deltas[stats_base + q_row] = delta[c];
        a.lse2[stats_base + q_row] = lse[c] / scale2;
      }
    }
  }
  if constexpr (!PREPARED) __syncthreads();  // the copies are out of the ring

  // What the loop statement takes.  Row reads start from the ring's last stage (the loop
  // moves them on before each block), transposed reads from its first; channels 64
  // and up lie 128 bytes further on.  Requests: chunk (4 wave + i) 64 + lane of a
  // tile; those of i + 2 lie eight rows further on.  An instruction's offset of 1024 i
  // moves the LDS and the global address: taken out of the latter again.
  const int base = static_cast<int>(lds_address(lds));
  int row_read[4], tr_read[2];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    row_read[ks] = base + (kRing - 1) * kStageBytes + tile_row_read<D>(n, 2 * ks + h);
#pragma unroll
  for (int db = 0; db < 2; ++db) tr_read[db] = base + tile_transpose_read<D>(lane, db);
  const uint32_t fill[2] = {tile_fill_offset<D>(wave * 256 + lane, kv_stride),
                            tile_fill_offset<D>(wave * 256 + 64 + lane, kv_stride) - 1024u};
  const uint32_t kv_bytes = static_cast<uint32_t>(((T - 1) * kv_stride + D) * 2);
  const int32x4 k_rsrc = make_rsrc(k_base, kv_bytes), v_rsrc = make_rsrc(v_base, kv_bytes);
  const uint32_t lds_q = __builtin_amdgcn_readfirstlane(lds_address(lds) + wave * 4096);
  const uint32_t k_step = static_cast<uint32_t>(32 * kv_stride * 2);
  const uint32_t k_eight = static_cast<uint32_t>(8 * kv_stride * 2) - 2048u;
  const uint32_t scale2_bits = __builtin_amdgcn_readfirstlane(__float_as_uint(scale2));
  // key blocks up to the wave's last query; a wave that has fewer than the
  // workgroup stays for the remaining steps (one more than blocks)
  const int steps = min(q0 + 127, T - 1) / 32 + 2;
  const int blocks = wave_first < T ? min(wave_first + 63, T - 1) / 32 + 1 : 0;
  const uint32_t wave_blocks = __builtin_amdgcn_readfirstlane(blocks);
  uint32_t idle_steps = __builtin_amdgcn_readfirstlane(blocks > 0 ? steps - 1 - blocks : steps);
  const uint32_t diagonal = __builtin_amdgcn_readfirstlane(wave_first / 32);
  const int bound = wave_first + n - 4 * h;
  const long long out_at = (seq_row0 + wave_first) * a.dq_row + head * D;
  const int rows_left = T - wave_first;
  const uint32_t out_bytes =
      rows_left <= 0 ? 0u : static_cast<uint32_t>((min(rows_left, 64) - 1) * a.dq_row + D) * 4u;
  const int32x4 dq_rsrc = make_rsrc(a.dq + out_at, out_bytes);
  const uint32_t area = __builtin_amdgcn_readfirstlane(lds_address(lds) + wave * 8192);
  uint32_t k_offset = 0, fill_stage = 0, row_stage = (kRing - 1) * kStageBytes, tr_stage = 0, block_count = 0;
  uint32_t saved_m0, temp0, temp1;
  asm volatile(FLASH_DQ_D128_ASM
               : FLASH_DQ_D128_ROWS(qf, gf), FLASH_DQ_D128_ADDRESSES(row_read, tr_read),
                 [koff] "+&s"(k_offset), [fstage] "+&s"(fill_stage), [rstage] "+&s"(row_stage),
                 [tstage] "+&s"(tr_stage), [idle] "+&s"(idle_steps), [bcount] "+&s"(block_count),
                 [m0save] "=&s"(saved_m0), [t0] "=&s"(temp0), [t1] "=&s"(temp1)
               : FLASH_DQ_D128_LANES(fill, lse, delta, bound),
                 [krsrc] "s"(k_rsrc), [vrsrc] "s"(v_rsrc), [dqrsrc] "s"(dq_rsrc),
                 [scale2] "s"(scale2_bits), [scale] "s"(a.scale), [kstep] "s"(k_step),
                 [keight] "s"(k_eight), [ldsq] "s"(lds_q), [nblk] "s"(wave_blocks),
                 [diagonal] "s"(diagonal), [area] "s"(area),
                 [rowbytes] "s"(static_cast<uint32_t>(a.dq_row * 4))
               : FLASH_DQ_D128_CLOBBERS);
}

}  // namespace

int launch_flash_dq_wide(hipStream_t stream, const FlashBackwardArgs& a) {
  const long long grid = (a.context_length + 127LL) / 128 * a.num_heads * a.sequences;
  if (grid > 0x7fffffffLL) return PLUTO_HIP_EINVAL;
  if (a.d_out)
    flash_dq_wide_kernel<false><<<static_cast<unsigned>(grid), kThreads, 0, stream>>>(a);
  else
    flash_dq_wide_kernel<true><<<static_cast<unsigned>(grid), kThreads, 0, stream>>>(a);
  return launch_status();
}

}  // namespace pluto_hip
