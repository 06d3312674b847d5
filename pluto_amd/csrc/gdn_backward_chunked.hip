// Chunked backward of the gated delta rule for 128 x 128 heads: the same
// gradients as the token-by-token kernels of gdn_backward.hip
// (RecurrenceForward / RecurrenceBackward, src/llm/layers/
// sequence_delta_net.cc:55-102 and :171-253), computed 64 tokens at a time on
// the matrix cores in FP32, and with one saved state per chunk instead of one per
// token.
//
// For a chunk entered with state S (rows: key channels, columns: value
// channels), tokens i = 0..63, G_i the running sum of the log decays inside
// the chunk, E_i = exp(G_i), D_ij = exp(G_i - G_j) (i >= j), L_j = exp(G_63 -
// G_j), q^ and k^ the normalised (and, for q, scaled) rows:
//   A   = strict_lower(beta_i (k^_i . k^_j) D_ij)        T = (I + A)^-1
//   W   = T diag(beta E) K^                               U = T diag(beta) V
//   Dl  = U - W S                 (the 64 delta rows of the chunk)
//   P   = lower((q^_i . k^_j) D_ij)
//   O   = diag(E) Q^ S + P Dl
//   S'  = E_63 S + (diag(L) K^)^T Dl
// which is the recurrence S <- decay S; delta = beta (v - S^T k^); S += k^ x
// delta; o = S^T q^ unrolled over the chunk.  In reverse, from the gradient dS'
// of the state leaving the chunk,
//   dDl = P^T dO + diag(L) K^ dS'
//   dS  = E_63 dS' + (diag(E) Q^)^T dO - W^T dDl.
// The kernels, in launch order:
//   chunk_prepare_kernel           T, W, U, P of every chunk          (parallel)
//   chunk_states_forward_kernel    S entering every chunk, Dl, O      (sequential)
//     -- the caller turns O into dO here --
//   chunk_states_backward_kernel   dS' leaving every chunk, dDl       (sequential)
//   chunk_gradients_kernel         everything else                    (parallel)
// The sequential kernels run one workgroup per (head, 16 or 32 value columns).
// Eliminating Dl instead makes both recurrences one 128 x 128 matrix a chunk
// (S' = M S + B) whose product is one link of the chain instead of two, but M, its
// transpose, B and the offsets of the reverse recurrence are four 64 KiB records a
// chunk that have to be computed, written and read.
//
// Layout of the records.  A memory instruction whose lanes take 16 bytes each of 16
// rows costs a compute unit about 40 clocks, one that takes a contiguous KiB 16, and
// the sequential kernels issue more of them than their matrix instructions hide.
// Every matrix is therefore kept in operand order: rows(M) is M in blocks of 16 rows
// by 4 columns, blocks of a row block after each other, so that the lanes of an
// operand of rows and of four contraction elements a lane read 1 KiB (16 x 16
// tiles) or 256-byte pieces (32 x 32 tiles).  columns(M) is rows(M^T): an
// accumulator, whose lanes are columns and whose registers are four neighbouring rows,
// is stored in that order as it is.
//
// Matrix products of the parallel kernels run on v_mfma_f32_32x32x2_f32 and
// v_mfma_f32_16x16x4_f32; the triangular factors are multiplied by halves.  Those of the
// sequential kernels take three bf16 pieces of a factor (bf16_pieces.h), of bf16 activations'
// keys and queries one.
#include "gdn.h"

#include "bf16_pieces.h"

#include <type_traits>

namespace pluto_hip {
namespace {

constexpr int kC = 64;       // tokens per chunk
constexpr int kD = 128;      // key and value channels per head
constexpr int kTile = 16;    // value columns of a tile of the sequential kernels
constexpr int kWide = kC * kD;     // elements of a [64, 128] record
constexpr int kSquare = kC * kC;   // elements of a [64, 64] record
constexpr int kState = kD * kD;    // elements of a state
constexpr int kWidePad = kD + 4;   // LDS rows: 16-byte aligned, neighbours four banks apart
constexpr int kSquarePad = kC + 4;

// Per (head, chunk) records in the workspace, in floats.
struct Records {
  // of a key head                                                        [64][128]
  float *q_rows = nullptr, *q_columns = nullptr, *k_rows = nullptr, *k_columns = nullptr;
  uint16_t* keys = nullptr;   // or, of bf16 activations, the four as KeyOperands has them
  float *w_rows, *w_columns;                          // W              [64][128]
  float *u_columns, *dl_rows, *ddl_rows;              // U, Dl, dDl     [64][128]
  float *p_rows, *p_columns;                          // P               [64][64]
  float *t_columns;                                   // T               [64][64]
  float *kkd;                 // columns(strict_lower((k^_i . k^_j) D_ij)) [64][64]
  float *gates;               // [8][64], see Gate
  float *s0, *ds1;            // rows(state entering the chunk), rows(gradient of the one leaving)
};

// Rows of a gates record; q^ and k^ are the convolved activations' rows times kQScale
// and kKScale (zero beyond the sequence).
// kEQ and kLK: kE and kL times the factors that the bf16 rows of Q and K lack.
enum Gate { kG, kBeta, kQScale, kKScale, kE, kL, kEQ, kLK, kGateRows };

// FP32: q and k, rows and columns; bf16: KeyOperands.
constexpr size_t key_record_floats(bool bf16) { return (bf16 ? 2 : 4) * static_cast<size_t>(kWide); }
constexpr size_t kRecordFloats = 5 * static_cast<size_t>(kWide) + 4 * kSquare + kGateRows * kC +
                                 2 * static_cast<size_t>(kState);

struct ChunkedArgs {
  const void* post = nullptr;      // [T, channels], bf16 where they are rounded to it, else FP32
  const uint16_t* a = nullptr;     // bf16 [T, vh]
  const uint16_t* b = nullptr;
  const float* a_log = nullptr;
  const float* dt_bias = nullptr;
  const float* dcore = nullptr;    // [T, vh, 128]
  float* core = nullptr;           // [T, vh, 128]
  float* dpost = nullptr;          // [T, channels]: the value part is written
  float* qk_partials = nullptr;    // [T, vh, 2, 128]
  float* da = nullptr;             // [T, vh]
  float* db = nullptr;
  float* scalar_partials = nullptr;  // [chunks, vh, 2]: a chunk's part of d A_log and d dt_bias
  Records r;
  int length = 0, chunks = 0, kh = 0, vh = 0;
  bool round = true;
};

__device__ inline float round_if(float x, bool round) { return round ? round_to_bf16(x) : x; }

__device__ inline floatx16 zero_tile() {
  floatx16 z;
#pragma unroll
  for (int i = 0; i < 16; ++i) z[i] = 0.0f;
  return z;
}

// Row of accumulator register i of a 32 x 32 tile in a lane of half h; the
// column is lane % 32.
__device__ inline int tile_row(int i, int h) { return 8 * (i / 4) + 4 * h + i % 4; }

__device__ inline float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ inline void store4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
__device__ inline float4 scaled(float4 v, float s) {
  return make_float4(v.x * s, v.y * s, v.z * s, v.w * s);
}

// acc += a b over four contraction elements a lane half: the halves of a wave take
// alternate groups of four (element e of half h is 8 s + 4 h + e, the row that
// accumulator register 4 s + e of that half holds), so that both operands can come
// in 16-byte pieces and an accumulator can be an operand as it is.
__device__ inline floatx16 mma(floatx16 acc, float4 a, float4 b) {
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, b.x, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, b.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, b.z, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, b.w, acc, 0, 0, 0);
  return acc;
}

// The same for 16 x 16 tiles: quarter q of the wave takes elements 16 s + 4 q + e, the
// row that register e of that quarter holds.
__device__ inline floatx4 mma16(floatx4 acc, float4 a, float4 b) {
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc, 0, 0, 0);
  return acc;
}
__device__ inline floatx4 mma16(floatx4 acc, float4 a, floatx4 b) {
  return mma16(acc, a, make_float4(b[0], b[1], b[2], b[3]));
}

__device__ inline float4 gather4(const float* p, int stride) {
  return make_float4(p[0], p[stride], p[2 * stride], p[3 * stride]);
}

__device__ inline void keep_order() { __builtin_amdgcn_sched_barrier(0); }

// Barrier for data exchanged through LDS only: pending global loads and
// stores stay in flight across it.
__device__ inline void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Sums over the 32 lanes of a half wave of sixteen values at once: lanes i and 16 + i of a
// half return the sum of value i.  Every step halves the values a lane holds; its
// partners mirror rows of 16, 8, 4 and 2 lanes, which is part of a vector addition.
__device__ inline float half_sums(const float (&values)[16]) {
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = values[i];
  const int n = threadIdx.x;
  auto step = [&](auto control, int width) {
    const bool upper = n & width;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (i >= width) break;
      const float kept = upper ? v[i + width] : v[i], sent = upper ? v[i] : v[i + width];
      v[i] = kept + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sent), decltype(control)::value,
                                                               0xf, 0xf, true));
    }
  };
  step(std::integral_constant<int, 0x140>(), 8);  // row_mirror
  step(std::integral_constant<int, 0x141>(), 4);  // row_half_mirror
  step(std::integral_constant<int, 0x4E>(), 2);   // quad_perm 2, 3, 0, 1
  step(std::integral_constant<int, 0xB1>(), 1);   // quad_perm 1, 0, 3, 2
  return v[0] + __shfl_xor(v[0], 16, 64);
}

__device__ inline float4 unpacked(uint2 bits) {
  return make_float4(__uint_as_float(bits.x << 16), __uint_as_float(bits.x & 0xffff0000u),
                     __uint_as_float(bits.y << 16), __uint_as_float(bits.y & 0xffff0000u));
}

// Memory behind a buffer descriptor: a lane's byte offset, computed once, and a uniform
// byte offset, so that a kernel keeps no addresses in vector registers.  Rows of
// TOKENS may lie beyond the end: there the sum is the offset the descriptor checks,
// reads give zero and writes are dropped, without a branch.
template <bool TOKENS>
struct Memory {
  const float* base;
  uint32_t bytes;
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ Memory(const float* base_, size_t elements)
      : base(base_), bytes(static_cast<uint32_t>(elements * 4)),
        rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, static_cast<int>(bytes),
                                               0x00020000)) {}
  __device__ int32x4 words() const { return make_rsrc(base, bytes); }
  __device__ float get(unsigned lane, unsigned uniform) const {
    const auto bits = TOKENS ? __builtin_amdgcn_raw_buffer_load_b32(rsrc, lane + uniform, 0, 0)
                             : __builtin_amdgcn_raw_buffer_load_b32(rsrc, lane, uniform, 0);
    return __uint_as_float(bits);
  }
  __device__ float2 get2(unsigned lane, unsigned uniform) const {
    const auto bits = TOKENS ? __builtin_amdgcn_raw_buffer_load_b64(rsrc, lane + uniform, 0, 0)
                             : __builtin_amdgcn_raw_buffer_load_b64(rsrc, lane, uniform, 0);
    return __builtin_bit_cast(float2, bits);
  }
  __device__ float4 get4(unsigned lane, unsigned uniform) const {
    const auto bits = TOKENS ? __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane + uniform, 0, 0)
                             : __builtin_amdgcn_raw_buffer_load_b128(rsrc, lane, uniform, 0);
    return __builtin_bit_cast(float4, bits);
  }
  __device__ float4 get4_bf16(unsigned lane, unsigned uniform) const {
    return unpacked(__builtin_bit_cast(uint2, get2(lane, uniform)));
  }
  __device__ uint32_t get_bf16(unsigned lane, unsigned uniform) const {
    return static_cast<uint16_t>(TOKENS ? __builtin_amdgcn_raw_buffer_load_b16(rsrc, lane + uniform, 0, 0)
                                        : __builtin_amdgcn_raw_buffer_load_b16(rsrc, lane, uniform, 0));
  }
  // elements `stride` bytes apart
  __device__ float4 gather4(unsigned lane, unsigned uniform, unsigned stride) const {
    return make_float4(get(lane, uniform), get(lane, uniform + stride), get(lane, uniform + 2 * stride),
                       get(lane, uniform + 3 * stride));
  }
  __device__ void put(float v, unsigned lane, unsigned uniform) const {
    if (TOKENS)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rsrc, lane + uniform, 0, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rsrc, lane, uniform, 0);
  }
  // The uniform part is added in either case: a store of four registers at a scalar offset
  // still reads them when the next instruction may already write them (seen as a fourth
  // element taken from a later value), and the compiler keeps the two apart only where
  // the offset is no register.
  __device__ void put4(float4 v, unsigned lane, unsigned uniform) const {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint32x4, v), rsrc, lane + uniform, 0, 0);
  }
};
using Record = Memory<false>;
using Tokens = Memory<true>;

// One chunk of one head.  Tokens beyond the sequence have zero rows, scales, beta and
// gradients.
struct ChunkView {
  const ChunkedArgs& a;
  size_t rec;
  int t0, head, tokens, channels;
  unsigned post_bytes, row_bytes, out_bytes;  // a token's row in the activations, their gradients, and dO and O
  const float* gates;
  __device__ ChunkView(const ChunkedArgs& args, int chunk, int head_)
      : a(args), rec(static_cast<size_t>(head_) * args.chunks + chunk), t0(chunk * kC), head(head_),
        tokens(min(args.length - t0, kC)), channels(2 * args.kh * kD + args.vh * kD),
        post_bytes(channels * (args.round ? 2 : 4)), row_bytes(channels * 4), out_bytes(args.vh * kD * 4),
        gates(args.r.gates + rec * kGateRows * kC) {}
  __device__ Tokens activations(int column) const {
    const int bytes = a.round ? 2 : 4;
    return Tokens(reinterpret_cast<const float*>(static_cast<const char*>(a.post) +
                                                 (static_cast<size_t>(t0) * channels + column) * bytes),
                  (static_cast<size_t>(tokens) * channels - column) * bytes / 4);
  }
  __device__ int key_head() const { return head / (a.vh / a.kh); }
  __device__ int value_column() const { return (2 * a.kh + head) * kD; }
  __device__ Record key(const float* records) const {
    return Record(records + (static_cast<size_t>(key_head()) * a.chunks + t0 / kC) * kWide, kWide);
  }
  __device__ Tokens v() const { return activations(value_column()); }
  __device__ Tokens dv() const {
    return Tokens(a.dpost + static_cast<size_t>(t0) * channels + value_column(),
                  static_cast<size_t>(tokens) * channels - value_column());
  }
  __device__ Tokens heads(const float* base) const {  // O, dO
    return Tokens(base + (static_cast<size_t>(t0) * a.vh + head) * kD,
                  (static_cast<size_t>(tokens) * a.vh - head) * kD);
  }
  __device__ Tokens qk_partials() const {
    return Tokens(a.qk_partials + (static_cast<size_t>(t0) * a.vh + head) * 2 * kD,
                  (static_cast<size_t>(tokens) * a.vh - head) * 2 * kD);
  }
  __device__ Record wide(const float* records) const { return Record(records + rec * kWide, kWide); }
  __device__ Record square(const float* records) const { return Record(records + rec * kSquare, kSquare); }
  __device__ Record state(const float* records) const { return Record(records + rec * kState, kState); }
};

// Byte offsets in rows(M) of a matrix with COLUMNS columns: four columns of sixteen rows,
// and a whole 16 x 16 operand.
constexpr unsigned kPiece = 16 * 4 * 4, kOperand = 4 * kPiece;
template <int COLUMNS>
__device__ constexpr unsigned piece_at(int row_block, int quad) {
  return (row_block * (COLUMNS / 4) + quad) * kPiece;
}
// The lane of half h and row n of a 32 x 32 operand: its quads are 2 s + h.
template <int COLUMNS>
__device__ inline unsigned lane_piece(int h, int n) {
  return piece_at<COLUMNS>(n / 16, h) + n % 16 * 16;
}

// ---------------------------------------------------------------------------
// The rows of Q and K as operands of the sequential kernels where the activations are
// bf16: a row times a power of two, which is what its scale is but for a fraction in [1, 2),
// is bf16 as well and one piece instead of three, half the bytes and half the products; the
// fractions go with the other factors of a token (kEQ, kLK).  Operand (row block, step) is 1 KiB: lane
// (n, quarter) has elements 32 step + 16 (e / 4) + 4 quarter + e % 4 of row n of the block.
struct KeyOperands {
  static constexpr unsigned kRowsOfK = 0, kRowsOfQ = 2 * kWide, kColumnsOfK = 4 * kWide, kColumnsOfQ = 6 * kWide;
  static constexpr unsigned kChunkBytes = 8 * kWide;
  Record memory;
  __device__ KeyOperands(const ChunkedArgs& a, int key_head)
      : memory(reinterpret_cast<const float*>(a.r.keys) + static_cast<size_t>(key_head) * a.chunks * (kChunkBytes / 4),
               static_cast<size_t>(a.chunks) * (kChunkBytes / 4)) {}
  __device__ void put(const uint2 (&bits)[2], unsigned lane, unsigned uniform) const {
    memory.put4(__builtin_bit_cast(float4, make_uint4(bits[0].x, bits[0].y, bits[1].x, bits[1].y)), lane, uniform);
  }
  __device__ bf16x8 get(unsigned lane, unsigned uniform) const {
    return __builtin_bit_cast(bf16x8, memory.get4(lane, uniform));
  }
};
__device__ inline float fraction_of(float scale) {
  return __uint_as_float((__float_as_uint(scale) & 0x007fffffu) | 0x3f800000u);
}
__device__ inline float4 product(float4 a, float4 b) { return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w); }

// T, W, U, P and the gates of one chunk.  The inverse is made by blocks: the four 16 x 16 diagonal blocks by forward
// substitution, one wave each, then -T22 A21 T11 twice on the matrix cores (a
// substitution over all 64 rows by one wave held the other three up for a third of
// the kernel).
//
// BF16: the activations are bf16, and the rows of K and Q are kept as such, each times the
// power of two in its scale (KeyOperands), in row-major tiles of 16 KiB as in mfma_tile.h.  The
// products of rows are then exact, those by T take three pieces of T and one of K or V, and
// with 52 KiB of LDS and 168 registers three workgroups share a compute unit instead of two.
// 2048 tokens of 48 heads 108.5 -> 64 us (260 MB, 50 us at the rate of a copy; 80.6 while bf16
// activations came as FP32 and these rows left as FP32 as well), one chunk 26 -> 18: every
// product took the FP32 instruction, 34 us of it.
template <bool BF16>
struct PrepareSmem;
template <>
struct PrepareSmem<false> {
  float k[kC][kWidePad];
  union {
    float q[kC][kWidePad];
    struct {
      float a[kC][kSquarePad], t[kC][kSquarePad];
    };
  };
  float g[kC], beta[kC], fk[kC];
  __device__ float (&w())[kC][kWidePad] { return k; }
};
template <>
struct PrepareSmem<true> {
  unsigned char k_tile[kC * kD * 2];
  union {
    unsigned char q_tile[kC * kD * 2];
    struct {
      float a[kC][kSquarePad], t[kC][kSquarePad];
    };
    float w_rows[kC][kWidePad];
  };
  float g[kC], beta[kC], fk[kC], q_fraction[kC], k_fraction[kC];
  __device__ float (&w())[kC][kWidePad] { return w_rows; }
};
// Place of a 16-byte piece of a row, of four rows of a column as a transpose read has them.
__device__ inline int tile_piece(int row, int piece) { return (row * (kD / 8) + (piece ^ tile_swizzle(row))) * 16; }
__device__ inline int tile_quad(int row, int column) { return tile_piece(row, column / 8) + column % 8 * 2; }

template <bool BF16>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(BF16 ? 3 : 2, BF16 ? 3 : 2)))
chunk_prepare_kernel(ChunkedArgs a) {
  __shared__ __attribute__((aligned(1024))) PrepareSmem<BF16> sm;
  const ChunkView v(a, blockIdx.x, blockIdx.y);
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int h = lane / 32, n = lane % 32, quarter = lane / 16, n16 = lane % 16;
  float* gates = a.r.gates + v.rec * kGateRows * kC;

  // normalised rows (1e-6 added to the sums of squares, sequence_delta_net.cc:84-85) of
  // sixteen tokens a wave, a row a quarter of it: channels 4 n16 .. + 3 and 64 further a
  // lane.  A row's squares are added by the tree of wave_sum over channels c and c +
  // 64, so that the scales are those of the other kernels to the bit (an error of a
  // scale moves a whole row of outputs over the ties of their rounding); the trees of
  // eight rows share their steps.
  {
    const float norm_scale = sqrtf(static_cast<float>(kD)), inverse_norm_scale = 1.0f / norm_scale;
    const Tokens q = v.activations(v.key_head() * kD), k = v.activations((a.kh + v.key_head()) * kD);
    const unsigned at = (16 * wave + quarter) * v.post_bytes + (BF16 ? 8 : 16) * n16;
    auto four = [&](const Tokens& from, unsigned uniform) {
      if constexpr (BF16)
        return from.get4_bf16(at, uniform);
      else
        return from.get4(at, uniform);
    };
    float rows[8][2][4], squares[8][4];  // q^ and k^ of rows quarter, 4 + quarter, ...
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const unsigned uniform = 4 * g * v.post_bytes + (BF16 ? 128 : 256) * j;
        const float4 qv = four(q, uniform), kv = four(k, uniform);
        rows[2 * g][j][0] = qv.x, rows[2 * g][j][1] = qv.y, rows[2 * g][j][2] = qv.z, rows[2 * g][j][3] = qv.w;
        rows[2 * g + 1][j][0] = kv.x, rows[2 * g + 1][j][1] = kv.y, rows[2 * g + 1][j][2] = kv.z,
        rows[2 * g + 1][j][3] = kv.w;
      }
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        squares[r][c] = rows[r][0][c] * rows[r][0][c] + rows[r][1][c] * rows[r][1][c];
    // lane n16 is left with row n16 / 2
#pragma unroll
    for (int width = 4; width > 0; width /= 2) {
      const bool upper = n16 & (2 * width);
#pragma unroll
      for (int r = 0; r < width; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float kept = upper ? squares[r + width][c] : squares[r][c];
          const float sent = upper ? squares[r][c] : squares[r + width][c];
          squares[r][c] = kept + __shfl_xor(sent, 2 * width, 64);
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) squares[0][c] += __shfl_xor(squares[0][c], 1, 64);
    const float inverse =
        rsqrtf((squares[0][0] + squares[0][2]) + (squares[0][1] + squares[0][3]) + 1e-6f);
    // x / norm_scale, rounded once: quotient, remainder and its part of the quotient
    auto normed = [&](float x) {
      const float y = x * inverse_norm_scale;
      return fmaf(fmaf(-y, norm_scale, x), inverse_norm_scale, y);
    };
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int i = 16 * wave + 4 * g + quarter;
      const bool ok = i < v.tokens;
      const float iq = ok ? __shfl(inverse, 16 * quarter + 4 * g, 64) : 0.0f;
      const float ik = ok ? __shfl(inverse, 16 * quarter + 4 * g + 2, 64) : 0.0f;
      const float q_scale = iq / norm_scale;
      // a scale's power of two and its fraction in [1, 2); a zero has neither
      const float q_fraction = q_scale == 0.0f ? 0.0f : fraction_of(q_scale);
      const float k_fraction = ik == 0.0f ? 0.0f : fraction_of(ik);
      const float q_power = __uint_as_float(__float_as_uint(q_scale) & 0x7f800000u);
      const float k_power = __uint_as_float(__float_as_uint(ik) & 0x7f800000u);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float(&qv)[4] = rows[2 * g][j], (&kv)[4] = rows[2 * g + 1][j];
        if constexpr (BF16) {
          const int place = tile_quad(i, 4 * n16 + 64 * j);
          *reinterpret_cast<uint2*>(sm.q_tile + place) = make_uint2(pack_bf16(qv[0] * q_power, qv[1] * q_power),
                                                                    pack_bf16(qv[2] * q_power, qv[3] * q_power));
          *reinterpret_cast<uint2*>(sm.k_tile + place) = make_uint2(pack_bf16(kv[0] * k_power, kv[1] * k_power),
                                                                    pack_bf16(kv[2] * k_power, kv[3] * k_power));
        } else {
          store4(&sm.q[i][4 * n16 + 64 * j], make_float4(normed(qv[0] * iq), normed(qv[1] * iq), normed(qv[2] * iq),
                                                         normed(qv[3] * iq)));
          store4(&sm.k[i][4 * n16 + 64 * j], make_float4(kv[0] * ik, kv[1] * ik, kv[2] * ik, kv[3] * ik));
        }
      }
      if (n16 == 0) {
        gates[kQScale * kC + i] = q_scale;
        gates[kKScale * kC + i] = ik;
        if constexpr (BF16) sm.q_fraction[i] = q_fraction, sm.k_fraction[i] = k_fraction;
      }
    }
  }
  // gates (sequence_delta_net.cc:88-96); tokens beyond the sequence neither
  // decay nor write
  float e = 0.0f, l = 0.0f, beta = 0.0f;
  if (wave == 0) {
    const int t = v.t0 + lane;
    float g = 0.0f;
    if (lane < v.tokens) {
      const float alpha =
          bf16_bits_to_float(a.a[static_cast<size_t>(t) * a.vh + v.head]) + a.dt_bias[v.head];
      const float softplus = fmaxf(alpha, 0.0f) + logf(1.0f + expf(-fabsf(alpha)));
      g = -expf(a.a_log[v.head]) * softplus;
      const float bv = bf16_bits_to_float(a.b[static_cast<size_t>(t) * a.vh + v.head]);
      beta = round_if(1.0f / (1.0f + expf(-bv)), a.round);
    }
    // one after the other: an error of the running sum scales whole rows
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < kC; ++i) {
      const float next = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g), i));
      sum = lane >= i ? sum + next : sum;
    }
    g = sum;
    e = expf(g), l = expf(__shfl(g, 63, 64) - g);
    gates[kG * kC + lane] = g;
    gates[kBeta * kC + lane] = beta;
    gates[kE * kC + lane] = e;
    gates[kL * kC + lane] = l;
    sm.g[lane] = g;
    sm.beta[lane] = beta;
    if constexpr (!BF16) sm.fk[lane] = beta * e;
  }
  __syncthreads();
  if constexpr (BF16)
    if (wave == 0) {
      gates[kEQ * kC + lane] = e * sm.q_fraction[lane];
      gates[kLK * kC + lane] = l * sm.k_fraction[lane];
      sm.fk[lane] = beta * e * sm.k_fraction[lane];
    }
  // k^ k^T and q^ k^T by 16 x 16 tiles on and below the diagonal: wave w takes row w of
  // the first and row 3 - w of the second, five tiles
  const bool first_of_group = v.head % (a.vh / a.kh) == 0;
  floatx4 kk[4], qk[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) kk[b] = qk[b] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (BF16) {
    auto row_operand = [&](const unsigned char* tile, int block, int s) {
      return as_bf16x8(*reinterpret_cast<const uint4*>(tile + tile_piece(16 * block + n16, 4 * s + quarter)));
    };
#pragma unroll
    for (int s = 0; s < kD / 32; ++s) {
      const bf16x8 kr = row_operand(sm.k_tile, wave, s), qr = row_operand(sm.q_tile, 3 - wave, s);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        if (b > wave && b > 3 - wave) continue;
        const bf16x8 kc = row_operand(sm.k_tile, b, s);
        if (b <= wave) kk[b] = mfma16(kr, kc, kk[b]);
        if (b <= 3 - wave) qk[b] = mfma16(qr, kc, qk[b]);
      }
    }
    if (first_of_group) {
      const KeyOperands operands(a, v.key_head());
      const unsigned operand_at = 16 * lane + blockIdx.x * KeyOperands::kChunkBytes;
      const int row = 16 * wave + n16;
#pragma unroll
      for (int s = 0; s < kD / 32; ++s) {
        uint2 kr[2], qr[2];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const int place = tile_quad(row, 32 * s + 16 * half + 4 * quarter);
          kr[half] = *reinterpret_cast<const uint2*>(sm.k_tile + place);
          qr[half] = *reinterpret_cast<const uint2*>(sm.q_tile + place);
        }
        operands.put(kr, operand_at, KeyOperands::kRowsOfK + (4 * wave + s) * 1024);
        operands.put(qr, operand_at, KeyOperands::kRowsOfQ + (4 * wave + s) * 1024);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int s = 0; s < kC / 32; ++s) {
          const int b = 2 * wave + t;
          uint2 kc[2], qc[2];
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            const int first = 32 * s + 16 * half + 4 * quarter;
            const int place = tile_quad(first + n16 / 4, 16 * b + 4 * (n16 % 4));
            kc[half] = lds_transpose_read(sm.k_tile, place);
            qc[half] = lds_transpose_read(sm.q_tile, place);
          }
          operands.put(kc, operand_at, KeyOperands::kColumnsOfK + (2 * b + s) * 1024);
          operands.put(qc, operand_at, KeyOperands::kColumnsOfQ + (2 * b + s) * 1024);
        }
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float k_col = sm.k_fraction[16 * b + n16];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kk[b][e] *= sm.k_fraction[16 * wave + 4 * quarter + e] * k_col;
        qk[b][e] *= sm.q_fraction[16 * (3 - wave) + 4 * quarter + e] * k_col;
      }
    }
  } else {
    const Record k_rows = v.key(a.r.k_rows), q_rows = v.key(a.r.q_rows);
#pragma unroll
    for (int s = 0; s < kD / 16; ++s) {
      const float4 kr = load4(&sm.k[16 * wave + n16][16 * s + 4 * quarter]);
      const float4 qr = load4(&sm.q[16 * (3 - wave) + n16][16 * s + 4 * quarter]);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        if (b > wave && b > 3 - wave) continue;
        const float4 kc = load4(&sm.k[16 * b + n16][16 * s + 4 * quarter]);
        if (b <= wave) kk[b] = mma16(kk[b], kr, kc);
        if (b <= 3 - wave) qk[b] = mma16(qk[b], qr, kc);
      }
      if (first_of_group) {
        k_rows.put4(kr, 16 * lane, piece_at<kD>(wave, 4 * s));
        q_rows.put4(qr, 16 * lane, piece_at<kD>(3 - wave, 4 * s));
      }
    }
    if (first_of_group) {
      const Record k_columns = v.key(a.r.k_columns), q_columns = v.key(a.r.q_columns);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int b = 2 * wave + t;
          k_columns.put4(gather4(&sm.k[16 * s + 4 * quarter][16 * b + n16], kWidePad), 16 * lane,
                         piece_at<kC>(b, 4 * s));
          q_columns.put4(gather4(&sm.q[16 * s + 4 * quarter][16 * b + n16], kWidePad), 16 * lane,
                         piece_at<kC>(b, 4 * s));
        }
    }
  }
  lds_barrier();  // the rows of q^ make room for P, then A, and for T
  {
    const Record kkd = v.square(a.r.kkd), p_columns = v.square(a.r.p_columns), p_rows = v.square(a.r.p_rows);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      float p[4], masked[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = 4 * quarter + e, col = 16 * b + n16;
        const int k_at = 16 * wave + row, q_at = 16 * (3 - wave) + row;
        masked[e] = k_at > col ? kk[b][e] * expf(sm.g[k_at] - sm.g[col]) : 0.0f;
        p[e] = q_at >= col ? qk[b][e] * expf(sm.g[q_at] - sm.g[col]) : 0.0f;
        kk[b][e] = sm.beta[k_at] * masked[e];
        sm.a[q_at][col] = p[e];
        sm.t[k_at][col] = 0.0f;
      }
      kkd.put4(make_float4(masked[0], masked[1], masked[2], masked[3]), 16 * lane, piece_at<kC>(b, 4 * wave));
      p_columns.put4(make_float4(p[0], p[1], p[2], p[3]), 16 * lane, piece_at<kC>(b, 4 * (3 - wave)));
    }
    lds_barrier();
#pragma unroll
    for (int s = 0; s < 4; ++s)
      p_rows.put4(load4(&sm.a[16 * wave + n16][16 * s + 4 * quarter]), 16 * lane, piece_at<kC>(wave, 4 * s));
    lds_barrier();
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) sm.a[16 * wave + 4 * quarter + e][16 * b + n16] = kk[b][e];
  }
  lds_barrier();
  {
    // diagonal block `wave`, column n16
    const int first = 16 * wave;
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float row[16];
#pragma unroll
      for (int j = 0; j < i; j += 4) {
        const float4 four = load4(&sm.a[first + i][first + j]);
        row[j] = four.x, row[j + 1] = four.y, row[j + 2] = four.z, row[j + 3] = four.w;
      }
      float s = i == n16 ? 1.0f : 0.0f;
#pragma unroll
      for (int j = 0; j < i; ++j) s -= row[j] * x[j];
      x[i] = s;
    }
    if (quarter == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) sm.t[first + i][first + n16] = x[i];
    }
  }
  lds_barrier();
  const floatx4 none = {0.0f, 0.0f, 0.0f, 0.0f};
  if (wave % 2 == 1) {
    // the block left of diagonal block `wave`: -T_ww A_w,w-1 T_w-1,w-1
    const int r0 = 16 * wave, c0 = r0 - 16;
    const floatx4 y = mma16(none, load4(&sm.a[r0 + n16][c0 + 4 * quarter]),
                            gather4(&sm.t[c0 + 4 * quarter][c0 + n16], kSquarePad));
    const floatx4 z = mma16(none, load4(&sm.t[r0 + n16][r0 + 4 * quarter]), y);
#pragma unroll
    for (int e = 0; e < 4; ++e) sm.t[r0 + 4 * quarter + e][c0 + n16] = -z[e];
  }
  lds_barrier();
  {
    // rows 32.., columns ..31 by 16 x 16 tiles, tile (wave / 2, wave % 2)
    const int r0 = 32 + 16 * (wave / 2), c0 = 16 * (wave % 2);
    floatx4 z = none;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      if (m > wave / 2) continue;
      floatx4 y = none;
#pragma unroll
      for (int l = 0; l < 2; ++l)
        if (l >= wave % 2)
          y = mma16(y, load4(&sm.a[32 + 16 * m + n16][16 * l + 4 * quarter]),
                    gather4(&sm.t[16 * l + 4 * quarter][c0 + n16], kSquarePad));
      z = mma16(z, load4(&sm.t[r0 + n16][32 + 16 * m + 4 * quarter]), y);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) sm.t[r0 + 4 * quarter + e][c0 + n16] = -z[e];
  }
  // W = T diag(beta E) K^, U = T diag(beta) V: the wave owns 32 columns
  const int col = 32 * wave + n;
  const auto value_memory = v.v();
  float4 values[8];
  uint32_t value_bits[4][8];
  if constexpr (BF16) {
    const unsigned at = 4 * h * v.post_bytes + 2 * col;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        value_bits[s][e] = value_memory.get_bf16(at, (16 * s + 8 * (e / 4) + e % 4) * v.post_bytes);
  } else {
#pragma unroll
    for (int s = 0; s < 8; ++s)
      values[s] = value_memory.gather4(4 * h * v.post_bytes + 4 * col, 8 * s * v.post_bytes, v.post_bytes);
  }
  __builtin_amdgcn_sched_barrier(0);
  lds_barrier();
  {
    const Record t_columns = v.square(a.r.t_columns);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      t_columns.put4(gather4(&sm.t[16 * s + 4 * quarter][16 * wave + n16], kSquarePad), 16 * lane,
                     piece_at<kC>(wave, 4 * s));
    }
  }
  const Record w_columns = v.wide(a.r.w_columns), w_rows = v.wide(a.r.w_rows), u_columns = v.wide(a.r.u_columns);
  const unsigned column_at = piece_at<kC>(2 * wave, 0) + lane_piece<kC>(h, n);
  bf16x8 value_rows[4];
  if constexpr (BF16) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      auto pair = [&](int e) { return value_bits[s][e] | value_bits[s][e + 1] << 16; };
      value_rows[s] = as_bf16x8(make_uint4(pair(0), pair(2), pair(4), pair(6)));
    }
    keep_order();
  }
  floatx16 w[2];
#pragma unroll
  for (int ti = 0; ti < 2; ++ti) {
    floatx16 u = zero_tile();
    w[ti] = zero_tile();
#pragma unroll
    for (int s = 0; s < 4 * (ti + 1); ++s) {
      if constexpr (BF16) {
        if (s % 2 == 1) continue;
        const int k = 8 * s + 4 * h;  // .. + 3 and eight further
        const float4 t0 = load4(&sm.t[32 * ti + n][k]), t1 = load4(&sm.t[32 * ti + n][k + 8]);
        const Pieces by_k = split_eight(product(t0, load4(&sm.fk[k])), product(t1, load4(&sm.fk[k + 8])));
        const Pieces by_v = split_eight(product(t0, load4(&sm.beta[k])), product(t1, load4(&sm.beta[k + 8])));
        const bf16x8 keys =
            tile_transposed_operand<kD>(sm.k_tile + 8 * s * (kD * 2), tile_transpose_read<kD>(lane, wave), 0);
#pragma unroll
        for (int part = 2; part >= 0; --part) {
          w[ti] = mfma32(by_k.part[part], keys, w[ti]);
          u = mfma32(by_v.part[part], value_rows[s / 2], u);
        }
        continue;
      }
      const int k = 8 * s + 4 * h;
      if constexpr (!BF16) {
        const float4 t = load4(&sm.t[32 * ti + n][k]);
        w[ti] = mma(w[ti], product(t, load4(&sm.fk[k])), gather4(&sm.k[k][col], kWidePad));
        u = mma(u, product(t, load4(&sm.beta[k])), values[s]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned at = piece_at<kC>(0, 8 * ti + 2 * j);
      w_columns.put4(make_float4(w[ti][4 * j], w[ti][4 * j + 1], w[ti][4 * j + 2], w[ti][4 * j + 3]), column_at, at);
      u_columns.put4(make_float4(u[4 * j], u[4 * j + 1], u[4 * j + 2], u[4 * j + 3]), column_at, at);
    }
  }
  lds_barrier();  // the rows of k^, or T, make room for W
  auto& w_tile = sm.w();
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int i = 0; i < 16; ++i) w_tile[32 * ti + tile_row(i, h)][col] = w[ti][i];
  lds_barrier();
#pragma unroll
  for (int s = 0; s < 8; ++s)
    w_rows.put4(load4(&w_tile[16 * wave + n16][16 * s + 4 * quarter]), 16 * lane, piece_at<kD>(wave, 4 * s));
}

// ---------------------------------------------------------------------------
// The workgroups of the sequential kernels: TILES times sixteen value columns of a head.
// The slices of a head read the same matrices: they are given block numbers with the
// same remainder mod 8, which the hardware places on one XCD, so that all reads but the
// first are served by that XCD's L2.
struct Slice {
  int head, col0;
};
template <int TILES>
__device__ inline Slice slice_of_block(const ChunkedArgs& a) {
  constexpr int kSlices = kD / (kTile * TILES);
  if (a.vh % 8 == 0)
    return {static_cast<int>((blockIdx.x % 8) * (a.vh / 8) + blockIdx.x / (8 * kSlices)),
            static_cast<int>(blockIdx.x / 8 % kSlices * kTile * TILES)};
  return {static_cast<int>(blockIdx.x / kSlices), static_cast<int>(blockIdx.x % kSlices * kTile * TILES)};
}

// The state of a slice lives in accumulators: tile t of wave w holds rows 32 w + 16 t ..
// + 15 of sixteen columns.  Its pieces (see bf16_pieces.h) go to LDS in operand order,
// where the contraction index runs over both tiles: element e of quarter q of step s is row
// 32 s + 16 (e / 4) + 4 q + e % 4, so that a wave's accumulators are step w as they are,
// and of 64 tokens a wave's are half of step w / 2.  The left operands come from the
// records as FP32, two pieces of four columns a lane and step, and are split between the
// products of the step before.
// The right operands: states, deltas and their gradients may be as large as FP32 holds, or
// infinite where they have left its range, and give with the left ones (k^, q^, P, W: finite,
// or no number) what FP32 gives.  What bf16 would round to infinity has its largest number
// as first piece; an infinity has that twice and itself as the last one, which only the
// left operand's first piece meets.  (814.5 -> 816.5 us for 2048 tokens of 48 heads.)
__device__ inline void split_right(float first, float second, uint32_t& high, uint32_t& middle, uint32_t& low) {
  constexpr float kLargest = 0x1.fep127f;
  auto pack = [](float a, float b) {
    return pack_bf16(__builtin_amdgcn_fmed3f(a, -kLargest, kLargest), __builtin_amdgcn_fmed3f(b, -kLargest, kLargest));
  };
  high = pack(first, second);
  first -= __uint_as_float(high << 16);
  second -= __uint_as_float(high & 0xffff0000u);
  middle = pack(first, second);
  first -= __uint_as_float(middle << 16);
  second -= __uint_as_float(middle & 0xffff0000u);
  low = pack_bf16(first, second);
}
template <int STEPS>
struct OperandLds {
  uint4 part[STEPS][3][64];
  __device__ void put(int step, int lane, const Pieces& p) {
#pragma unroll
    for (int i = 0; i < 3; ++i) part[step][i][lane] = __builtin_bit_cast(uint4, p.part[i]);
  }
  // four elements of a lane: the first or second half of a step's
  __device__ void put_half(int step, int half, int lane, float4 v) {
    uint32_t words[3][2];
    split_right(v.x, v.y, words[0][0], words[1][0], words[2][0]);
    split_right(v.z, v.w, words[0][1], words[1][1], words[2][1]);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      reinterpret_cast<uint2*>(&part[step][i][lane])[half] = make_uint2(words[i][0], words[i][1]);
  }
  __device__ Pieces get(int step, int lane) const {
    Pieces p;
#pragma unroll
    for (int i = 0; i < 3; ++i) p.part[i] = as_bf16x8(part[step][i][lane]);
    return p;
  }
};
__device__ inline Pieces state_pieces(const floatx4& first, const floatx4& second) {
  uint32_t words[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const floatx4& from = i < 2 ? first : second;
    split_right(from[2 * (i % 2)], from[2 * (i % 2) + 1], words[0][i], words[1][i], words[2][i]);
  }
  Pieces p;
#pragma unroll
  for (int i = 0; i < 3; ++i) p.part[i] = as_bf16x8(make_uint4(words[i][0], words[i][1], words[i][2], words[i][3]));
  return p;
}
// Eight elements of any size.
__device__ inline Pieces pieces_of_any(float4 a, float4 b) {
  const floatx4 first = {a.x, a.y, a.z, a.w}, second = {b.x, b.y, b.z, b.w};
  return state_pieces(first, second);
}
__device__ inline float4 as_float4(const floatx4& v) { return make_float4(v[0], v[1], v[2], v[3]); }

// The records of a head as the sequential kernels walk them: one descriptor for all
// chunks, a lane offset that moves with the chunk and a uniform place in the record.
// Chunks have the same size in all records of one kind, so that the kinds share their
// lane offsets.
__device__ inline Record head_records(const ChunkedArgs& a, const float* records, int head, size_t elements) {
  return Record(records + static_cast<size_t>(head) * a.chunks * elements, a.chunks * elements);
}

// A chunk's operands on their way into the XCD's L2 two chunks ahead of the products: a piece
// of 8 KiB, 64 lines, is touched by one wave, and a head's workgroups share the pieces.  A
// compute unit has few lines on their way at a time, and those from memory stay longest.
// With two tiles a workgroup each wave off the chain touches one (2048 tokens, 48 heads,
// both kernels: 232 -> 217 us).  With one tile a chunk is too short to wait for a touched line
// before the operands behind it, as a wave's loads return in order, and a ninth wave does it
// (8192 tokens, 16 heads: 605 -> 470 us; as with two tiles 567); with two tiles that wave took
// registers that the others need (237).  Chunks of FP32 keys are long enough.
template <int TILES, bool BF16>
struct Ahead {
  static constexpr bool kOwnWave = TILES == 1 && BF16;
  static constexpr unsigned kBytes = 8192;
  static constexpr int kChunks = 2;  // ahead
  const void* base = nullptr;
  unsigned at = 0, step = 0, bytes = 0;
  float touched = 0.0f;
  int index;  // of the pieces not yet given away
  __device__ Ahead(const Slice& slice, int i) : index(slice.col0 / (kTile * TILES) * (2 * TILES) + i) {}
  // a head's records of `per_chunk` bytes a chunk, of which `wanted` from `offset` on
  __device__ void add(const void* records, size_t chunks, unsigned per_chunk, unsigned offset, unsigned wanted, int lane) {
    const int pieces = wanted / kBytes;
    if (index >= 0 && index < pieces) {
      base = records, step = per_chunk, bytes = static_cast<unsigned>(chunks * per_chunk);
      at = offset + index * kBytes + 128 * lane;
    }
    index -= pieces;
  }
  // a chunk's tokens of a head in [tokens, heads, 128]
  __device__ void add_tokens(const float* head, int tokens, unsigned row_bytes, int lane) {
    if (index >= 0 && index < 4) {
      const size_t all = static_cast<size_t>(tokens - 1) * row_bytes + kD * 4;
      base = head, step = kC * row_bytes, bytes = static_cast<unsigned>(all < 0xffffffffu ? all : 0xffffffffu);
      at = (16 * index + lane / 4) * row_bytes + 128 * (lane % 4);
    }
    index -= 4;
  }
  // chunks that do not exist lie beyond the descriptor or are the first again
  __device__ void touch(int chunk) {
    asm volatile("" ::"v"(touched));
    touched = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000),
        at + max(chunk, 0) * step, 0, 0));
  }
};
// The ninth wave: its pieces, chunk after chunk, and the barriers of the others.
template <class Made>
__device__ inline void touch_chunks(Made made, int first, int direction, int steps) {
  auto one = made(0), two = made(1);
  for (int i = 0; i < steps; ++i) {
    one.touch(first + i * direction);
    two.touch(first + i * direction);
    lds_barrier();
    lds_barrier();
  }
}

// Both sequential kernels are chains of products with a barrier between them; requests
// and stores stand between the multiplications, each request for a register right
// after the multiplication that read it, and none between a product and the barrier
// that publishes it.  The fences keep that order.

// Eight elements of a left operand as they come from memory: FP32 numbers that become three
// pieces, or bf16.
struct Eight {
  float4 first, second;
};
template <bool BF16>
using KeyEight = std::conditional_t<BF16, bf16x8, Eight>;
struct Nothing {};
__device__ inline Pieces as_left(const Eight& e) { return split_eight(e.first, e.second); }

// The products of one left operand while the next one is made and its right sides are
// read (step -1: they stay): a matrix instruction and a few vector instructions take turns.
template <int TILES, int STEPS, class Left, class Next>
__device__ inline void step(floatx4 (&acc)[TILES], const Left& left, Pieces (&right)[TILES], const Next& next,
                            Pieces& next_left, const OperandLds<STEPS>* from, int next_step, int lane) {
  constexpr bool kThree = std::is_same_v<Left, Pieces>, kSplit = std::is_same_v<Next, Eight>;
  keep_order();
  Pieces read[TILES];
#pragma unroll
  for (int c = 0; c < TILES; ++c) read[c] = next_step >= 0 ? from[c].get(next_step, lane) : right[c];
  keep_order();
  Eight numbers{};
  if constexpr (kSplit) numbers = next;
  Splitter split(numbers.first, numbers.second);
  // smallest products first
  constexpr int kProducts = kThree ? 6 : 3, kSlots = kProducts * TILES;
  constexpr int kLeft[6] = {2, 1, 1, 0, 0, 0}, kRight[6] = {0, 1, 0, 2, 1, 0};
#pragma unroll
  for (int i = 0; i < kProducts; ++i) {
#pragma unroll
    for (int c = 0; c < TILES; ++c) {
      if constexpr (kThree)
        acc[c] = mfma16(left.part[kLeft[i]], right[c].part[kRight[i]], acc[c]);
      else
        acc[c] = mfma16(left, right[c].part[2 - i], acc[c]);
      if constexpr (kSplit) {
        constexpr int kEach = (Splitter::kSteps + kSlots - 1) / kSlots;
#pragma unroll
        for (int s = 0; s < kEach; ++s)
          if ((i * TILES + c) * kEach + s < Splitter::kSteps) split((i * TILES + c) * kEach + s, true);
      }
      keep_order();
    }
  }
  if constexpr (kSplit) next_left = split.pieces();
#pragma unroll
  for (int c = 0; c < TILES; ++c) right[c] = read[c];
}
template <int TILES, int STEPS>
__device__ inline void read_right(Pieces (&right)[TILES], const OperandLds<STEPS>* from, int step, int lane) {
#pragma unroll
  for (int c = 0; c < TILES; ++c) right[c] = from[c].get(step, lane);
}

// The four steps of a product by keys or queries.  As bf16 they are multiplied from the
// registers that they arrive in and requested again for the next chunk right after; a copy of
// one that is still on its way would wait for it.  As FP32 each is split a step ahead.
template <int TILES, bool BF16>
struct KeySteps {
  KeyEight<BF16> eight[4];
  // the step before the first
  template <int STEPS>
  __device__ void enter(floatx4 (&acc)[TILES], Pieces& left, Pieces (&right)[TILES], const OperandLds<STEPS>* from,
                        int next_step, int lane) {
    if constexpr (BF16)
      step<TILES>(acc, left, right, Nothing(), left, from, next_step, lane);
    else
      step<TILES>(acc, left, right, eight[0], left, from, next_step, lane);
  }
  template <class Request>
  __device__ void entered(Request request) const {
    if constexpr (!BF16) request(0);
  }
  // step i < 3
  template <int STEPS, class Request>
  __device__ void go(int i, floatx4 (&acc)[TILES], Pieces& left, Pieces (&right)[TILES], const OperandLds<STEPS>* from,
                     int next_step, int lane, Request request) {
    if constexpr (BF16) {
      step<TILES>(acc, eight[i], right, Nothing(), left, from, next_step, lane);
      request(i);
    } else {
      step<TILES>(acc, left, right, eight[i + 1], left, from, next_step, lane);
      request(i + 1);
    }
  }
  // the last one, next to the splitting of the next product's left operand
  template <int STEPS, class Request>
  __device__ void finish(floatx4 (&acc)[TILES], Pieces& left, Pieces (&right)[TILES], const Eight& next,
                         const OperandLds<STEPS>* from, int next_step, int lane, Request request) {
    if constexpr (BF16) {
      step<TILES>(acc, eight[3], right, next, left, from, next_step, lane);
      request(3);
    } else {
      step<TILES>(acc, left, right, next, left, from, next_step, lane);
    }
  }
};

// Eight waves: the first four carry the chain, wave w rows 16 w .. + 15 of the 64-row
// products and rows 32 w .. + 31 of the state; the others do what the chain does not wait
// for, the same rows.  Two waves a SIMD cover each other's waits for LDS and barriers.
// With bf16 activations a chunk of two tiles is 1900 cycles of matrix instructions a SIMD,
// 3400 of vector instructions and 88 KiB of operands a compute unit, which at the 20 bytes a
// clock that one gets of a busy L2 are 4400: with 48 heads a chunk takes 7300, 5700 of them
// where few heads leave the memory idle.  2048 tokens of 48 heads: 117 and 101 us; with keys and
// queries of three pieces 147 and 138, with all operands kept as pieces (6 bytes an element
// instead of 4 and the splitting) 178 and 159, with the FP32 instruction 184 and 187.  The
// stores stay with the chain's waves: through LDS by the others they took 1 and 10 us more.
template <int TILES, bool BF16>
constexpr int kSequentialThreads = Ahead<TILES, BF16>::kOwnWave ? 576 : 512;

// S entering every chunk, Dl and O of every chunk.  60 matrix instructions a row of waves,
// chunk and tile, the 24 of O off the chain (84 and 36 with FP32 keys).  Operands are requested a chunk ahead.
template <int TILES, bool BF16>
__global__ void __launch_bounds__((kSequentialThreads<TILES, BF16>))
chunk_states_forward_kernel(ChunkedArgs a) {
  __shared__ OperandLds<4> state[TILES];
  __shared__ OperandLds<2> delta[TILES], left_delta[TILES];
  const Slice slice = slice_of_block<TILES>(a);
  const int lane = threadIdx.x % 64, quarter = lane / 16, n = lane % 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64 % 4);
  const bool chain = __builtin_amdgcn_readfirstlane(threadIdx.x) < 256;
  const int rows = 16 * wave + 4 * quarter;  // of the lane's part of Dl and O
  const int head = slice.head, key_head = head / (a.vh / a.kh);
  const Record gates = head_records(a, a.r.gates, head, kGateRows * kC);
  // the lane's places in the records of the chunk whose operands are requested next
  // four rows of a column -> four columns of a row: the lane's place in rows(Dl), rows(S)
  const int transposed_at = n / 4 * kPiece + (4 * quarter + n % 4) * 16 - 16 * lane;
  unsigned wide_at = 16 * lane, keys_at = 16 * lane, square_at = 16 * lane, gates_at = 4 * rows;
  constexpr unsigned kKeysBytes = BF16 ? KeyOperands::kChunkBytes : kWide * 4;
  const KeyOperands operands(a, key_head);
  const floatx4 none = {0.0f, 0.0f, 0.0f, 0.0f};
  Pieces left, right[TILES];  // the operands of the products that come next
  auto ahead_of = [&](int i) {
    Ahead<TILES, BF16> ahead(slice, i);
    const size_t of_head = static_cast<size_t>(head) * a.chunks;
    ahead.add(a.r.w_rows + of_head * kWide, a.chunks, kWide * 4, 0, kWide * 4, lane);
    ahead.add(a.r.u_columns + of_head * kWide, a.chunks, kWide * 4, 0, kWide * 4, lane);
    ahead.add(a.r.p_rows + of_head * kSquare, a.chunks, kSquare * 4, 0, kSquare * 4, lane);
    if constexpr (BF16) {
      ahead.add(operands.memory.base, a.chunks, kKeysBytes, KeyOperands::kRowsOfQ, 2 * kWide, lane);
      ahead.add(operands.memory.base, a.chunks, kKeysBytes, KeyOperands::kColumnsOfK, 2 * kWide, lane);
    }
    return ahead;
  };
  if constexpr (Ahead<TILES, BF16>::kOwnWave)
    if (__builtin_amdgcn_readfirstlane(threadIdx.x) >= 512) {
      touch_chunks(ahead_of, Ahead<TILES, BF16>::kChunks, 1, a.chunks);
      return;
    }
  if (chain) {
    __builtin_amdgcn_s_setprio(2);
    Eight w[4];
    KeySteps<TILES, BF16> k;  // step i: operand tile i % 2, tokens 32 (i / 2) ..
    float4 u[TILES], l_rows;
    float decay;
    const Record w_memory = head_records(a, a.r.w_rows, head, kWide),
                 k_memory = head_records(a, a.r.k_columns, key_head, kWide),
                 u_memory = head_records(a, a.r.u_columns, head, kWide),
                 dl_memory = head_records(a, a.r.dl_rows, head, kWide),
                 s0_memory = head_records(a, a.r.s0, head, kState);
    const unsigned u_at = piece_at<kC>(slice.col0 / 16, 4 * wave);
    auto request_w = [&](int s) {
      w[s] = {w_memory.get4(wide_at, piece_at<kD>(wave, 8 * s)), w_memory.get4(wide_at, piece_at<kD>(wave, 8 * s + 4))};
    };
    auto request_k = [&](int i) {
      const int block = 2 * wave + i % 2, s = i / 2;
      if constexpr (BF16)
        k.eight[i] = operands.get(keys_at, KeyOperands::kColumnsOfK + (2 * block + s) * 1024);
      else
        k.eight[i] = {k_memory.get4(keys_at, piece_at<kC>(block, 8 * s)),
                      k_memory.get4(keys_at, piece_at<kC>(block, 8 * s + 4))};
    };
    auto request_rest = [&]() {
#pragma unroll
      for (int c = 0; c < TILES; ++c) u[c] = u_memory.get4(wide_at, u_at + piece_at<kC>(c, 0));
      l_rows = gates.get4(gates_at, 4 * (BF16 ? kLK : kL) * kC);
      decay = gates.get(gates_at - 4 * rows, 4 * (kE * kC + kC - 1));
    };
    floatx4 acc[2][TILES];
#pragma unroll
    for (int c = 0; c < TILES; ++c) acc[0][c] = acc[1][c] = none;
    // in the loop's order, so that the waits in it need not cover another one
#pragma unroll
    for (int s = 0; s < 4; ++s) request_w(s), keep_order();
    request_rest();
    keep_order();
#pragma unroll
    for (int i = 0; i < 4; ++i) request_k(i), keep_order();
    left = as_left(w[0]);
    int chunk = 0;
    do {
      // past the end the last chunk's operands are requested again
      const unsigned delta_now = wide_at + transposed_at, state_now = 16 * lane + transposed_at + chunk * (kState * 4);
      const bool more = chunk + 1 < a.chunks;
      wide_at += more ? kWide * 4 : 0, keys_at += more ? kKeysBytes : 0, gates_at += more ? kGateRows * kC * 4 : 0;
#pragma unroll
      for (int c = 0; c < TILES; ++c) state[c].put(wave, lane, state_pieces(acc[0][c], acc[1][c]));
      keep_order();
      lds_barrier();
      floatx4 part[TILES];
      read_right<TILES>(right, state, 0, lane);
      request_w(0);  // split before the loop and at its end
      keep_order();
      // rows(S): 16 rows a store, four columns a lane
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
          s0_memory.put4(quad_transpose(as_float4(acc[t][c])), state_now,
                         piece_at<kD>(2 * wave + t, (slice.col0 + kTile * c) / 4));
        part[c] = none;
      }
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        step<TILES>(part, left, right, w[s + 1], left, state, s + 1, lane);
        request_w(s + 1);
      }
      k.enter(part, left, right, state, -1, lane);
      float4 dl[TILES];
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
        dl[c] = make_float4(u[c].x - part[c][0], u[c].y - part[c][1], u[c].z - part[c][2], u[c].w - part[c][3]);
        left_delta[c].put_half(wave / 2, wave % 2, lane,
                               make_float4(dl[c].x * l_rows.x, dl[c].y * l_rows.y, dl[c].z * l_rows.z, dl[c].w * l_rows.w));
        delta[c].put_half(wave / 2, wave % 2, lane, dl[c]);
        acc[0][c] *= decay;
        acc[1][c] *= decay;
      }
      keep_order();
      lds_barrier();
      read_right<TILES>(right, left_delta, 0, lane);
      request_rest();
      k.entered(request_k);
      keep_order();
#pragma unroll
      for (int c = 0; c < TILES; ++c)
        dl_memory.put4(quad_transpose(dl[c]), delta_now, piece_at<kD>(wave, (slice.col0 + kTile * c) / 4));
#pragma unroll
      for (int i = 0; i < 3; ++i) k.go(i, acc[i % 2], left, right, left_delta, i == 1 ? 1 : -1, lane, request_k);
      k.finish(acc[1], left, right, w[0], left_delta, -1, lane, request_k);
    } while (++chunk < a.chunks);
  } else {
    KeySteps<TILES, BF16> q;
    Eight p[2];
    float4 e_rows;
    const Record q_memory = head_records(a, a.r.q_rows, key_head, kWide),
                 p_memory = head_records(a, a.r.p_rows, head, kSquare);
    const unsigned core_at = (rows + n % 4) * (a.vh * kD * 4) + 4 * (slice.col0 + n / 4 * 4);
    auto request_q = [&](int s) {
      if constexpr (BF16)
        q.eight[s] = operands.get(keys_at, KeyOperands::kRowsOfQ + (4 * wave + s) * 1024);
      else
        q.eight[s] = {q_memory.get4(keys_at, piece_at<kD>(wave, 8 * s)),
                      q_memory.get4(keys_at, piece_at<kD>(wave, 8 * s + 4))};
    };
    auto request_p = [&](int s) {
      p[s] = {p_memory.get4(square_at, piece_at<kC>(wave, 8 * s)), p_memory.get4(square_at, piece_at<kC>(wave, 8 * s + 4))};
    };
    auto request_e = [&]() { e_rows = gates.get4(gates_at, 4 * (BF16 ? kEQ : kE) * kC); };
#pragma unroll
    for (int s = 0; s < 4; ++s) request_q(s), keep_order();
    request_e();
    keep_order();
#pragma unroll
    for (int s = 0; s < 2; ++s) request_p(s), keep_order();
    Ahead<TILES, BF16> ahead = ahead_of(wave);
    if constexpr (!BF16) left = as_left(q.eight[0]);
    int chunk = 0;
    do {
      const Tokens core = ChunkView(a, chunk, head).heads(a.core);
      const bool more = chunk + 1 < a.chunks;
      keys_at += more ? kKeysBytes : 0, square_at += more ? kSquare * 4 : 0, gates_at += more ? kGateRows * kC * 4 : 0;
      lds_barrier();
      floatx4 out[TILES];
      read_right<TILES>(right, state, 0, lane);
      q.entered(request_q);
#pragma unroll
      for (int c = 0; c < TILES; ++c) out[c] = none;
#pragma unroll
      for (int s = 0; s < 3; ++s) q.go(s, out, left, right, state, s + 1, lane, request_q);
      q.finish(out, left, right, p[0], state, -1, lane, request_q);
      if constexpr (!ahead.kOwnWave) ahead.touch(chunk + ahead.kChunks);
#pragma unroll
      for (int c = 0; c < TILES; ++c)
        out[c][0] *= e_rows.x, out[c][1] *= e_rows.y, out[c][2] *= e_rows.z, out[c][3] *= e_rows.w;
      keep_order();
      request_e();
      request_p(0);
      lds_barrier();
      read_right<TILES>(right, delta, 0, lane);
      step<TILES>(out, left, right, p[1], left, delta, 1, lane);
      request_p(1);
      q.enter(out, left, right, delta, -1, lane);
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
        // four tokens of a column -> four columns of a token
        const float4 o =
            quad_transpose(make_float4(round_if(out[c][0], a.round), round_if(out[c][1], a.round),
                                       round_if(out[c][2], a.round), round_if(out[c][3], a.round)));
        core.put4(o, core_at, 4 * kTile * c);
      }
    } while (++chunk < a.chunks);
  }
}

// The gradient of the state leaving every chunk and dDl of every chunk, chunks in
// reverse.  60 matrix instructions a row of waves, chunk and tile, the 24 with dO off the
// chain (84 and 36 with FP32 keys): the other waves leave P^T dO and (diag(E) Q^)^T dO of the next chunk in LDS.
template <int TILES, bool BF16>
__global__ void __launch_bounds__((kSequentialThreads<TILES, BF16>))
chunk_states_backward_kernel(ChunkedArgs a) {
  __shared__ OperandLds<4> state[TILES];
  __shared__ OperandLds<2> delta[TILES], grad[TILES], query_grad[TILES];
  // [P^T dO, two row tiles of Q^T dO]: a wave's accumulators
  __shared__ floatx4 handed[2][3][TILES][4][64];
  const Slice slice = slice_of_block<TILES>(a);
  const int lane = threadIdx.x % 64, quarter = lane / 16, n = lane % 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64 % 4);
  const bool chain = __builtin_amdgcn_readfirstlane(threadIdx.x) < 256;
  const int rows = 16 * wave + 4 * quarter;
  const int head = slice.head, key_head = head / (a.vh / a.kh);
  const Record gates = head_records(a, a.r.gates, head, kGateRows * kC);
  const unsigned last = a.chunks - 1;
  constexpr unsigned kKeysBytes = BF16 ? KeyOperands::kChunkBytes : kWide * 4;
  unsigned wide_at = 16 * lane + last * (kWide * 4), keys_at = 16 * lane + last * kKeysBytes,
           square_at = 16 * lane + last * (kSquare * 4), gates_at = 4 * rows + last * (kGateRows * kC * 4);
  const KeyOperands operands(a, key_head);
  const floatx4 none = {0.0f, 0.0f, 0.0f, 0.0f};
  Pieces left, right[TILES];  // the operands of the products that come next
  auto ahead_of = [&](int i) {
    Ahead<TILES, BF16> ahead(slice, i);
    const size_t of_head = static_cast<size_t>(head) * a.chunks;
    ahead.add(a.r.w_columns + of_head * kWide, a.chunks, kWide * 4, 0, kWide * 4, lane);
    ahead.add_tokens(a.dcore + head * kD, a.length, a.vh * kD * 4, lane);
    ahead.add(a.r.p_columns + of_head * kSquare, a.chunks, kSquare * 4, 0, kSquare * 4, lane);
    if constexpr (BF16) {
      ahead.add(operands.memory.base, a.chunks, kKeysBytes, KeyOperands::kRowsOfK, 2 * kWide, lane);
      ahead.add(operands.memory.base, a.chunks, kKeysBytes, KeyOperands::kColumnsOfQ, 2 * kWide, lane);
    }
    return ahead;
  };
  if constexpr (Ahead<TILES, BF16>::kOwnWave)
    if (__builtin_amdgcn_readfirstlane(threadIdx.x) >= 512) {
      touch_chunks(ahead_of, static_cast<int>(last) + 1 - Ahead<TILES, BF16>::kChunks, -1, a.chunks + 1);
      return;
    }
  if (chain) {
    __builtin_amdgcn_s_setprio(2);
    KeySteps<TILES, BF16> k;
    Eight w[2][2];
    float4 k_scale;
    float decay;
    const Record k_memory = head_records(a, a.r.k_rows, key_head, kWide),
                 w_memory = head_records(a, a.r.w_columns, head, kWide),
                 ddl_rows = head_records(a, a.r.ddl_rows, head, kWide), ds1_memory = head_records(a, a.r.ds1, head, kState);
    const int transposed_at = n / 4 * kPiece + (4 * quarter + n % 4) * 16 - 16 * lane;  // as above
    auto request_k = [&](int s) {
      if constexpr (BF16)
        k.eight[s] = operands.get(keys_at, KeyOperands::kRowsOfK + (4 * wave + s) * 1024);
      else
        k.eight[s] = {k_memory.get4(keys_at, piece_at<kD>(wave, 8 * s)),
                      k_memory.get4(keys_at, piece_at<kD>(wave, 8 * s + 4))};
    };
    auto request_w = [&](int t, int s) {
      w[t][s] = {w_memory.get4(wide_at, piece_at<kC>(2 * wave + t, 8 * s)),
                 w_memory.get4(wide_at, piece_at<kC>(2 * wave + t, 8 * s + 4))};
    };
    auto request_gates = [&]() {
      k_scale = gates.get4(gates_at, 4 * (BF16 ? kLK : kL) * kC);
      decay = gates.get(gates_at - 4 * rows, 4 * (kE * kC + kC - 1));
    };
    floatx4 acc[2][TILES];
#pragma unroll
    for (int c = 0; c < TILES; ++c) acc[0][c] = acc[1][c] = none;
    // in the loop's order, so that the waits in it need not cover another one
#pragma unroll
    for (int s = 0; s < 4; ++s) request_k(s), keep_order();
    request_gates();
    keep_order();
#pragma unroll
    for (int s = 0; s < 4; ++s) request_w(s % 2, s / 2), keep_order();
    if constexpr (!BF16) left = as_left(k.eight[0]);
    lds_barrier();  // the first chunk's dO is in LDS,
    lds_barrier();  // and what the other waves hand over
    int chunk = a.chunks - 1;
    do {
      // before the first the first chunk's operands are requested again
      const unsigned wide_now = wide_at, state_now = 16 * lane + transposed_at + chunk * (kState * 4);
      const bool more = chunk > 0;
      wide_at -= more ? kWide * 4 : 0, keys_at -= more ? kKeysBytes : 0, gates_at -= more ? kGateRows * kC * 4 : 0;
#pragma unroll
      for (int c = 0; c < TILES; ++c) state[c].put(wave, lane, state_pieces(acc[0][c], acc[1][c]));
      keep_order();
      lds_barrier();
      floatx4 part[TILES];
      read_right<TILES>(right, state, 0, lane);
      k.entered(request_k);
      keep_order();
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
          ds1_memory.put4(quad_transpose(as_float4(acc[t][c])), state_now,
                          piece_at<kD>(2 * wave + t, (slice.col0 + kTile * c) / 4));
        part[c] = none;
      }
#pragma unroll
      for (int s = 0; s < 3; ++s) k.go(s, part, left, right, state, s + 1, lane, request_k);
      k.finish(part, left, right, w[0][0], state, -1, lane, request_k);
      float4 dd[TILES];
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
        const floatx4 from_out = handed[chunk % 2][0][c][wave][lane];
        dd[c] = make_float4(from_out[0] + k_scale.x * part[c][0], from_out[1] + k_scale.y * part[c][1],
                            from_out[2] + k_scale.z * part[c][2], from_out[3] + k_scale.w * part[c][3]);
        delta[c].put_half(wave / 2, wave % 2, lane, scaled(dd[c], -1.0f));
      }
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int c = 0; c < TILES; ++c) {
          const floatx4 queries = handed[chunk % 2][1 + t][c][wave][lane];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[t][c][e] = fmaf(acc[t][c][e], decay, queries[e]);
        }
      keep_order();
      lds_barrier();
      read_right<TILES>(right, delta, 0, lane);
      request_gates();
      request_w(0, 0);
      keep_order();
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
        ddl_rows.put4(quad_transpose(dd[c]), wide_now + transposed_at,
                      piece_at<kD>(wave, (slice.col0 + kTile * c) / 4));
      }
      // w[t][s] in the order s, t
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int t = (i + 1) % 2, s = (i + 1) / 2;
        step<TILES>(acc[i % 2], left, right, w[t][s], left, delta, i == 1 ? 1 : -1, lane);
        request_w(t, s);
      }
      k.enter(acc[1], left, right, delta, -1, lane);
    } while (--chunk >= 0);
  } else {
    Eight p[2];
    KeySteps<TILES, BF16> q;  // step i: operand tile i % 2, tokens 32 (i / 2) ..
    float4 out[TILES], q_scale;
    const Record p_memory = head_records(a, a.r.p_columns, head, kSquare),
                 q_memory = head_records(a, a.r.q_columns, key_head, kWide);
    const unsigned out_at = (rows + n % 4) * (a.vh * kD * 4) + 4 * (slice.col0 + n / 4 * 4);
    auto request_p = [&](int s) {
      p[s] = {p_memory.get4(square_at, piece_at<kC>(wave, 8 * s)), p_memory.get4(square_at, piece_at<kC>(wave, 8 * s + 4))};
    };
    auto request_q = [&](int i) {
      const int block = 2 * wave + i % 2, s = i / 2;
      if constexpr (BF16)
        q.eight[i] = operands.get(keys_at, KeyOperands::kColumnsOfQ + (2 * block + s) * 1024);
      else
        q.eight[i] = {q_memory.get4(keys_at, piece_at<kC>(block, 8 * s)),
                      q_memory.get4(keys_at, piece_at<kC>(block, 8 * s + 4))};
    };
    auto request_out = [&](int chunk) {
      const Tokens d_out = ChunkView(a, max(chunk, 0), head).heads(a.dcore);
#pragma unroll
      for (int c = 0; c < TILES; ++c) out[c] = d_out.get4(out_at, 4 * kTile * c);
      q_scale = gates.get4(gates_at, 4 * (BF16 ? kEQ : kE) * kC);
    };
    request_out(last);
    keep_order();
#pragma unroll
    for (int s = 0; s < 2; ++s) request_p(s), keep_order();
#pragma unroll
    for (int i = 0; i < 4; ++i) request_q(i), keep_order();
    Ahead<TILES, BF16> ahead = ahead_of(wave);
    left = as_left(p[0]);
    // a chunk ahead of the chain: what is handed over lies in LDS before the chain's
    // chunk begins
    int chunk = a.chunks - 1;
    do {
      const bool more = chunk > 0;
      keys_at -= more ? kKeysBytes : 0, square_at -= more ? kSquare * 4 : 0, gates_at -= more ? kGateRows * kC * 4 : 0;
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
        const float4 o = quad_transpose(out[c]);  // four columns of a token -> four tokens of a column
        grad[c].put_half(wave / 2, wave % 2, lane, o);
        query_grad[c].put_half(wave / 2, wave % 2, lane,
                               make_float4(o.x * q_scale.x, o.y * q_scale.y, o.z * q_scale.z, o.w * q_scale.w));
      }
      keep_order();
      lds_barrier();
      floatx4 from_out[TILES], queries[2][TILES];
      read_right<TILES>(right, grad, 0, lane);
      request_out(chunk - 1);
      request_p(0);
#pragma unroll
      for (int c = 0; c < TILES; ++c) from_out[c] = queries[0][c] = queries[1][c] = none;
      step<TILES>(from_out, left, right, p[1], left, grad, 1, lane);
      request_p(1);
      q.enter(from_out, left, right, query_grad, 0, lane);
      q.entered(request_q);
#pragma unroll
      for (int i = 0; i < 3; ++i) q.go(i, queries[i % 2], left, right, query_grad, i == 1 ? 1 : -1, lane, request_q);
      q.finish(queries[1], left, right, p[0], query_grad, -1, lane, request_q);
      if constexpr (!ahead.kOwnWave) ahead.touch(chunk - ahead.kChunks);
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
        handed[chunk & 1][0][c][wave][lane] = from_out[c];
        handed[chunk & 1][1][c][wave][lane] = queries[0][c];
        handed[chunk & 1][2][c][wave][lane] = queries[1][c];
      }
      keep_order();
      lds_barrier();
    } while (--chunk >= 0);
    lds_barrier();  // the chain's last chunk
    lds_barrier();
  }
}

// ---------------------------------------------------------------------------
// The gradients of one chunk.  Wave w owns columns 32w..32w+31 of the [64, 128]
// matrices (two 32-row tiles) and one 32 x 32 tile of the [64, 64] matrices, of which
// only those on and below the diagonal are needed.
//   1. contractions over value channels, 32 of them at a time, dDl, dO, Dl and V in LDS
//      and the states straight from memory (each element is used by one wave):
//        dW = -dDl S^T        dq^ = diag(E) dO S^T        dk^ = diag(L) Dl dS'^T
//        dP = lower(dO Dl^T)  dT = dDl (diag(beta) V)^T   and <dS', S>
//   2. dT += dW (diag(beta E) K^)^T;  dA = -strict_lower(T^T dT T^T);  R = diag(beta) dA D
//   3. dq^ += Pd K^ with Pd = dP D;  dk^ += (R + R^T) K^ + Pd^T Q^ + diag(beta E) T^T dW;
//      dv = diag(beta) T^T dDl;  dq and dk back through the normalisations
//   4. d log-decay and d beta from row and column sums of the above, through the gates
//      to da, db and the contribution to d A_log
// 78 KiB of LDS and 250 registers, none of them spilled: two workgroups a compute unit.  2048
// tokens of 48 heads 267 -> 226 us when 45 registers no longer went to scratch (140 MB there
// and back): the contributions of U before those of W, one product's accumulator at a time,
// and a sum whose factors the compiler kept for its end.  dDl and T are read here in the one
// order they are kept in and exchanged between lanes (230 us; the kernels that write them 137
// -> 129 and 106 -> 103).
// BF16: the products with rows of K and Q take three pieces and one (KeyOperands), their
// fractions go with the other factor or, in sums over a row's channels, with the sum: 232 ->
// 220 us, and the preparation, which no longer writes these rows as FP32, 73 -> 64.  What
// multiplies them may be as large as FP32 holds (split_right; 3 us).  The other products stay
// with the FP32 instruction: those with the states on pieces made by every wave took as long,
// the vector instructions for them being as many as the matrix instructions saved.
constexpr int kSlab = 32;
constexpr unsigned kSlabBytes = kC * kSlab * 4;
struct GradientSmem {
  union {
    unsigned char slab[2][4][kSlabBytes];  // two stages of rows(M) of dDl, dO, Dl, V, 32 columns each
    struct {
      float dw[kC][kWidePad], pd[kC][kSquarePad], x[kC][kSquarePad];
    };
  };
  float parts[6][kC][4];     // row sums of the waves' columns, see RowSum
  float row_n[kC][2], col_n[kC][2], row_p[kC][2], col_p[kC][2];  // by tile
  float gate[kGateRows][kC], dots[2][kC];
  float dot[4];
};
enum RowSum { kSumQ, kSumK, kSumW, kSumV, kDotQ, kDotK };

template <bool BF16>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(2, 2)))
chunk_gradients_kernel(ChunkedArgs a) {
  __shared__ __attribute__((aligned(16))) GradientSmem sm;
  const ChunkView v(a, blockIdx.x, blockIdx.y);
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int h = lane / 32, n = lane % 32, col = 32 * wave + n;
  const int ti_own = wave / 2, tj_own = wave % 2;   // the [64, 64] tile
  const bool lower = ti_own >= tj_own;
  for (int i = tid; i < kGateRows * kC; i += 256) {
    const int row = i / kC;
    if (!BF16 || row < kEQ) {
      sm.gate[row][i % kC] = v.gates[i];
    } else {  // what the bf16 rows of Q and K lack
      const float scale = v.gates[(row == kEQ ? kQScale : kKScale) * kC + i % kC];
      sm.gate[row][i % kC] = scale == 0.0f ? 0.0f : fraction_of(scale);
    }
  }
  if (tid < kC) {
    sm.row_n[tid][0] = sm.row_n[tid][1] = sm.col_n[tid][0] = sm.col_n[tid][1] = 0.0f;
    sm.row_p[tid][0] = sm.row_p[tid][1] = sm.col_p[tid][0] = sm.col_p[tid][1] = 0.0f;
  }
  floatx16 dw[2], dq[2], dk[2], dp = zero_tile(), dt = zero_tile();
#pragma unroll
  for (int ti = 0; ti < 2; ++ti) dw[ti] = dq[ti] = dk[ti] = zero_tile();
  float dot = 0.0f;
  const int tile_col = 32 * tj_own + n;
  const unsigned square_at = lane_piece<kC>(h, n);
  // the lane's places in columns(M) of [64, 64] and [64, 128] matrices (four rows of one
  // column, as in an accumulator), and a token's in the activations
  const unsigned tile_at = square_at + piece_at<kC>(2 * tj_own, 8 * ti_own);
  const unsigned column_at = square_at + piece_at<kC>(2 * wave, 0);
  // Rows of a matrix that is kept in columns, and the other way round: four columns of one of
  // four rows a lane, exchanged between neighbouring lanes when they have arrived.
  const unsigned quad_at = n / 4 * kPiece + (4 * h + n % 4) * 16;
  // rows of tokens are read and written four columns of one token a lane: token n % 4 of
  // the four of a register quad, columns 4 (n / 4) .. + 3 of the wave's
  const unsigned token_row = 4 * h + n % 4, token_column = 4 * (32 * wave + n / 4 * 4);
  const unsigned token_at = token_row * v.row_bytes + token_column;
  // Four tokens of a column or columns of a token of K or Q, as they are kept.  bf16: of
  // quad s of a row of operand blocks, a lane's place and a uniform one.
  using KeyQuad = std::conditional_t<BF16, uint2, float4>;
  auto numbers = [](KeyQuad quad) {
    if constexpr (BF16) {
      asm volatile("" : "+v"(quad.x), "+v"(quad.y));  // unpacked at each use: the numbers take twice the registers
      return unpacked(quad);
    } else {
      return quad;
    }
  };
  const KeyOperands operands(a, v.key_head());
  const unsigned key_lane = blockIdx.x * KeyOperands::kChunkBytes + (16 * h + n % 16) * 16;
  auto key_quad = [&](unsigned lane_at, unsigned first, int quad) {
    const unsigned place = first + quad / 4 * 1024 + quad % 2 * 512 + quad % 4 / 2 * 8;
    return __builtin_bit_cast(uint2, operands.memory.get2(lane_at, place));
  };
  auto as_operand = [](uint2 first, uint2 second) { return as_bf16x8(make_uint4(first.x, first.y, second.x, second.y)); };
  auto mma_exact = [](floatx16 acc, const Pieces& left, bf16x8 right) {
#pragma unroll
    for (int part = 2; part >= 0; --part) acc = mfma32(left.part[part], right, acc);
    return acc;
  };
  // row tile t of a per-row quantity in LDS, rows of register quad j
  auto rows4 = [&](const float* rows, int t, int j) { return load4(rows + 32 * t + 8 * j + 4 * h); };
  auto element = [](const float4& four, int i) {
    return i % 4 == 0 ? four.x : i % 4 == 1 ? four.y : i % 4 == 2 ? four.z : four.w;
  };
  {
    const Record s0_memory = v.state(a.r.s0), s1_memory = v.state(a.r.ds1);
    const unsigned state_at = piece_at<kD>(2 * wave, 0) + lane_piece<kD>(h, n);
    // fills of a stage: wave w brings row block w of the four matrices, in two parts
    const int32x4 sources[4] = {
        make_rsrc(a.r.ddl_rows + v.rec * kWide, kWide * 4), v.heads(a.dcore).words(),
        make_rsrc(a.r.dl_rows + v.rec * kWide, kWide * 4), v.v().words()};
    const unsigned record_at = piece_at<kD>(wave, 0) + 16 * lane;
    const unsigned fill_at[4] = {record_at, (16 * wave + lane % 16) * v.out_bytes + lane / 16 * 16, record_at,
                                 (16 * wave + lane % 16) * v.post_bytes + lane / 16 * 16};
    // (bf16 rows of V in one: eight columns a piece)
    auto fill = [&](int slab) {
      if constexpr (BF16)
        lds_fill<16>(sources[3], sm.slab[slab % 2][3] + 1024 * wave, fill_at[3] + slab * (kSlab * 2));
#pragma unroll
      for (int m = 0; m < (BF16 ? 3 : 4); ++m)
#pragma unroll
        for (int part = 0; part < 2; ++part) {
          const int quad = kSlab / 4 * slab + 4 * part;
          lds_fill<16>(sources[m], sm.slab[slab % 2][m] + piece_at<kSlab>(wave, 4 * part),
                       fill_at[m] + quad * (m % 2 == 0 ? kPiece : 16));
        }
    };
    // a lane's place in a matrix of a stage: row n of row tile 0, quads 2 g + h
    const unsigned tile_row_at = piece_at<kSlab>(n / 16, h) + n % 16 * 16;
    float4 s0[4], s1[4];
    auto request = [&](int slab, int g) {
      s0[g] = s0_memory.get4(state_at, piece_at<kD>(0, kSlab / 4 * slab + 2 * g));
      s1[g] = s1_memory.get4(state_at, piece_at<kD>(0, kSlab / 4 * slab + 2 * g));
    };
#pragma unroll
    for (int g = 0; g < 4; ++g) request(0, g);
    keep_order();
    fill(0);
    float fv = 0.0f;
#pragma unroll
    for (int slab = 0; slab < kD / kSlab; ++slab) {
      // The stage and the states' registers have arrived; naming the registers keeps the
      // compiler from waiting for them below, behind requests it does not count.
      asm volatile("s_waitcnt vmcnt(0)"
                   : "+v"(s0[0].x), "+v"(s0[1].x), "+v"(s0[2].x), "+v"(s0[3].x), "+v"(s1[0].x), "+v"(s1[1].x),
                     "+v"(s1[2].x), "+v"(s1[3].x)
                   :
                   : "memory");
      __syncthreads();
      if (slab == 0) fv = sm.gate[kBeta][32 * tj_own + n];
      if (slab + 1 < kD / kSlab) fill(slab + 1);
      keep_order();
      const unsigned char(&stage)[4][kSlabBytes] = sm.slab[slab % 2];
      auto operand = [&](int m, int ti, int g) {
        return *reinterpret_cast<const float4*>(stage[m] + tile_row_at + piece_at<kSlab>(2 * ti, 2 * g));
      };
      auto value_operand = [&](int ti, int g) {
        if constexpr (!BF16) return operand(3, ti, g);
        const int place = 1024 * (2 * ti + n / 16) + 256 * g + n % 16 * 16 + 8 * h;
        return unpacked(*reinterpret_cast<const uint2*>(stage[3] + place));
      };
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        dot += (s0[g].x * s1[g].x + s0[g].y * s1[g].y) + (s0[g].z * s1[g].z + s0[g].w * s1[g].w);
        asm volatile("" : "+v"(dot));  // here, not where it is needed: its factors' registers are
#pragma unroll
        for (int ti = 0; ti < 2; ++ti) {
          dw[ti] = mma(dw[ti], operand(0, ti, g), s0[g]);
          dq[ti] = mma(dq[ti], operand(1, ti, g), s0[g]);
          dk[ti] = mma(dk[ti], operand(2, ti, g), s1[g]);
        }
        keep_order();
        if (slab + 1 < kD / kSlab) request(slab + 1, g);
        keep_order();
        if (lower) {
          dp = mma(dp, operand(1, ti_own, g), operand(2, tj_own, g));
          dt = mma(dt, operand(0, ti_own, g), scaled(value_operand(tj_own, g), fv));
        }
        keep_order();
      }
    }
    dot = wave_sum(dot);
    if (lane == 0) sm.dot[wave] = dot;
  }
  lds_barrier();  // the slabs make room for dW, Pd and X
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int i = 0; i < 16; ++i) sm.dw[32 * ti + tile_row(i, h)][col] = -dw[ti][i];
  keep_order();
  // Everything the [64, 64] part reads is requested a step before it is used.
  // (Descriptors of what is read or written are made where that is: all at once they do not
  // fit in the scalar registers and go to scratch.)
  float4 p_tile[4];
  KeyQuad k_own[kD / 8];
  if (lower) {
    const Record p_memory = v.square(a.r.p_columns);
#pragma unroll
    for (int j = 0; j < 4; ++j) p_tile[j] = p_memory.get4(tile_at, piece_at<kC>(0, 2 * j));
    keep_order();
    if constexpr (BF16) {
#pragma unroll
      for (int s = 0; s < kD / 8; ++s)
        k_own[s] = key_quad(key_lane + n / 16 * 4096, KeyOperands::kRowsOfK + 2 * tj_own * 4096, s);
    } else {
      const Record k_rows = v.key(a.r.k_rows);
      const unsigned k_at = piece_at<kD>(2 * tj_own, 0) + lane_piece<kD>(h, n);
#pragma unroll
      for (int s = 0; s < kD / 8; ++s) k_own[s] = k_rows.get4(k_at, piece_at<kD>(0, 2 * s));
    }
  }
  keep_order();
  // row and column sums of a tile held in an accumulator, for its rows and columns
  auto tile_sums = [&](const float (&values)[16], float (&row_sums)[kC][2], float (&col_sums)[kC][2],
                       bool weighted) {
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      sum += weighted ? element(rows4(sm.gate[kBeta], ti_own, i / 4), i) * values[i] : values[i];
    sum += __shfl_xor(sum, 32, 64);
    if (h == 0) col_sums[tile_col][ti_own] = sum;
    const float row_sum = half_sums(values);
    if (n < 16) row_sums[32 * ti_own + tile_row(n, h)][tj_own] = row_sum;
  };
  float decay[16];  // D of the tile
  if (lower) {
    float products[16];
    const float g_col = sm.gate[kG][tile_col];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 32 * ti_own + tile_row(i, h);
      const bool in = row >= tile_col;
      decay[i] = in ? expf(element(rows4(sm.gate[kG], ti_own, i / 4), i) - g_col) : 0.0f;
      sm.pd[row][tile_col] = in ? dp[i] * decay[i] : 0.0f;
      products[i] = in ? dp[i] * element(p_tile[i / 4], i) : 0.0f;
    }
    tile_sums(products, sm.row_p, sm.col_p, false);
  }
  float4 t_own[8];  // T^T for rows of the tile, then T for its columns
  keep_order();
  if (lower) {
    const Record t_columns = v.square(a.r.t_columns);
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (s >= 4 * ti_own) t_own[s] = t_columns.get4(square_at, piece_at<kC>(2 * ti_own, 2 * s));
  }
  keep_order();
  lds_barrier();
  if (lower) {
    const float fk = sm.gate[kBeta][tile_col] * sm.gate[kE][tile_col];
    if constexpr (BF16) {
      floatx16 by_k = zero_tile();
#pragma unroll
      for (int s = 0; s < kD / 8; s += 2) {
        const float* row = &sm.dw[32 * ti_own + n][8 * s + 4 * h];
        by_k = mma_exact(by_k, pieces_of_any(load4(row), load4(row + 8)), as_operand(k_own[s], k_own[s + 1]));
      }
      const float factor = fk * sm.gate[kLK][tile_col];
#pragma unroll
      for (int i = 0; i < 16; ++i) dt[i] = fmaf(factor, by_k[i], dt[i]);
    } else {
#pragma unroll
      for (int s = 0; s < kD / 8; ++s)
        dt = mma(dt, load4(&sm.dw[32 * ti_own + n][8 * s + 4 * h]), scaled(k_own[s], fk));
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) sm.x[32 * ti_own + tile_row(i, h)][tile_col] = dt[i];
  }
  keep_order();
  // columns of K^ and Q^, both as operands and in the accumulators' rows
  KeyQuad kc[8], qc[8];
  float4 kkd_tile[4];
  const unsigned key_columns = key_lane + n / 16 * 2048;
  if constexpr (BF16) {
#pragma unroll
    for (int s = 0; s < 8; ++s) kc[s] = key_quad(key_columns, KeyOperands::kColumnsOfK + 2 * wave * 2048, s);
  } else {
    const Record k_memory = v.key(a.r.k_columns);
#pragma unroll
    for (int s = 0; s < 8; ++s) kc[s] = k_memory.get4(column_at, piece_at<kC>(0, 2 * s));
  }
  keep_order();
  lds_barrier();
  floatx16 z = zero_tile();
  if (lower) {
    // T^T dT: rows k < i of T's column i are zero, tile (0, 1) of dT is not needed
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (s >= 4 * ti_own) z = mma(z, t_own[s], gather4(&sm.x[8 * s + 4 * h][tile_col], kSquarePad));
    keep_order();
    const Record t_columns = v.square(a.r.t_columns), kkd = v.square(a.r.kkd);
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (s < 4 * (tj_own + 1)) t_own[s] = t_columns.get4(quad_at, piece_at<kC>(s / 2, 8 * tj_own) + 128 * (s % 2));
#pragma unroll
    for (int j = 0; j < 4; ++j) kkd_tile[j] = kkd.get4(tile_at, piece_at<kC>(0, 2 * j));
  }
  keep_order();
  if constexpr (BF16) {
#pragma unroll
    for (int s = 0; s < 8; ++s) qc[s] = key_quad(key_columns, KeyOperands::kColumnsOfQ + 2 * wave * 2048, s);
  } else {
    const Record q_memory = v.key(a.r.q_columns);
#pragma unroll
    for (int s = 0; s < 8; ++s) qc[s] = q_memory.get4(column_at, piece_at<kC>(0, 2 * s));
  }
  keep_order();
  lds_barrier();
  if (lower) {
#pragma unroll
    for (int i = 0; i < 16; ++i) sm.x[32 * ti_own + tile_row(i, h)][tile_col] = z[i];
  }
  lds_barrier();
  floatx16 da = zero_tile();
  if (lower) {
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (s < 4 * (tj_own + 1)) da = mma(da, load4(&sm.x[32 * ti_own + n][8 * s + 4 * h]), quad_transpose(t_own[s]));
  }
  lds_barrier();
  if (lower) {
    // R + R^T, and the sums of N = dA (k^ . k^) D
    float products[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 32 * ti_own + tile_row(i, h);
      const float value = row > tile_col ? -da[i] : 0.0f;
      products[i] = value * element(kkd_tile[i / 4], i);
      const float r = value * element(rows4(sm.gate[kBeta], ti_own, i / 4), i) * decay[i];
      if (row >= tile_col) sm.x[row][tile_col] = sm.x[tile_col][row] = r;
    }
    tile_sums(products, sm.row_n, sm.col_n, true);
  }
  keep_order();
  // T^T for both row tiles (the columns of T of the second start at row 32), dDl's columns
  float4 t_first[8], t_second[4], dd[8];
  const Record t_columns = v.square(a.r.t_columns), ddl = v.wide(a.r.ddl_rows);
  const Tokens v_memory = v.v(), dv = v.dv();
#pragma unroll
  for (int s = 0; s < 8; ++s) t_first[s] = t_columns.get4(square_at, piece_at<kC>(0, 2 * s));
#pragma unroll
  for (int s = 0; s < 8; ++s) dd[s] = ddl.get4(quad_at, piece_at<kD>(s / 2, 8 * wave) + 128 * (s % 2));
  keep_order();
  // over the columns of products with rows of V, K or Q, which with bf16 lack their fraction
  auto row_sums = [&](RowSum which, int ti, const float (&values)[16]) {
    const float sum = half_sums(values);
    const int row = 32 * ti + tile_row(n % 16, h);
    const bool query = which == kSumQ || which == kDotQ;
    const float factor = !BF16 || which == kSumV ? 1.0f : sm.gate[query ? kEQ : kLK][row];
    if (n < 16) sm.parts[which][row][wave] = sum * factor;
  };
#pragma unroll
  for (int ti = 0; ti < 2; ++ti) {
    float products[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      dq[ti][i] *= element(rows4(sm.gate[kE], ti, i / 4), i);
      products[i] = dq[ti][i] * element(numbers(qc[4 * ti + i / 4]), i);
    }
    row_sums(kSumQ, ti, products);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      dk[ti][i] *= element(rows4(sm.gate[kL], ti, i / 4), i);
      products[i] = dk[ti][i] * element(numbers(kc[4 * ti + i / 4]), i);
    }
    row_sums(kSumK, ti, products);
  }
  keep_order();
  lds_barrier();
#pragma unroll
  for (int s = 0; s < 8; ++s) dd[s] = quad_transpose(dd[s]);
#pragma unroll
  for (int ti = 0; ti < 2; ++ti) {
    const int m = 32 * ti + n;
    auto t_col = [&](int s) { return ti == 0 ? t_first[s] : t_second[s - 4]; };
    float products[16];
    float4 values[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned uniform = (32 * ti + 8 * j) * v.post_bytes;
      if constexpr (BF16) {  // half of a row of gradients, unpacked where it is used
        const float2 bits = v_memory.get2(token_at / 2, uniform);
        values[j].x = bits.x, values[j].y = bits.y;
      } else {
        values[j] = v_memory.get4(token_at, uniform);
      }
    }
    keep_order();
    {
      floatx16 tu = zero_tile();
#pragma unroll
      for (int s = 4 * ti; s < 8; ++s) tu = mma(tu, t_col(s), dd[s]);
      keep_order();
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (BF16) values[j] = unpacked(make_uint2(__float_as_uint(values[j].x), __float_as_uint(values[j].y)));
        const float4 value = quad_transpose(values[j]), beta = rows4(sm.gate[kBeta], ti, j);
        products[4 * j] = tu[4 * j] * value.x, products[4 * j + 1] = tu[4 * j + 1] * value.y;
        products[4 * j + 2] = tu[4 * j + 2] * value.z, products[4 * j + 3] = tu[4 * j + 3] * value.w;
        dv.put4(quad_transpose(make_float4(beta.x * tu[4 * j], beta.y * tu[4 * j + 1], beta.z * tu[4 * j + 2],
                                           beta.w * tu[4 * j + 3])),
                token_at, (32 * ti + 8 * j) * v.row_bytes);
      }
      row_sums(kSumV, ti, products);
    }
    keep_order();
    {
      floatx16 tw = zero_tile();
#pragma unroll
      for (int s = 4 * ti; s < 8; ++s) tw = mma(tw, t_col(s), gather4(&sm.dw[8 * s + 4 * h][col], kWidePad));
      keep_order();
      if (ti == 0) {
#pragma unroll
        for (int s = 4; s < 8; ++s) t_second[s - 4] = t_columns.get4(square_at, piece_at<kC>(2, 2 * s));
      }
      keep_order();
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float e = element(rows4(sm.gate[kE], ti, i / 4), i);
        products[i] = tw[i] * element(numbers(kc[4 * ti + i / 4]), i) * e;
        dk[ti][i] += element(rows4(sm.gate[kBeta], ti, i / 4), i) * e * tw[i];
      }
      row_sums(kSumW, ti, products);
    }
    keep_order();
    if constexpr (BF16) {
#pragma unroll
      for (int s = 0; s < 8; s += 2) {
        const int k = 8 * s + 4 * h;  // .. + 3 and eight further
        const float4 k0 = load4(&sm.gate[kLK][k]), k1 = load4(&sm.gate[kLK][k + 8]);
        const bf16x8 key = as_operand(kc[s], kc[s + 1]);
        const float *pd = &sm.pd[m][k], *x = &sm.x[m][k];
        if (s < 4 * (ti + 1))
          dq[ti] = mma_exact(dq[ti], pieces_of_any(product(load4(pd), k0), product(load4(pd + 8), k1)), key);
        dk[ti] = mma_exact(dk[ti], pieces_of_any(product(load4(x), k0), product(load4(x + 8), k1)), key);
        if (s >= 4 * ti) {
          const float4 q0 = load4(&sm.gate[kEQ][k]), q1 = load4(&sm.gate[kEQ][k + 8]);
          const Pieces left = pieces_of_any(product(gather4(&sm.pd[k][m], kSquarePad), q0),
                                            product(gather4(&sm.pd[k + 8][m], kSquarePad), q1));
          dk[ti] = mma_exact(dk[ti], left, as_operand(qc[s], qc[s + 1]));
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        const int k = 8 * s + 4 * h;
        if (s < 4 * (ti + 1)) dq[ti] = mma(dq[ti], load4(&sm.pd[m][k]), kc[s]);
        dk[ti] = mma(dk[ti], load4(&sm.x[m][k]), kc[s]);
        if (s >= 4 * ti) dk[ti] = mma(dk[ti], gather4(&sm.pd[k][m], kSquarePad), qc[s]);
      }
    }
    keep_order();
#pragma unroll
    for (int i = 0; i < 16; ++i) products[i] = dq[ti][i] * element(numbers(qc[4 * ti + i / 4]), i);
    row_sums(kDotQ, ti, products);
#pragma unroll
    for (int i = 0; i < 16; ++i) products[i] = dk[ti][i] * element(numbers(kc[4 * ti + i / 4]), i);
    row_sums(kDotK, ti, products);
    keep_order();
  }
  lds_barrier();
  // over the waves; the two that every lane needs below once for all of them
  auto across_waves = [&](RowSum which, int row) {
    const float4 four = load4(sm.parts[which][row]);
    return (four.x + four.y) + (four.z + four.w);
  };
  if (tid < 2 * kC) sm.dots[tid / kC][tid % kC] = across_waves(tid < kC ? kDotQ : kDotK, tid % kC);
  lds_barrier();
  const Tokens partials = v.qk_partials();
  // back through the L2 normalisations (and the 1/sqrt(d) of q, which kQScale has)
  const unsigned partial_at = 2 * token_row * v.out_bytes + token_column;
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float4 q = numbers(qc[4 * ti + j]), k = numbers(kc[4 * ti + j]), q_scale = rows4(sm.gate[kQScale], ti, j),
                   k_scale = rows4(sm.gate[kKScale], ti, j);
      float4 q_dot = rows4(sm.dots[0], ti, j), k_dot = rows4(sm.dots[1], ti, j);
      if constexpr (BF16) {
        q_dot = product(q_dot, rows4(sm.gate[kEQ], ti, j));
        k_dot = product(k_dot, rows4(sm.gate[kLK], ti, j));
      }
      float from_q[4], from_k[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        from_q[e] = element(q_scale, e) *
                    (dq[ti][4 * j + e] - static_cast<float>(kD) * element(q, e) * element(q_dot, e));
        from_k[e] = element(k_scale, e) * (dk[ti][4 * j + e] - element(k, e) * element(k_dot, e));
      }
      const unsigned uniform = 2 * (32 * ti + 8 * j) * v.out_bytes;
      partials.put4(quad_transpose(make_float4(from_q[0], from_q[1], from_q[2], from_q[3])), partial_at, uniform);
      partials.put4(quad_transpose(make_float4(from_k[0], from_k[1], from_k[2], from_k[3])), partial_at,
                    uniform + 4 * kD);
    }
  if (wave != 0) return;
  // the gates: lane i is token i
  const float beta = sm.gate[kBeta][lane];
  const float r = across_waves(kSumW, lane), state_k = across_waves(kSumK, lane);
  const float row_n = sm.row_n[lane][0] + sm.row_n[lane][1];
  float dg = across_waves(kSumQ, lane) + beta * r +
             (beta * row_n - (sm.col_n[lane][0] + sm.col_n[lane][1])) +
             ((sm.row_p[lane][0] + sm.row_p[lane][1]) - (sm.col_p[lane][0] + sm.col_p[lane][1])) -
             state_k;
  const float total = wave_sum(state_k);
  if (lane == kC - 1)
    dg += total + ((sm.dot[0] + sm.dot[1]) + (sm.dot[2] + sm.dot[3])) * sm.gate[kE][kC - 1];
#pragma unroll
  for (int offset = 1; offset < 64; offset <<= 1) {
    const float after = __shfl_down(dg, offset, 64);
    if (lane + offset < 64) dg += after;
  }
  const bool valid = lane < v.tokens;
  const size_t at = static_cast<size_t>(v.t0 + min(lane, v.tokens - 1)) * a.vh + v.head;
  const float dbeta = row_n + r + across_waves(kSumV, lane);
  const float alpha = bf16_bits_to_float(a.a[at]) + a.dt_bias[v.head];
  const float softplus = fmaxf(alpha, 0.0f) + logf(1.0f + expf(-fabsf(alpha)));
  const float rate = expf(a.a_log[v.head]);
  const float bv = bf16_bits_to_float(a.b[at]);
  const float sigmoid = 1.0f / (1.0f + expf(-bv));
  const float d_alpha = -dg * rate / (1.0f + expf(-alpha));
  if (valid) {
    a.da[at] = d_alpha;
    a.db[at] = dbeta * sigmoid * (1.0f - sigmoid);
  }
  const float log_sum = wave_sum(valid ? -dg * rate * softplus : 0.0f), bias_sum = wave_sum(valid ? d_alpha : 0.0f);
  if (lane == 0) {
    float* out = a.scalar_partials + (static_cast<size_t>(blockIdx.x) * a.vh + v.head) * 2;
    out[0] = log_sum;
    out[1] = bias_sum;
  }
}

ChunkedArgs make_args(const GdnChunkedBackward& c) {
  ChunkedArgs a;
  a.post = c.post;
  a.a = c.a;
  a.b = c.b;
  a.a_log = c.a_log;
  a.dt_bias = c.dt_bias;
  a.dcore = c.dcore;
  a.core = c.core;
  a.dpost = c.dpost;
  a.qk_partials = c.qk_partials;
  a.da = c.da;
  a.db = c.db;
  a.scalar_partials = c.scalar_partials;
  a.length = c.length;
  a.chunks = (c.length + kC - 1) / kC;
  a.kh = c.key_heads;
  a.vh = c.value_heads;
  a.round = c.round;
  const size_t n = static_cast<size_t>(a.chunks) * a.vh;
  float* at = c.records;
  auto take = [&](size_t floats) {
    float* result = at;
    at += n * floats;
    return result;
  };
  a.r.w_rows = take(kWide);
  a.r.w_columns = take(kWide);
  a.r.u_columns = take(kWide);
  a.r.dl_rows = take(kWide);
  a.r.ddl_rows = take(kWide);
  a.r.p_rows = take(kSquare);
  a.r.p_columns = take(kSquare);
  a.r.t_columns = take(kSquare);
  a.r.kkd = take(kSquare);
  a.r.gates = take(kGateRows * kC);
  a.r.s0 = take(kState);
  a.r.ds1 = take(kState);
  const size_t keys = static_cast<size_t>(a.chunks) * a.kh * kWide;
  if (a.round) {
    a.r.keys = reinterpret_cast<uint16_t*>(at);
  } else {
    a.r.q_rows = at;
    a.r.q_columns = at + keys;
    a.r.k_rows = at + 2 * keys;
    a.r.k_columns = at + 3 * keys;
  }
  return a;
}

// Tiles of sixteen columns a workgroup of the sequential kernels takes.  While every
// tile gets a compute unit of its own one is faster; beyond that compute units hold
// two tiles anyway, and one workgroup with both loads the operands once.
int column_tiles(int value_heads) { return value_heads * (kD / kTile) > 256 ? 2 : 1; }
template <class Launch>
void by_tiles(const ChunkedArgs& a, Launch launch) {
  auto with = [&](auto tiles) { a.round ? launch(tiles, std::true_type()) : launch(tiles, std::false_type()); };
  column_tiles(a.vh) == 2 ? with(std::integral_constant<int, 2>()) : with(std::integral_constant<int, 1>());
}

}  // namespace

bool gdn_backward_chunked_supported(const pluto_hip_delta_params* p) {
  return p->key_head_dim == kD && p->value_head_dim == kD && p->key_heads > 0 &&
         p->value_heads % p->key_heads == 0;
}

size_t gdn_backward_chunked_bytes(const pluto_hip_delta_params* p, int length) {
  const size_t chunks = (static_cast<size_t>(length) + kC - 1) / kC;
  const size_t keys = p->key_heads * key_record_floats(p->round_to_bfloat16 != 0);
  return align_up(chunks * (p->value_heads * kRecordFloats + keys) * sizeof(float), 256);
}

int launch_gdn_backward_chunked_forward(hipStream_t stream, const GdnChunkedBackward& c) {
  const ChunkedArgs a = make_args(c);
  const dim3 per_chunk(a.chunks, a.vh);
  if (a.round)
    chunk_prepare_kernel<true><<<per_chunk, 256, 0, stream>>>(a);
  else
    chunk_prepare_kernel<false><<<per_chunk, 256, 0, stream>>>(a);
  const int status = launch_status();
  if (status != 0) return status;
  by_tiles(a, [&](auto tiles, auto bf16) {
    chunk_states_forward_kernel<tiles, bf16><<<a.vh * (kD / (tiles * kTile)), kSequentialThreads<tiles, bf16>, 0, stream>>>(a);
  });
  return launch_status();
}

int launch_gdn_backward_chunked_reverse(hipStream_t stream, const GdnChunkedBackward& c) {
  const ChunkedArgs a = make_args(c);
  by_tiles(a, [&](auto tiles, auto bf16) {
    chunk_states_backward_kernel<tiles, bf16><<<a.vh * (kD / (tiles * kTile)), kSequentialThreads<tiles, bf16>, 0, stream>>>(a);
  });
  const int status = launch_status();
  if (status != 0) return status;
  if (a.round)
    chunk_gradients_kernel<true><<<dim3(a.chunks, a.vh), 256, 0, stream>>>(a);
  else
    chunk_gradients_kernel<false><<<dim3(a.chunks, a.vh), 256, 0, stream>>>(a);
  return launch_status();
}

}  // namespace pluto_hip
