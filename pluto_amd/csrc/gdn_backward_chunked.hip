// Chunked backward of the gated delta rule for 128 x 128 heads: the same
// gradients as the token-by-token kernels of gdn_backward.hip
// (RecurrenceForward / RecurrenceBackward, src/llm/layers/
// sequence_delta_net.cc:55-102 and :171-253), computed 64 tokens at a time on
// the FP32 matrix cores, and with one saved state per chunk instead of one per
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
//   chunk_states_forward_kernel    S entering every chunk, Dl         (sequential)
//   chunk_outputs_kernel           O                                  (parallel)
//     -- the caller turns O into dO here --
//   chunk_states_backward_kernel   dS' leaving every chunk, dDl       (sequential)
//   chunk_gradients_kernel         everything else                    (parallel)
// The sequential kernels run one workgroup per (head, 16 value columns).
// Eliminating Dl instead makes both recurrences one 128 x 128 matrix a chunk
// (S' = M S + B) whose product is one link of the chain instead of two, but M, its
// transpose, B and the offsets of the reverse recurrence are four 64 KiB records a
// chunk that have to be computed, written and read: at 2048 tokens of 48 heads the
// kernels that did so took 624 us where the two below take 380.
// Everything between two states is consumed in the kernel that makes it (LDS and
// accumulators), so that a chunk's records are 0.27 MB instead of 0.74 MB: all kernels
// of this file 1766 -> 930 us at that size.
// Matrix products run on v_mfma_f32_32x32x2_f32 and v_mfma_f32_16x16x4_f32, whose
// rate (about 25 GFLOP of them, 165 us of the card's FP32 matrix rate) bounds the
// gradients kernel; the triangular factors are multiplied by halves.
#include "gdn.h"

namespace pluto_hip {
namespace {

constexpr int kC = 64;       // tokens per chunk
constexpr int kD = 128;      // key and value channels per head
constexpr int kSlice = 16;   // value columns per workgroup of the sequential kernels
constexpr int kWide = kC * kD;     // elements of a [64, 128] record
constexpr int kSquare = kC * kC;   // elements of a [64, 64] record
constexpr int kState = kD * kD;    // elements of a state
constexpr int kWidePad = kD + 4;   // LDS rows: 16-byte aligned, neighbours four banks apart
constexpr int kSquarePad = kC + 4;

// Per (head, chunk) records in the workspace, in floats.
struct Records {
  float *w, *dl, *ddl;        // W; U, which Dl replaces; dDl            [64][128]
  float *p, *tm, *kkd;        // P, T, strict_lower((k^_i . k^_j) D_ij)  [64][64]
  float *gates;               // [8][64], see Gate
  float *s0, *ds1;            // state entering the chunk, gradient of the state leaving it
};

// Rows of a gates record.  q^ and k^ are not stored: their rows are those of the
// convolved activations times kQScale and kKScale (zero beyond the sequence).
enum Gate { kG, kBeta, kQScale, kKScale, kE, kL, kLK, kEQ, kGateRows };  // kLK = L kKScale, ...

constexpr size_t kRecordFloats = 3 * static_cast<size_t>(kWide) + 3 * kSquare + kGateRows * kC +
                                 2 * static_cast<size_t>(kState);

struct ChunkedArgs {
  const float* post = nullptr;     // [T, channels]
  const uint16_t* a = nullptr;     // bf16 [T, vh]
  const uint16_t* b = nullptr;
  const float* a_log = nullptr;
  const float* dt_bias = nullptr;
  const float* dcore = nullptr;    // [T, vh, 128]
  float* core = nullptr;           // [T, vh, 128]
  float* dpost = nullptr;          // [T, channels]: the value part is written
  float* qk_partials = nullptr;    // [T, vh, 2, 128]
  float* scalar_partials = nullptr;  // [T, vh, 3]
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

// Barrier for data exchanged through LDS only: pending global loads and
// stores stay in flight across it.
__device__ inline void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Sums over the 32 lanes of a half wave of sixteen values at once: lanes 2 j and 2 j + 1
// of a half return the sum of value j.  Each exchange halves the values a lane holds.
__device__ inline float half_sums(const float (&values)[16]) {
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = values[i];
  const int n = threadIdx.x % 32;
#pragma unroll
  for (int width = 8; width > 0; width /= 2) {
    const bool upper = n & (2 * width);
#pragma unroll
    for (int i = 0; i < width; ++i) {
      const float kept = upper ? v[i + width] : v[i], sent = upper ? v[i] : v[i + width];
      v[i] = kept + __shfl_xor(sent, 2 * width, 64);
    }
  }
  return v[0] + __shfl_xor(v[0], 1, 64);
}

// Memory behind a buffer descriptor: a lane's byte offset, computed once, and a uniform
// byte offset, so that a kernel keeps no addresses in vector registers.  Rows of
// TOKENS may lie beyond the end: there the sum is the offset the descriptor checks,
// reads give zero and writes are dropped, without a branch.
template <bool TOKENS>
struct Memory {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ Memory(const float* base, size_t elements)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0,
                                               static_cast<int>(elements * 4), 0x00020000)) {}
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
};
using Record = Memory<false>;
using Tokens = Memory<true>;

// One chunk of one head.  Tokens beyond the sequence have zero rows, scales, beta and
// gradients.
struct ChunkView {
  const ChunkedArgs& a;
  size_t rec;
  int t0, head, tokens, channels;
  unsigned row_bytes, out_bytes;   // a token's row in the activations, in dO and O
  const float* gates;
  __device__ ChunkView(const ChunkedArgs& args, int chunk, int head_)
      : a(args), rec(static_cast<size_t>(head_) * args.chunks + chunk), t0(chunk * kC), head(head_),
        tokens(min(args.length - t0, kC)), channels(2 * args.kh * kD + args.vh * kD),
        row_bytes(channels * 4), out_bytes(args.vh * kD * 4), gates(args.r.gates + rec * kGateRows * kC) {}
  __device__ Tokens activations(const float* base, int column) const {
    return Tokens(base + static_cast<size_t>(t0) * channels + column,
                  static_cast<size_t>(tokens) * channels - column);
  }
  __device__ int key_head() const { return head / (a.vh / a.kh); }
  __device__ int value_column() const { return (2 * a.kh + head) * kD; }
  __device__ Tokens q() const { return activations(a.post, key_head() * kD); }
  __device__ Tokens k() const { return activations(a.post, (a.kh + key_head()) * kD); }
  __device__ Tokens v() const { return activations(a.post, value_column()); }
  __device__ Tokens dv() const { return activations(a.dpost, value_column()); }
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
constexpr unsigned kWideRow = kD * 4, kSquareRow = kC * 4;  // bytes

// ---------------------------------------------------------------------------
// T, W, U, P and the gates of one chunk.  68 KiB of LDS, two workgroups a compute
// unit.  The inverse is made by blocks: the four 16 x 16 diagonal blocks by forward
// substitution, one wave each, then -T22 A21 T11 twice on the matrix cores (a
// substitution over all 64 rows by one wave held the other three up for a third of
// the kernel).
__global__ void __launch_bounds__(256)
chunk_prepare_kernel(ChunkedArgs a) {
  __shared__ __attribute__((aligned(16))) struct {
    float k[kC][kWidePad];
    union {
      float q[kC][kWidePad];
      struct {
        float a[kC][kSquarePad], t[kC][kSquarePad];
      };
    };
    float g[kC], beta[kC], fk[kC];
  } sm;
  const ChunkView v(a, blockIdx.x, blockIdx.y);
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int h = lane / 32, n = lane % 32, quarter = lane / 16, n16 = lane % 16;
  float* gates = a.r.gates + v.rec * kGateRows * kC;

  // normalised rows (1e-6 added to the sums of squares, sequence_delta_net.cc:84-85):
  // half a wave a row, row 16 wave + 2 r + h
  {
    const float norm_scale = sqrtf(static_cast<float>(kD));
    const Tokens q = v.q(), k = v.k();
    const unsigned at = (16 * wave + h) * v.row_bytes + 16 * n;
    float4 rows[16];
    float squares[16];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      rows[2 * r] = q.get4(at, 2 * r * v.row_bytes);
      rows[2 * r + 1] = k.get4(at, 2 * r * v.row_bytes);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r)
      squares[r] = (rows[r].x * rows[r].x + rows[r].y * rows[r].y) +
                   (rows[r].z * rows[r].z + rows[r].w * rows[r].w);
    const float sum = half_sums(squares);  // lane 2 j holds that of rows[j]
    const float inverse = rsqrtf(sum + 1e-6f);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int i = 16 * wave + 2 * r + h;
      const bool ok = i < v.tokens;
      const float iq = ok ? __shfl(inverse, 32 * h + 4 * r, 64) / norm_scale : 0.0f;
      const float ik = ok ? __shfl(inverse, 32 * h + 4 * r + 2, 64) : 0.0f;
      store4(&sm.q[i][4 * n], scaled(rows[2 * r], iq));
      store4(&sm.k[i][4 * n], scaled(rows[2 * r + 1], ik));
      if (n == 0) {
        gates[kQScale * kC + i] = iq;
        gates[kKScale * kC + i] = ik;
        sm.fk[i] = ik;  // until the gates below
        sm.beta[i] = iq;
      }
    }
  }
  __syncthreads();
  // gates (sequence_delta_net.cc:88-96); tokens beyond the sequence neither
  // decay nor write
  if (wave == 0) {
    const int t = v.t0 + lane;
    float g = 0.0f, beta = 0.0f;
    if (lane < v.tokens) {
      const float alpha =
          bf16_bits_to_float(a.a[static_cast<size_t>(t) * a.vh + v.head]) + a.dt_bias[v.head];
      const float softplus = fmaxf(alpha, 0.0f) + logf(1.0f + expf(-fabsf(alpha)));
      g = -expf(a.a_log[v.head]) * softplus;
      const float bv = bf16_bits_to_float(a.b[static_cast<size_t>(t) * a.vh + v.head]);
      beta = round_if(1.0f / (1.0f + expf(-bv)), a.round);
    }
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
      const float before = __shfl_up(g, offset, 64);
      if (lane >= offset) g += before;
    }
    const float e = expf(g), l = expf(__shfl(g, 63, 64) - g);
    gates[kG * kC + lane] = g;
    gates[kBeta * kC + lane] = beta;
    gates[kE * kC + lane] = e;
    gates[kL * kC + lane] = l;
    gates[kLK * kC + lane] = l * sm.fk[lane];
    gates[kEQ * kC + lane] = e * sm.beta[lane];
    sm.g[lane] = g;
    sm.beta[lane] = beta;
    sm.fk[lane] = beta * e;
  }
  __syncthreads();
  // k^ k^T and q^ k^T by 16 x 16 tiles on and below the diagonal: wave w takes row w of
  // the first and row 3 - w of the second, five tiles
  floatx4 kk[4], qk[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) kk[b] = qk[b] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
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
  }
  __syncthreads();  // the rows of q^ make room for A and T
  const auto kkd = v.square(a.r.kkd), p = v.square(a.r.p);
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = 4 * quarter + e, col = 16 * b + n16;
      const int k_at = 16 * wave + row, q_at = 16 * (3 - wave) + row;
      const float kv = k_at > col ? kk[b][e] * expf(sm.g[k_at] - sm.g[col]) : 0.0f;
      kkd.put(kv, 4 * (k_at * kC + n16), 64 * b);
      p.put(q_at >= col ? qk[b][e] * expf(sm.g[q_at] - sm.g[col]) : 0.0f, 4 * (q_at * kC + n16), 64 * b);
      sm.a[k_at][col] = sm.beta[k_at] * kv;
      sm.t[k_at][col] = 0.0f;
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
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    values[s] = value_memory.gather4(4 * h * v.row_bytes + 4 * col, 8 * s * v.row_bytes, v.row_bytes);
  }
  __builtin_amdgcn_sched_barrier(0);
  lds_barrier();
#pragma unroll
  for (int i = 0; i < kC * kC / 4 / 256; ++i) {
    const int at = tid + 256 * i;
    store4(a.r.tm + v.rec * kSquare + 4 * at, load4(&sm.t[at / 16][at % 16 * 4]));
  }
  const auto w_out = v.wide(a.r.w), u_out = v.wide(a.r.dl);
#pragma unroll
  for (int ti = 0; ti < 2; ++ti) {
    floatx16 w = zero_tile(), u = zero_tile();
#pragma unroll
    for (int s = 0; s < 4 * (ti + 1); ++s) {
      const int k = 8 * s + 4 * h;
      const float4 t = load4(&sm.t[32 * ti + n][k]), f = load4(&sm.fk[k]), b = load4(&sm.beta[k]);
      w = mma(w, make_float4(t.x * f.x, t.y * f.y, t.z * f.z, t.w * f.w), gather4(&sm.k[k][col], kWidePad));
      u = mma(u, make_float4(t.x * b.x, t.y * b.y, t.z * b.z, t.w * b.w), values[s]);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const unsigned at = 4 * h * kWideRow + 4 * col, row = (32 * ti + tile_row(i, 0)) * kWideRow;
      w_out.put(w[i], at, row);
      u_out.put(u[i], at, row);
    }
  }
}

// ---------------------------------------------------------------------------
// The workgroups of the sequential kernels.  The eight column slices of a head read
// the same matrices: they are given block numbers with the same remainder mod 8,
// which the hardware places on one XCD, so that seven of the eight reads are served
// by that XCD's L2.
struct Slice {
  int head, col0;
};
__device__ inline Slice slice_of_block(const ChunkedArgs& a) {
  constexpr int kSlices = kD / kSlice;
  static_assert(kSlices == 8, "one slice of a head per block of an XCD's share");
  if (a.vh % 8 == 0)
    return {static_cast<int>((blockIdx.x % 8) * (a.vh / 8) + blockIdx.x / 64),
            static_cast<int>(blockIdx.x / 8 % kSlices * kSlice)};
  return {static_cast<int>(blockIdx.x / kSlices), static_cast<int>(blockIdx.x % kSlices * kSlice)};
}

// The state of a slice lives in accumulators: wave w holds rows 32 w .. 32 w + 31, as two
// 16 x 16 tiles whose rows are interleaved (row 32 w + 2 i + t is row i of tile t), so
// that an operand row that is contiguous along them is read two elements a lane and a
// lane's eight elements are rows 32 w + 8 quarter .. + 7.  `rows` is the LDS copy
// [column][row] that the other waves multiply.
__device__ inline void publish_state(const floatx4 (&acc)[2], float* rows) {
  store4(rows, make_float4(acc[0][0], acc[1][0], acc[0][1], acc[1][1]));
  store4(rows + 4, make_float4(acc[0][2], acc[1][2], acc[0][3], acc[1][3]));
}

__device__ inline void save_state(const floatx4 (&acc)[2], const Record& state, unsigned lane) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int t = 0; t < 2; ++t) state.put(acc[t][e], lane, (2 * e + t) * kWideRow);
}

// S entering every chunk and Dl of every chunk.  Wave w computes rows 16 w .. 16 w + 15
// of Dl from the whole state and then its rows of the new state from all of Dl: two
// dependent products of 32 matrix instructions a chunk.  The operands of the chunk
// after next are requested as soon as this chunk's have been multiplied.
__global__ void __launch_bounds__(256)
chunk_states_forward_kernel(ChunkedArgs a) {
  __shared__ __attribute__((aligned(16))) float state[kSlice][kWidePad], delta[kSlice][kSquarePad];
  const Slice slice = slice_of_block(a);
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int quarter = lane / 16, n = lane % 16;
  const int col = slice.col0 + n;
  struct Operands {
    float4 w[8];
    float2 k[16];
    float u[4];
    float4 scale;
    float decay;
  };
  auto view = [&](int chunk) { return ChunkView(a, min(chunk, a.chunks - 1), slice.head); };
  // a lane's places in a record of rows of all channels: its row as the left operand,
  // its rows as a result, its rows and channels as the transposed left operand
  const unsigned row_at = (16 * wave + n) * kWideRow + 16 * quarter;
  const unsigned result_at = (16 * wave + 4 * quarter) * kWideRow + 4 * col;
  const unsigned state_at = (32 * wave + 8 * quarter) * kWideRow + 4 * col;
  auto request_delta = [&](const ChunkView& v, Operands& o) {
    const auto w = v.wide(a.r.w), u = v.wide(a.r.dl);
#pragma unroll
    for (int s = 0; s < 8; ++s) o.w[s] = w.get4(row_at, 64 * s);
#pragma unroll
    for (int e = 0; e < 4; ++e) o.u[e] = u.get(result_at, e * kWideRow);
    o.scale = load4(v.gates + kLK * kC + 16 * wave + 4 * quarter);
  };
  auto request_state = [&](const ChunkView& v, Operands& o) {
    const auto k = v.k();
    const unsigned at = 4 * quarter * v.row_bytes + 4 * (32 * wave + 2 * n);
#pragma unroll
    for (int j = 0; j < 16; ++j) o.k[j] = k.get2(at, (16 * (j / 4) + j % 4) * v.row_bytes);
    o.decay = v.gates[kE * kC + kC - 1];
  };
  floatx4 acc[2];
  acc[0] = acc[1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  auto advance = [&](int chunk, Operands& o) {
    const ChunkView v(a, chunk, slice.head), later = view(chunk + 2);
    const auto dl_out = v.wide(a.r.dl);
    publish_state(acc, &state[n][32 * wave + 8 * quarter]);
    save_state(acc, v.state(a.r.s0), state_at);
    lds_barrier();
    floatx4 even = {0.0f, 0.0f, 0.0f, 0.0f}, odd = even;
    float4 b[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) b[s] = load4(&state[n][16 * s + 4 * quarter]);
#pragma unroll
    for (int s = 0; s < 8; s += 2) {
      even = mma16(even, o.w[s], b[s]);
      odd = mma16(odd, o.w[s + 1], b[s + 1]);
    }
    float dl[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      dl[e] = o.u[e] - (even[e] + odd[e]);
      dl_out.put(dl[e], result_at, e * kWideRow);
    }
    store4(&delta[n][16 * wave + 4 * quarter],
           make_float4(dl[0] * o.scale.x, dl[1] * o.scale.y, dl[2] * o.scale.z, dl[3] * o.scale.w));
    __builtin_amdgcn_sched_barrier(0);
    request_delta(later, o);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
#pragma unroll
    for (int s = 0; s < 4; ++s) b[s] = load4(&delta[n][16 * s + 4 * quarter]);
    acc[0] *= o.decay;
    acc[1] *= o.decay;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      acc[0] = mma16(acc[0], make_float4(o.k[4 * s].x, o.k[4 * s + 1].x, o.k[4 * s + 2].x, o.k[4 * s + 3].x), b[s]);
      acc[1] = mma16(acc[1], make_float4(o.k[4 * s].y, o.k[4 * s + 1].y, o.k[4 * s + 2].y, o.k[4 * s + 3].y), b[s]);
    }
    __builtin_amdgcn_sched_barrier(0);
    request_state(later, o);
    __builtin_amdgcn_sched_barrier(0);
  };
  Operands even, odd;
  request_delta(view(0), even);
  request_state(view(0), even);
  request_delta(view(1), odd);
  request_state(view(1), odd);
  for (int chunk = 0; chunk < a.chunks; chunk += 2) {
    advance(chunk, even);
    if (chunk + 1 < a.chunks) advance(chunk + 1, odd);
  }
}

// The gradient of the state leaving every chunk and dDl of every chunk, chunks in
// reverse.  112 matrix instructions a wave and chunk; the products with dO do not
// depend on the chain and run while it waits.
__global__ void __launch_bounds__(256)
chunk_states_backward_kernel(ChunkedArgs a) {
  __shared__ __attribute__((aligned(16))) float state[kSlice][kWidePad], delta[kSlice][kSquarePad],
      grad[kSlice][kSquarePad], query_grad[kSlice][kSquarePad];
  const Slice slice = slice_of_block(a);
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int quarter = lane / 16, n = lane % 16;
  const int col = slice.col0 + n;
  auto view = [&](int chunk) { return ChunkView(a, max(chunk, 0), slice.head); };
  float4 k[8];
  float p[16], out[4];
  float2 q[16], w[16];
  float4 k_scale, q_scale;
  float decay;
  const int rows = 16 * wave + 4 * quarter;
  const unsigned result_at = rows * kWideRow + 4 * col;
  const unsigned state_at = (32 * wave + 8 * quarter) * kWideRow + 4 * col;
  auto request_out = [&](const ChunkView& v) {
    const auto d_out = v.heads(a.dcore);
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = d_out.get(rows * v.out_bytes + 4 * col, e * v.out_bytes);
    q_scale = load4(v.gates + kEQ * kC + rows);
  };
  auto request_delta = [&](const ChunkView& v) {
    const Record p_memory = v.square(a.r.p);
    const Tokens k_memory = v.k();
#pragma unroll
    for (int j = 0; j < 16; ++j)
      p[j] = p_memory.get(4 * quarter * kSquareRow + 4 * (16 * wave + n), (16 * (j / 4) + j % 4) * kSquareRow);
#pragma unroll
    for (int s = 0; s < 8; ++s) k[s] = k_memory.get4((16 * wave + n) * v.row_bytes + 16 * quarter, 64 * s);
    k_scale = load4(v.gates + kLK * kC + rows);
  };
  auto request_query = [&](const ChunkView& v) {
    const auto q_memory = v.q();
    const unsigned at = 4 * quarter * v.row_bytes + 4 * (32 * wave + 2 * n);
#pragma unroll
    for (int j = 0; j < 16; ++j) q[j] = q_memory.get2(at, (16 * (j / 4) + j % 4) * v.row_bytes);
    decay = v.gates[kE * kC + kC - 1];
  };
  auto request_weights = [&](const ChunkView& v) {
    const auto w_memory = v.wide(a.r.w);
#pragma unroll
    for (int j = 0; j < 16; ++j)
      w[j] = w_memory.get2(4 * quarter * kWideRow + 4 * (32 * wave + 2 * n), (16 * (j / 4) + j % 4) * kWideRow);
  };
  floatx4 acc[2];
  acc[0] = acc[1] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  {
    const ChunkView v = view(a.chunks - 1);
    request_out(v);
    request_delta(v);
    request_query(v);
    request_weights(v);
  }
  for (int chunk = a.chunks - 1; chunk >= 0; --chunk) {
    const ChunkView v(a, chunk, slice.head), later = view(chunk - 1);
    const auto ddl_out = v.wide(a.r.ddl);
    publish_state(acc, &state[n][32 * wave + 8 * quarter]);
    store4(&grad[n][rows], make_float4(out[0], out[1], out[2], out[3]));
    store4(&query_grad[n][rows],
           make_float4(out[0] * q_scale.x, out[1] * q_scale.y, out[2] * q_scale.z, out[3] * q_scale.w));
    save_state(acc, v.state(a.r.ds1), state_at);
    __builtin_amdgcn_sched_barrier(0);
    request_out(later);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    floatx4 from_out = {0.0f, 0.0f, 0.0f, 0.0f}, even = from_out, odd = from_out;
    float4 b[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) b[s] = load4(&state[n][16 * s + 4 * quarter]);
    float4 g[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) g[s] = load4(&grad[n][16 * s + 4 * quarter]);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      even = mma16(even, k[2 * s], b[2 * s]);
      odd = mma16(odd, k[2 * s + 1], b[2 * s + 1]);
      from_out = mma16(from_out, make_float4(p[4 * s], p[4 * s + 1], p[4 * s + 2], p[4 * s + 3]), g[s]);
    }
    float dd[4];
    const float scale[4] = {k_scale.x, k_scale.y, k_scale.z, k_scale.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      dd[e] = from_out[e] + scale[e] * (even[e] + odd[e]);
      ddl_out.put(dd[e], result_at, e * kWideRow);
    }
    store4(&delta[n][rows], make_float4(-dd[0], -dd[1], -dd[2], -dd[3]));
    __builtin_amdgcn_sched_barrier(0);
    request_delta(later);
    __builtin_amdgcn_sched_barrier(0);
    acc[0] *= decay;
    acc[1] *= decay;
#pragma unroll
    for (int s = 0; s < 4; ++s) g[s] = load4(&query_grad[n][16 * s + 4 * quarter]);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      acc[0] = mma16(acc[0], make_float4(q[4 * s].x, q[4 * s + 1].x, q[4 * s + 2].x, q[4 * s + 3].x), g[s]);
      acc[1] = mma16(acc[1], make_float4(q[4 * s].y, q[4 * s + 1].y, q[4 * s + 2].y, q[4 * s + 3].y), g[s]);
    }
    __builtin_amdgcn_sched_barrier(0);
    request_query(later);
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
#pragma unroll
    for (int s = 0; s < 4; ++s) g[s] = load4(&delta[n][16 * s + 4 * quarter]);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      acc[0] = mma16(acc[0], make_float4(w[4 * s].x, w[4 * s + 1].x, w[4 * s + 2].x, w[4 * s + 3].x), g[s]);
      acc[1] = mma16(acc[1], make_float4(w[4 * s].y, w[4 * s + 1].y, w[4 * s + 2].y, w[4 * s + 3].y), g[s]);
    }
    __builtin_amdgcn_sched_barrier(0);
    request_weights(later);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// ---------------------------------------------------------------------------
// O = diag(E) Q^ S + P Dl of one chunk.  Wave w owns value columns 32w..32w+31 and has
// its part of S and Dl in registers, requested before the rows of Q^ and P are staged
// for all waves.
__global__ void __launch_bounds__(256)
chunk_outputs_kernel(ChunkedArgs a) {
  __shared__ __attribute__((aligned(16))) float q_s[kC][kWidePad], p_s[kC][kSquarePad];
  const ChunkView v(a, blockIdx.x, blockIdx.y);
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int h = lane / 32, n = lane % 32;
  const int col = 32 * wave + n;
  const Tokens q = v.q(), core = v.heads(a.core);
  const Record p = v.square(a.r.p), state = v.state(a.r.s0), delta = v.wide(a.r.dl);
  float4 rows[8], p_rows[4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    rows[i] = scaled(q.get4(tid / 32 * v.row_bytes + tid % 32 * 16, 8 * i * v.row_bytes),
                     v.gates[kEQ * kC + tid / 32 + 8 * i]);
#pragma unroll
  for (int i = 0; i < 4; ++i) p_rows[i] = p.get4(16 * tid, 4096 * i);
  const unsigned column_at = 4 * h * kWideRow + 4 * col;
  float4 s_col[16], d_col[8];
#pragma unroll
  for (int s = 0; s < 16; ++s) s_col[s] = state.gather4(column_at, 8 * s * kWideRow, kWideRow);
#pragma unroll
  for (int s = 0; s < 8; ++s) d_col[s] = delta.gather4(column_at, 8 * s * kWideRow, kWideRow);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int at = tid + 256 * i;
    store4(&q_s[at / 32][at % 32 * 4], rows[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = tid + 256 * i;
    store4(&p_s[at / 16][at % 16 * 4], p_rows[i]);
  }
  lds_barrier();
  floatx16 out[2];
  out[0] = out[1] = zero_tile();
#pragma unroll
  for (int s = 0; s < 16; ++s)
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
      out[ti] = mma(out[ti], load4(&q_s[32 * ti + n][8 * s + 4 * h]), s_col[s]);
#pragma unroll
  for (int s = 0; s < 8; ++s)
#pragma unroll
    for (int ti = 0; ti < 2; ++ti)
      if (s < 4 * (ti + 1)) out[ti] = mma(out[ti], load4(&p_s[32 * ti + n][8 * s + 4 * h]), d_col[s]);
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int i = 0; i < 16; ++i)
      core.put(round_if(out[ti][i], a.round), 4 * h * v.out_bytes + 4 * col,
               (32 * ti + tile_row(i, 0)) * v.out_bytes);
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
// 75 KiB of LDS and 256 registers: two workgroups a compute unit.
constexpr int kSlab = 32;
struct GradientSmem {
  union {
    float slab[4][kC][kSlab + 4];  // dDl, dO, Dl, V
    struct {
      float dw[kC][kWidePad], pd[kC][kSquarePad], x[kC][kSquarePad];
    };
  };
  float parts[6][kC][4];     // row sums of the waves' columns, see RowSum
  float row_n[kC][2], col_n[kC][2], row_p[kC][2], col_p[kC][2];  // by tile
  float gate[kGateRows][kC];
  float dot[4];
};
enum RowSum { kSumQ, kSumK, kSumW, kSumV, kDotQ, kDotK };

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
  for (int i = tid; i < kGateRows * kC; i += 256) sm.gate[i / kC][i % kC] = v.gates[i];
  if (tid < kC) {
    sm.row_n[tid][0] = sm.row_n[tid][1] = sm.col_n[tid][0] = sm.col_n[tid][1] = 0.0f;
    sm.row_p[tid][0] = sm.row_p[tid][1] = sm.col_p[tid][0] = sm.col_p[tid][1] = 0.0f;
  }
  floatx16 dw[2], dq[2], dk[2], dp = zero_tile(), dt = zero_tile();
#pragma unroll
  for (int ti = 0; ti < 2; ++ti) dw[ti] = dq[ti] = dk[ti] = zero_tile();
  float dot = 0.0f;
  {
    const Record s0_memory = v.state(a.r.s0), s1_memory = v.state(a.r.ds1), ddl = v.wide(a.r.ddl),
                 dl = v.wide(a.r.dl);
    const Tokens d_out = v.heads(a.dcore), values = v.v();
    const unsigned state_at = col * kWideRow + 16 * h;
    // thread (row, piece) of the slabs: rows r and r + 32, 16 bytes
    const int row = tid / 8, piece = tid % 8 * 4;
    float4 staged[8];
    auto request = [&](int slab) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const unsigned c = 4 * kSlab * slab;
        staged[4 * j] = ddl.get4(row * kWideRow + 4 * piece, 32 * j * kWideRow + c);
        staged[4 * j + 1] = d_out.get4(row * v.out_bytes + 4 * piece, 32 * j * v.out_bytes + c);
        staged[4 * j + 2] = dl.get4(row * kWideRow + 4 * piece, 32 * j * kWideRow + c);
        staged[4 * j + 3] = values.get4(row * v.row_bytes + 4 * piece, 32 * j * v.row_bytes + c);
      }
    };
    request(0);
    float4 s0[4], s1[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) s0[g] = s0_memory.get4(state_at, 32 * g), s1[g] = s1_memory.get4(state_at, 32 * g);
    float fv = 0.0f;
#pragma unroll
    for (int slab = 0; slab < kD / kSlab; ++slab) {
      if (slab > 0) lds_barrier();
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int m = 0; m < 4; ++m)
          store4(&sm.slab[m][row + 32 * j][piece], staged[4 * j + m]);
      if (slab == 0)
        __syncthreads();
      else
        lds_barrier();
      if (slab == 0) fv = sm.gate[kBeta][32 * tj_own + n];
      if (slab + 1 < kD / kSlab) request(slab + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int c = 8 * g + 4 * h;
        dot += (s0[g].x * s1[g].x + s0[g].y * s1[g].y) + (s0[g].z * s1[g].z + s0[g].w * s1[g].w);
#pragma unroll
        for (int ti = 0; ti < 2; ++ti) {
          dw[ti] = mma(dw[ti], load4(&sm.slab[0][32 * ti + n][c]), s0[g]);
          dq[ti] = mma(dq[ti], load4(&sm.slab[1][32 * ti + n][c]), s0[g]);
          dk[ti] = mma(dk[ti], load4(&sm.slab[2][32 * ti + n][c]), s1[g]);
        }
        if (slab + 1 < kD / kSlab) {
          s0[g] = s0_memory.get4(state_at, 4 * kSlab * (slab + 1) + 32 * g);
          s1[g] = s1_memory.get4(state_at, 4 * kSlab * (slab + 1) + 32 * g);
        }
        if (lower) {
          dp = mma(dp, load4(&sm.slab[1][32 * ti_own + n][c]), load4(&sm.slab[2][32 * tj_own + n][c]));
          dt = mma(dt, load4(&sm.slab[0][32 * ti_own + n][c]), scaled(load4(&sm.slab[3][32 * tj_own + n][c]), fv));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    dot = wave_sum(dot);
    if (lane == 0) sm.dot[wave] = dot;
  }
  lds_barrier();  // the slabs make room for dW, Pd and X
  const int tile_col = 32 * tj_own + n;
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int i = 0; i < 16; ++i) sm.dw[32 * ti + tile_row(i, h)][col] = -dw[ti][i];
  // row and column sums of a tile held in an accumulator, for its rows and columns
  auto tile_sums = [&](const float (&values)[16], float (&row_sums)[kC][2], float (&col_sums)[kC][2],
                       const float* weights) {
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      sum += weights ? weights[32 * ti_own + tile_row(i, h)] * values[i] : values[i];
    sum += __shfl_xor(sum, 32, 64);
    if (h == 0) col_sums[tile_col][ti_own] = sum;
    const float row_sum = half_sums(values);
    if (n % 2 == 0) row_sums[32 * ti_own + tile_row(n / 2, h)][tj_own] = row_sum;
  };
  const Record p_memory = v.square(a.r.p), kkd = v.square(a.r.kkd), tm = v.square(a.r.tm),
               ddl = v.wide(a.r.ddl);
  const Tokens q_memory = v.q(), k_memory = v.k(), v_memory = v.v(), dv = v.dv();
  // the accumulator's places in a [64, 64] tile and in a column of the [64, 128] matrices
  const unsigned tile_at = (32 * ti_own + 4 * h) * kSquareRow + 4 * tile_col;
  const unsigned column_at = 4 * h * kWideRow + 4 * col, token_at = 4 * h * v.row_bytes + 4 * col;
  float decay[16];  // D of the tile
  if (lower) {
    float products[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 32 * ti_own + tile_row(i, h);
      const bool in = row >= tile_col;
      decay[i] = in ? expf(sm.gate[kG][row] - sm.gate[kG][tile_col]) : 0.0f;
      sm.pd[row][tile_col] = in ? dp[i] * decay[i] : 0.0f;
      products[i] = in ? dp[i] * p_memory.get(tile_at, tile_row(i, 0) * kSquareRow) : 0.0f;
    }
    tile_sums(products, sm.row_p, sm.col_p, nullptr);
  }
  lds_barrier();
  if (lower) {
    const float fk = sm.gate[kBeta][tile_col] * sm.gate[kE][tile_col] * sm.gate[kKScale][tile_col];
    const unsigned k_at = tile_col * v.row_bytes + 16 * h;
#pragma unroll
    for (int s = 0; s < kD / 8; ++s)
      dt = mma(dt, load4(&sm.dw[32 * ti_own + n][8 * s + 4 * h]), scaled(k_memory.get4(k_at, 32 * s), fk));
#pragma unroll
    for (int i = 0; i < 16; ++i) sm.x[32 * ti_own + tile_row(i, h)][tile_col] = dt[i];
  }
  lds_barrier();
  floatx16 z = zero_tile();
  if (lower) {
    // T^T dT: rows k < i of T's column i are zero, tile (0, 1) of dT is not needed
#pragma unroll
    for (int s = 0; s < 8; ++s)
      if (s >= 4 * ti_own)
        z = mma(z, tm.gather4(4 * h * kSquareRow + 4 * (32 * ti_own + n), 8 * s * kSquareRow, kSquareRow),
                gather4(&sm.x[8 * s + 4 * h][tile_col], kSquarePad));
  }
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
      if (s < 4 * (tj_own + 1))
        da = mma(da, load4(&sm.x[32 * ti_own + n][8 * s + 4 * h]),
                 tm.get4(tile_col * kSquareRow + 16 * h, 32 * s));
  }
  lds_barrier();
  if (lower) {
    // R + R^T, and the sums of N = dA (k^ . k^) D
    float products[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 32 * ti_own + tile_row(i, h);
      const bool in = row > tile_col;
      const float value = in ? -da[i] : 0.0f;
      products[i] = value * kkd.get(tile_at, tile_row(i, 0) * kSquareRow);
      const float r = value * sm.gate[kBeta][row] * decay[i];
      if (row >= tile_col) sm.x[row][tile_col] = sm.x[tile_col][row] = r;
    }
    tile_sums(products, sm.row_n, sm.col_n, sm.gate[kBeta]);
  }
  // columns of K^ and Q^, both as operands and in the accumulators' rows
  float4 kc[8], qc[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int i = 8 * s + 4 * h;
    const float4 ks = load4(&sm.gate[kKScale][i]), qs = load4(&sm.gate[kQScale][i]);
    const float4 k = k_memory.gather4(token_at, 8 * s * v.row_bytes, v.row_bytes);
    const float4 q = q_memory.gather4(token_at, 8 * s * v.row_bytes, v.row_bytes);
    kc[s] = make_float4(k.x * ks.x, k.y * ks.y, k.z * ks.z, k.w * ks.w);
    qc[s] = make_float4(q.x * qs.x, q.y * qs.y, q.z * qs.z, q.w * qs.w);
  }
  auto element = [](const float4 (&c)[8], int ti, int i) {
    const float4 four = c[4 * ti + i / 4];
    return i % 4 == 0 ? four.x : i % 4 == 1 ? four.y : i % 4 == 2 ? four.z : four.w;
  };
  auto row_sums = [&](RowSum which, int ti, const float (&values)[16]) {
    const float sum = half_sums(values);
    if (n % 2 == 0) sm.parts[which][32 * ti + tile_row(n / 2, h)][wave] = sum;
  };
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int ti = 0; ti < 2; ++ti) {
    float first[16], second[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 32 * ti + tile_row(i, h);
      dq[ti][i] *= sm.gate[kE][row];
      dk[ti][i] *= sm.gate[kL][row];
      first[i] = dq[ti][i] * element(qc, ti, i);
      second[i] = dk[ti][i] * element(kc, ti, i);
    }
    row_sums(kSumQ, ti, first);
    row_sums(kSumK, ti, second);
  }
  lds_barrier();
#pragma unroll
  for (int ti = 0; ti < 2; ++ti) {
    const int m = 32 * ti + n;
    float4 t_col[8];
#pragma unroll
    for (int s = 4 * ti; s < 8; ++s) t_col[s] = tm.gather4(4 * h * kSquareRow + 4 * m, 8 * s * kSquareRow, kSquareRow);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int k = 8 * s + 4 * h;
      if (s < 4 * (ti + 1)) dq[ti] = mma(dq[ti], load4(&sm.pd[m][k]), kc[s]);
      dk[ti] = mma(dk[ti], load4(&sm.x[m][k]), kc[s]);
      if (s >= 4 * ti) dk[ti] = mma(dk[ti], gather4(&sm.pd[k][m], kSquarePad), qc[s]);
    }
    __builtin_amdgcn_sched_barrier(0);
    float products[16];
    {
      floatx16 tw = zero_tile();
#pragma unroll
      for (int s = 4 * ti; s < 8; ++s)
        tw = mma(tw, t_col[s], gather4(&sm.dw[8 * s + 4 * h][col], kWidePad));
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = 32 * ti + tile_row(i, h);
        products[i] = tw[i] * element(kc, ti, i) * sm.gate[kE][row];
        dk[ti][i] += sm.gate[kBeta][row] * sm.gate[kE][row] * tw[i];
      }
      row_sums(kSumW, ti, products);
    }
    __builtin_amdgcn_sched_barrier(0);
    {
      floatx16 tu = zero_tile();
#pragma unroll
      for (int s = 4 * ti; s < 8; ++s)
        tu = mma(tu, t_col[s], ddl.gather4(column_at, 8 * s * kWideRow, kWideRow));
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const unsigned row = (32 * ti + tile_row(i, 0)) * v.row_bytes;
        products[i] = tu[i] * v_memory.get(token_at, row);
        dv.put(sm.gate[kBeta][32 * ti + tile_row(i, h)] * tu[i], token_at, row);
      }
      row_sums(kSumV, ti, products);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 16; ++i) products[i] = dq[ti][i] * element(qc, ti, i);
    row_sums(kDotQ, ti, products);
#pragma unroll
    for (int i = 0; i < 16; ++i) products[i] = dk[ti][i] * element(kc, ti, i);
    row_sums(kDotK, ti, products);
  }
  lds_barrier();
  auto across_waves = [&](RowSum which, int row) {
    const float4 four = load4(sm.parts[which][row]);
    return (four.x + four.y) + (four.z + four.w);
  };
  const auto partials = v.qk_partials();
  // back through the L2 normalisations (and the 1/sqrt(d) of q, which kQScale has)
#pragma unroll
  for (int ti = 0; ti < 2; ++ti)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int row = 32 * ti + tile_row(i, h);
      const unsigned uniform = 2 * (32 * ti + tile_row(i, 0)) * v.out_bytes;
      partials.put(sm.gate[kQScale][row] *
                       (dq[ti][i] - static_cast<float>(kD) * element(qc, ti, i) * across_waves(kDotQ, row)),
                   8 * h * v.out_bytes + 4 * col, uniform);
      partials.put(sm.gate[kKScale][row] * (dk[ti][i] - element(kc, ti, i) * across_waves(kDotK, row)),
                   8 * h * v.out_bytes + 4 * (kD + col), uniform);
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
  const int t = v.t0 + lane;
  if (lane >= v.tokens) return;
  const float dbeta = row_n + r + across_waves(kSumV, lane);
  const float alpha = bf16_bits_to_float(a.a[static_cast<size_t>(t) * a.vh + v.head]) + a.dt_bias[v.head];
  const float softplus = fmaxf(alpha, 0.0f) + logf(1.0f + expf(-fabsf(alpha)));
  const float rate = expf(a.a_log[v.head]);
  const float bv = bf16_bits_to_float(a.b[static_cast<size_t>(t) * a.vh + v.head]);
  const float sigmoid = 1.0f / (1.0f + expf(-bv));
  float* out = a.scalar_partials + (static_cast<size_t>(t) * a.vh + v.head) * 3;
  out[0] = -dg * rate / (1.0f + expf(-alpha));
  out[1] = dbeta * sigmoid * (1.0f - sigmoid);
  out[2] = -dg * rate * softplus;
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
  a.r.w = take(kWide);
  a.r.dl = take(kWide);
  a.r.ddl = take(kWide);
  a.r.p = take(kSquare);
  a.r.tm = take(kSquare);
  a.r.kkd = take(kSquare);
  a.r.gates = take(kGateRows * kC);
  a.r.s0 = take(kState);
  a.r.ds1 = take(kState);
  return a;
}

}  // namespace

bool gdn_backward_chunked_supported(const pluto_hip_delta_params* p) {
  return p->key_head_dim == kD && p->value_head_dim == kD && p->key_heads > 0 &&
         p->value_heads % p->key_heads == 0;
}

size_t gdn_backward_chunked_bytes(const pluto_hip_delta_params* p, int length) {
  const size_t chunks = (static_cast<size_t>(length) + kC - 1) / kC;
  return align_up(chunks * p->value_heads * kRecordFloats * sizeof(float), 256);
}

int launch_gdn_backward_chunked_forward(hipStream_t stream, const GdnChunkedBackward& c) {
  const ChunkedArgs a = make_args(c);
  const dim3 per_chunk(a.chunks, a.vh);
  chunk_prepare_kernel<<<per_chunk, 256, 0, stream>>>(a);
  int status = launch_status();
  if (status != 0) return status;
  chunk_states_forward_kernel<<<a.vh * (kD / kSlice), 256, 0, stream>>>(a);
  status = launch_status();
  if (status != 0) return status;
  chunk_outputs_kernel<<<per_chunk, 256, 0, stream>>>(a);
  return launch_status();
}

int launch_gdn_backward_chunked_reverse(hipStream_t stream, const GdnChunkedBackward& c) {
  const ChunkedArgs a = make_args(c);
  chunk_states_backward_kernel<<<a.vh * (kD / kSlice), 256, 0, stream>>>(a);
  const int status = launch_status();
  if (status != 0) return status;
  chunk_gradients_kernel<<<dim3(a.chunks, a.vh), 256, 0, stream>>>(a);
  return launch_status();
}

}  // namespace pluto_hip
