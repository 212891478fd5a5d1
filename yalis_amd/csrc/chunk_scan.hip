// The recurrences of state_scan.hip over long spans, 64 tokens at a time, in float32 on the matrix cores
// (v_mfma_f32_16x16x4_f32).  With t, j the places in a chunk, S the memory before it, a_t the decays
// (one a head, or one a key channel), u_t what a token writes:
//
//   A[t][j] = k_t . (a_(j+1) .. a_t) k_j   (j < t)        B[t][j] = q_t . (a_(j+1) .. a_t) k_j   (j <= t)
//   delta rule:  u = T (v - K' S),  T = (I + diag(beta) A)^-1 diag(beta),  K'_t = (a_1 .. a_t) k_t
//   else:        u = (strength) v, the strength folded into B and into the keys of the last line
//   o_t = Q'_t S + sum over j <= t of B[t][j] u_j,   Q'_t = (a_1 .. a_t) q_t
//   S <- (a_1 .. a_n) S + sum over j of ((a_(j+1) .. a_n) k_j) u_j^T
// and with a bonus, where the read-out sees the memory as it was before the token: the products of Q' and of B
// end at a_(t-1), and B[t][t] = q_t . diag(bonus) k_t.
//
// chunk_prepare makes Q', K', the last line's keys, B and T of every (chunk, head): these do not depend on
// S, so all chunks are made side by side.  chunk_walk then takes a request's chunks one after the other, a
// workgroup a (request, head, 16 columns of S); the columns never meet.
//
// Products of decays are made by multiplication only, from a place between j and t outwards, so every
// factor is at most 1 and nothing is divided by what may have vanished: with a decay per channel the
// lower triangle of 64 x 64 is cut into blocks n x n below the diagonal, n = 32, 16, 8, 4, 2, 1, and in a block the
// rows' vectors carry the decays from the block's first token on, the columns' those up to the token before it.
//
// Bound by the walk, whose chunks come one after the other along the span: 3,700 clocks of matrix products a SIMD (128 channels, delta
// rule; 1.5 us) in 2.9 us, the rest being three meetings through LDS and what waits between them.  Four waves carry S on and four make
// the read-outs beside them: 2,048 tokens, 4 heads of 256 x 512 135 -> 95 us, 16 of 128 x 128 by the delta rule 123 -> 94, where the same four
// waves did both in turn; 8 requests of 400 tokens 137 -> 103 and 120 -> 94.  What that rests on: the loads of the next chunk are asked
// for between the products, a few at a time as their registers come free (all together they hold a wave's products up: 119 and 102 us),
// with one scalar base a chunk; asking two chunks ahead is no faster (132, 110: it is the loads' issue that costs, not their time).
//
// 2,048 tokens of one request in bfloat16, us (of which prepare; token by token: yk_linear_state_scan): 16 heads of 128 x 128, delta rule 120
// (33; 465), with decays per channel 131 (496); 4 of 256 x 512 gated 121 (33; 497); 32 of 64 x 64 with a bonus 66 (396); 32 of
// 128 x 64 by step 97 (396).  Errors against float64, of their size, of the read-outs 1.1e-7, 1.1e-7, 2.5e-7, 0.7e-7, 0.8e-7 (walked
// 1.1e-7, 1.1e-7, 2.6e-7, 0.9e-7, 0.9e-7) and of the kept memories 0.8e-7, 0.8e-7, 2.4e-7, 0.4e-7, 0.6e-7 (0.8e-7, 0.8e-7, 2.6e-7, 0.4e-7, 0.6e-7).
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef double f64x4_t __attribute__((ext_vector_type(4)));

constexpr int kTok = 64;         // tokens of a chunk
constexpr int kRow = 64 + 4;     // LDS rows of 64 floats: 16 lanes that read 16 bytes of neighbouring rows meet different banks
constexpr int kChannel = 1, kDelta = 2, kReadFirst = 4;  // KIND is a sum of these

// c + the products of 16 elements, which are summed on their own first (a sum of K terms then carries the rounding of
// about 16 + K / 16 additions)
__device__ __forceinline__ f32x4_t mma16(f32x4_t a, f32x4_t b, f32x4_t c) {
  f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; ++i) s = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], s, 0, 0, 0);
  return c + s;
}

// the same for four such pieces, and the sum of theirs without c (made side by side: a product waits for the one it adds to)
__device__ __forceinline__ f32x4_t mma64(const f32x4_t* a, const f32x4_t* b) {
  f32x4_t s[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int n = 0; n < 4; ++n)
      s[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[n][i], b[n][i], i == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : s[n], 0, 0, 0);
  return (s[0] + s[1]) + (s[2] + s[3]);
}

// c + a tile of 16 x 16 with zeros above its diagonal times 16 x 16: what is not finite in the second stays away from the rows
// before it (zero times it would not be zero)
__device__ __forceinline__ f32x4_t triangle16(f32x4_t a, f32x4_t b, f32x4_t c) {
  const float sum = fabsf(b[0]) + fabsf(b[1]) + fabsf(b[2]) + fabsf(b[3]);
  if (!__any(!(sum < INFINITY))) return mma16(a, b, c);
  const int r = threadIdx.x % 16, lg = threadIdx.x % 64 / 16;
  f32x4_t finite;
#pragma unroll
  for (int e = 0; e < 4; ++e) finite[e] = fabsf(b[e]) < INFINITY ? b[e] : 0.f;
  c = mma16(a, finite, c);
#pragma unroll 1
  for (int kk = 0; kk < 4; ++kk)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float y = __shfl(b[e], 16 * kk + r, 64);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = __shfl(a[e], 16 * kk + 4 * lg + i, 64);
        if (4 * kk + e <= 4 * lg + i && !(fabsf(y) < INFINITY)) c[i] = fmaf(x, y, c[i]);
      }
    }
  return c;
}

// c + row ROW of tiles, up to the diagonal's, times a column of them (the tiles' products side by side, added in their order)
template <int ROW>
__device__ __forceinline__ f32x4_t lower_row(const f32x4_t* a, const f32x4_t* b, f32x4_t c) {
  const float sum = fabsf(b[ROW][0]) + fabsf(b[ROW][1]) + fabsf(b[ROW][2]) + fabsf(b[ROW][3]);
  if (__any(!(sum < INFINITY))) {
#pragma unroll
    for (int m = 0; m < ROW; ++m) c = mma16(a[m], b[m], c);
    return triangle16(a[ROW], b[ROW], c);
  }
  f32x4_t s[ROW + 1];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int m = 0; m <= ROW; ++m)
      s[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m][i], b[m][i], i == 0 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : s[m], 0, 0, 0);
#pragma unroll
  for (int m = 0; m <= ROW; ++m) c = c + s[m];
  return c;
}

// eight consecutive elements of a 16-byte aligned row as floats
__device__ __forceinline__ void load8(const float* p, float* out) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  out[0] = a.x; out[1] = a.y; out[2] = a.z; out[3] = a.w; out[4] = b.x; out[5] = b.y; out[6] = b.z; out[7] = b.w;
}
__device__ __forceinline__ void load8(const bf16_t* p, float* out) {
  const uint4 w = *reinterpret_cast<const uint4*>(p);
  out[0] = __uint_as_float(w.x << 16); out[1] = __uint_as_float(w.x & 0xffff0000u);
  out[2] = __uint_as_float(w.y << 16); out[3] = __uint_as_float(w.y & 0xffff0000u);
  out[4] = __uint_as_float(w.z << 16); out[5] = __uint_as_float(w.z & 0xffff0000u);
  out[6] = __uint_as_float(w.w << 16); out[7] = __uint_as_float(w.w & 0xffff0000u);
}

// a decay per key channel from its biased logit: kinds 1, 2 and 3 of yk_linear_state_scan
__device__ __forceinline__ float decay_of(float x, int mode, float tau, float rate) {
  if (mode == 1) return expf(-softplus_f32(-x) / tau);
  if (mode == 2) return expf(-rate * softplus_f32(x));
  return expf(-expf(x));
}

__device__ __forceinline__ uint32_t raw_bits(float x) { return __float_as_uint(x); }
__device__ __forceinline__ uint32_t raw_bits(bf16_t x) { return x; }
template <typename T>
__device__ __forceinline__ float from_raw(uint32_t x) {
  return sizeof(T) == 2 ? __uint_as_float(x << 16) : __uint_as_float(x);
}

struct ChunkArgs {
  const int32_t *seq_qstart, *seq_qlen, *state_slots;
  int qkv_stride, n_heads, n_kv, vdim, q_col, k_col, v_col, head0;
  float q_scale, unit_eps;
  int decay_mode;
  const float* decay;
  int decay_stride, decay_col;
  const float *decay_p0, *decay_p1;
  float tau;
  const float* beta;
  int beta_stride, beta_col, by_step;
  const float *skip, *bonus;
  float* ws;
};

// what chunk_prepare leaves of a (chunk, head), in floats
template <int D, int KIND>
struct Part {
  static constexpr int Q = 0;                                            // [64][D]
  static constexpr int KE = Q + kTok * D;                                // [D][64]: the keys of the last line, channel first
  static constexpr int B = KE + kTok * D;                                // [64][64]
  static constexpr int DEC = B + kTok * kTok;                            // [D]: the chunk's decays
  static constexpr int K = DEC + D;                                      // [64][D], with the delta rule
  static constexpr int T = K + (KIND & kDelta ? kTok * D : 0);           // [64][64], with the delta rule
  static constexpr int SIZE = T + (KIND & kDelta ? kTok * kTok : 0);
};
// Matrices lie as the walk's products take them: tile (i, m) of 16 x 16, of m0 tiles a row, as lane (row % 16) + 16 (column / 4 %
// 4)'s four columns one lane after the other, so a wave's load of a tile is 1,024 bytes in one piece.
template <int M0>
__device__ __forceinline__ int at(int i, int m, int lane) {
  return ((i * M0 + m) * 64 + lane) * 4;
}
// Chunk c of request seq: its place among the n_tokens / 64 + n_seqs parts.  First chunks by request, the others by the token they start
// at: 64 tokens of the span lie before it, so no two of them start in the same 64 tokens, whatever the order of the spans in the batch.
__device__ __forceinline__ size_t part_of(int seq, int n_seqs, int q0, int c, int n_heads_here, int head_local) {
  return static_cast<size_t>(c == 0 ? seq : n_seqs + q0 / kTok + c - 1) * n_heads_here + head_local;
}

// ------------------------------------------------------------------------------------------- prepare
constexpr int prepare_groups(int dim) { return dim > 128 ? 2 : 1; }
// A workgroup a (chunk, request, head); with 256 key channels two groups of waves divide them.  64 key channels at a time: thread (channel, quarter) holds its channel of 16 tokens in registers
// and makes the running products of decays there, doubling the blocks; the vectors of a block size go to LDS and meet on the
// matrix cores, where a wave owns the diagonal tile of 16 x 16 of its quarter.
// Bound by the issue of instructions (a wave of 128 channels with the delta rule some 7,000, two waves a SIMD) and the matrix cores' float64
// (60 of 84 us in sum): hence two block sizes a product within 16 tokens, the diagonal without one, no meeting there, loads all asked
// for at once, A's and B's triangles from opposite ends, and the logarithm of softplus_f32.  8 requests of 111 to 700 tokens, us: 16 heads of
// 128 x 128, delta rule with decays per channel 138 -> 84; 32 of 64 x 64 with a bonus 80 -> 49; one of 2,048 tokens: 4 of 256 x 512 gated
// 61 -> 33, 16 of 128 x 128 by the delta rule 40 -> 33.
template <typename T, int D, int KIND>
__global__ __launch_bounds__(256 * prepare_groups(D), 2) void chunk_prepare_kernel(const T* __restrict__ qkv, const T* __restrict__ beta_rows, ChunkArgs g) {
  constexpr bool CH = KIND & kChannel, DELTA = KIND & kDelta, FIRST = KIND & kReadFirst;
  constexpr int G = prepare_groups(D);
  static_assert(G == 1 || !DELTA, "only B is summed over the groups");
  using P = Part<D, KIND>;
  __shared__ __attribute__((aligned(16))) float ks_all[G][kTok * kRow], qs_all[G][kTok * kRow];  // later A and B
  __shared__ float dm[CH ? 1 : kTok * (kTok + 1)];                                               // a_(j+1) .. a_t where there is one decay a head
  __shared__ __attribute__((aligned(16))) float mul_k[kTok], mul_q[kTok];
  __shared__ float a_s[kTok], b_s[kTok], total_all[G][4][64];
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / 256), tid = threadIdx.x % 256;
  float *ks = ks_all[group], *qs = qs_all[group];
  float(*total)[64] = total_all[group];
  const int c = blockIdx.x, hl = blockIdx.y, h = g.head0 + hl, seq = blockIdx.z, kvh = h / (g.n_heads / g.n_kv);
  const int q0 = g.seq_qstart[seq], ql = g.seq_qlen[seq];
  if (c * kTok >= ql) return;
  const int n = min(kTok, ql - c * kTok);
  const size_t n0 = static_cast<size_t>(q0) + c * kTok;
  float* part = g.ws + part_of(seq, gridDim.z, q0, c, gridDim.y, hl) * P::SIZE;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), r = lane % 16, lg = lane / 16;

  // the tokens' scalars
  if (threadIdx.x < kTok) {
    const int t = threadIdx.x;
    float a = 1.f, b = DELTA ? 0.f : 1.f;
    if (t < n) {
      const size_t at = n0 + t;
      float step = 1.f;
      if (!CH) {
        step = softplus_f32(g.decay[at * g.decay_stride + g.decay_col + h] + g.decay_p1[h]);
        a = expf(-expf(g.decay_p0[h]) * step);
      }
      if (DELTA) b = 1.f / (1.f + expf(-(beta_rows != nullptr ? to_f32<T>(beta_rows[at * g.beta_stride + g.beta_col + h]) : g.beta[at * g.beta_stride + g.beta_col + h])));
      else if (g.by_step) b = step;
    }
    a_s[t] = a;
    b_s[t] = b;
  }
  // unit norms: four threads a token (in float64: an error here would be one of the token's whole write)
  {
    const int t = tid / 4, s = tid % 4;  // (every group for itself: the same numbers)
    double ssq = 0., ssk = 0.;
    if (g.unit_eps >= 0.f && t < n) {
      const T* row = qkv + (n0 + t) * g.qkv_stride + kvh * D;
#pragma unroll
      for (int i = 8 * s; i < D; i += 32) {
        float x[8], y[8];
        load8(row + g.q_col + i, x);
        load8(row + g.k_col + i, y);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          ssq = fma(static_cast<double>(x[e]), static_cast<double>(x[e]), ssq);
          ssk = fma(static_cast<double>(y[e]), static_cast<double>(y[e]), ssk);
        }
      }
    }
    ssq += __shfl_xor(ssq, 1, 64);
    ssk += __shfl_xor(ssk, 1, 64);
    ssq += __shfl_xor(ssq, 2, 64);
    ssk += __shfl_xor(ssk, 2, 64);
    if (s == 0) {
      mul_q[t] = g.unit_eps >= 0.f ? static_cast<float>(g.q_scale / sqrt(ssq + g.unit_eps)) : g.q_scale;
      mul_k[t] = g.unit_eps >= 0.f ? static_cast<float>(1. / sqrt(ssk + g.unit_eps)) : 1.f;
    }
  }
  __syncthreads();
  if (!CH && threadIdx.x < kTok) {
    double p = 1.;  // (up to 64 factors: each product is rounded once)
    for (int j = threadIdx.x; j >= 0; --j) {
      dm[threadIdx.x * (kTok + 1) + j] = static_cast<float>(p);
      p *= a_s[j];
    }
    for (int x = 0; x < G; ++x) total_all[x][0][threadIdx.x] = static_cast<float>(p);  // a_1 .. a_t
  }
  if (!CH) __syncthreads();
  const float dec_rate = CH && g.decay_mode == 2 ? expf(g.decay_p0[h]) : 1.f;
  const float* dec_bias = g.decay_mode == 2 ? g.decay_p1 : g.decay_p0;

  // with decays per channel: tiles of A and B (near: blocks of 1 and 2, of 4 and 8 within the wave's own diagonal tile), B's diagonal
  f32x4_t near_a[2] = {}, near_b[2] = {}, mid = {}, far_a = {}, far_b = {};
  float diag = 0.f;
  f32x4_t low_a[4] = {}, low_b[4] = {};  // without: the tiles (wave, 0 .. wave) of B and, as many for all waves together, (3 - wave, 0 .. 3 - wave) of A
  // a wave's own rows of LDS, which no other reads before the next meeting: written before this, read behind it
  auto own_rows = [] {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  for (int cb = 64 * group; cb < D; cb += 64 * G) {
    float k[16], q[16];
    const int ch = cb + lane, tok0 = 16 * wave;
    // All of them asked for before the first is used: each under its own condition t < n, as the compiler leaves a load whose value is
    // wanted on one side only, was a wait for each (32 one after the other, two thirds of the kernel's time).
    // Rows by steps from one base (sixteen bases of each kept from one turn to the next went to and from a vector register).
    uint32_t kr[16], qr[16];
    float z[CH ? 16 : 1], bias = 0.f;
    {
      const int first = min(tok0, n - 1);
      const T *k_row = qkv + (n0 + first) * g.qkv_stride + kvh * D + g.k_col + cb, *q_row = k_row + (g.q_col - g.k_col);
      const float* z_row = CH ? g.decay + (n0 + first) * g.decay_stride + g.decay_col + h * D + cb : nullptr;
      int left = n - 1 - first;
      asm volatile("" : "+s"(k_row), "+s"(q_row), "+s"(z_row), "+s"(left));
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        kr[x] = raw_bits(k_row[lane]);
        qr[x] = raw_bits(q_row[lane]);
        if (CH) z[x] = z_row[lane];
        const int step = x < left ? g.qkv_stride : 0;
        k_row += step;
        q_row += step;
        if (CH) z_row += x < left ? g.decay_stride : 0;
      }
    }
    if (CH) bias = dec_bias[h * D + ch];
    f32x4_t km[4], qm[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      km[x] = *reinterpret_cast<const f32x4_t*>(&mul_k[tok0 + 4 * x]);
      qm[x] = *reinterpret_cast<const f32x4_t*>(&mul_q[tok0 + 4 * x]);
    }
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      k[x] = from_raw<T>(kr[x]) * km[x / 4][x % 4];
      q[x] = from_raw<T>(qr[x]) * qm[x / 4][x % 4];
      asm volatile("" : "+v"(k[x]), "+v"(q[x]));
    }
    if (tok0 + 16 > n) {
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        k[x] = tok0 + x < n ? k[x] : 0.f;
        q[x] = tok0 + x < n ? q[x] : 0.f;
      }
    }
    // operands of a tile product: rows of LDS, 16 bytes at 16 m + 4 lg
    auto tile = [&](const float* rows, const float* cols, int i, int j, f32x4_t acc) {
      const float* a = rows + (16 * i + r) * kRow + 4 * lg;
      const float* b = cols + (16 * j + r) * kRow + 4 * lg;
#pragma unroll
      for (int m = 0; m < 4; ++m) acc = mma16(*reinterpret_cast<const f32x4_t*>(a + 16 * m), *reinterpret_cast<const f32x4_t*>(b + 16 * m), acc);
      return acc;
    };
    // Q' and K' of these channels, from qs and ks: a wave's own 16 tokens
    auto write_rows = [&](int first) {
      own_rows();
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int row = (tok0 + r) * kRow + 16 * m + 4 * lg;
        *reinterpret_cast<f32x4_t*>(part + P::Q + at<D / 16>(wave, first / 16 + m, lane)) = *reinterpret_cast<const f32x4_t*>(&qs[row]);
        if (DELTA) *reinterpret_cast<f32x4_t*>(part + P::K + at<D / 16>(wave, first / 16 + m, lane)) = *reinterpret_cast<const f32x4_t*>(&ks[row]);
      }
    };
    // the same in float64, rounded once (B's roundings were half of a read-out's: with these sums in float32 its error at 128 channels
    // was 1.5e-7 of its size); its products leave row lg + 4 i in lane (r, lg), so the rows are handed over in that order
    auto tile64 = [&](const float* rows, const float* cols, int i, int j, f32x4_t acc) {
      const float* a = rows + (16 * i + 4 * (r % 4) + r / 4) * kRow + 4 * lg;
      const float* b = cols + (16 * j + r) * kRow + 4 * lg;
      f64x4_t sum = {0., 0., 0., 0.};
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const f32x4_t x = *reinterpret_cast<const f32x4_t*>(a + 16 * m), y = *reinterpret_cast<const f32x4_t*>(b + 16 * m);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(x[e]), static_cast<double>(y[e]), sum, 0, 0, 0);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += static_cast<float>(sum[e]);
      return acc;
    };
    if (CH) {
      // pre: the decays from the block's first token to this one (or, reading first, to the one before); suf: from the next one
      // to the block's last
      float a[16], pre[16], suf[16];
#pragma unroll
      for (int x = 0; x < 16; ++x) qs[(tok0 + x) * kRow + lane] = z[x];  // (only this thread reads them)
      auto decays = [&](int mode) {
#pragma unroll 4
        for (int x = 0; x < 16; ++x) {
          float* at = qs + (tok0 + x) * kRow + lane;
          *at = decay_of(*at + bias, mode, g.tau, dec_rate);
        }
      };
      if (g.decay_mode == 1) decays(1);
      else if (g.decay_mode == 2) decays(2);
      else decays(3);
#pragma unroll
      for (int x = 0; x < 16; ++x) a[x] = qs[(tok0 + x) * kRow + lane];  // (this thread's own writes)
#pragma unroll
      for (int x = 0; x < 16; ++x) asm volatile("" : "+v"(a[x]));
      if (tok0 + 16 > n) {
#pragma unroll
        for (int x = 0; x < 16; ++x) a[x] = tok0 + x < n ? a[x] : 1.f;
      }
      // the diagonal itself: lane (token, quarter of 16 channels)
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        qs[(tok0 + x) * kRow + lane] = q[x];
        ks[(tok0 + x) * kRow + lane] = FIRST ? k[x] * g.bonus[h * D + ch] : k[x];
      }
      own_rows();
      {
        double sum = 0.;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const int row = (tok0 + r) * kRow + 16 * m + 4 * lg;
          const f32x4_t x = *reinterpret_cast<const f32x4_t*>(&qs[row]), y = *reinterpret_cast<const f32x4_t*>(&ks[row]);
#pragma unroll
          for (int e = 0; e < 4; ++e) sum = fma(static_cast<double>(x[e]), static_cast<double>(y[e]), sum);
        }
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        diag += static_cast<float>(sum);
      }
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        pre[x] = FIRST ? 1.f : a[x];
        suf[x] = 1.f;
      }
      auto twice = [&](int w) {  // blocks twice as long
#pragma unroll
        for (int x = 0; x < 16; ++x)
          if ((x / w) % 2 == 1) {
            const int last = x / (2 * w) * (2 * w) + w - 1;  // of the first half; its whole product
            pre[x] *= FIRST ? pre[last] * a[last] : pre[last];
          }
#pragma unroll
        for (int x = 0; x < 16; ++x)
          if ((x / w) % 2 == 0) {
            const int second = x / (2 * w) * (2 * w) + w;  // the second half's whole product
            suf[x] *= a[second] * (w > 1 ? suf[second] : 1.f);
          }
      };
      // within 16 tokens, where at each size eight are rows and eight columns: two sizes a product, and nobody to meet
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        float rows[16];  // of A
        own_rows();
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const int w = 1 << (2 * half + s);
#pragma unroll
          for (int x = 0; x < 16; ++x) {
            const int place = 8 * s + x / (2 * w) * w + x % w;
            if ((x / w) % 2 == 1) {
              qs[(tok0 + place) * kRow + lane] = q[x] * pre[x];
              rows[place] = DELTA ? k[x] * pre[x] : 0.f;
            } else {
              ks[(tok0 + place) * kRow + lane] = k[x] * suf[x];
            }
          }
          twice(w);
        }
        own_rows();
        near_b[half] = tile64(qs, ks, wave, wave, near_b[half]);
        if (DELTA) {
          own_rows();
#pragma unroll
          for (int x = 0; x < 16; ++x) qs[(tok0 + x) * kRow + lane] = rows[x];
          own_rows();
          near_a[half] += tile(qs, ks, wave, wave, f32x4_t{0.f, 0.f, 0.f, 0.f});
        }
      }
      own_rows();
#pragma unroll
      for (int w = 16; w <= 32; w *= 2) {
        if (w == 16) {
          total[wave][lane] = FIRST ? pre[15] * a[15] : pre[15];
        } else {
          __syncthreads();  // the vectors before have been read
          if (wave == 0) {
            const float m = total[1][lane];
#pragma unroll
            for (int x = 0; x < 16; ++x) suf[x] *= m;
          } else if (wave == 3) {
            const float m = total[2][lane];
#pragma unroll
            for (int x = 0; x < 16; ++x) pre[x] *= m;
          }
        }
        if ((wave / (w / 16)) % 2 == 1) {
#pragma unroll
          for (int x = 0; x < 16; ++x) {
            if (DELTA) ks[(tok0 + x) * kRow + lane] = k[x] * pre[x];
            qs[(tok0 + x) * kRow + lane] = q[x] * pre[x];
          }
        } else {
#pragma unroll
          for (int x = 0; x < 16; ++x) ks[(tok0 + x) * kRow + lane] = k[x] * suf[x];
        }
        __syncthreads();
        if (w == 16) {
          // tiles (1, 0) and (3, 2): of A by waves 0 and 1, of B by waves 2 and 3
          const int i = wave % 2 * 2 + 1;
          if (wave >= 2) mid = tile64(qs, ks, i, i - 1, mid);
          else if (DELTA) mid = tile(ks, ks, i, i - 1, mid);
        } else {
          const int i = 2 + wave / 2, j = wave % 2;
          far_b = tile64(qs, ks, i, j, far_b);
          if (DELTA) far_a = tile(ks, ks, i, j, far_a);
        }
      }
      // the chunk's own products: undo nothing, the quarters' wholes join what a quarter's tokens have
      const float t0 = total[0][lane], t1 = total[1][lane], t2 = total[2][lane], t3 = total[3][lane];
      const float whole = ((t0 * t1) * t2) * t3;
      const float before = wave == 0 ? 1.f : wave == 1 ? t0 : t0 * t1;              // (wave 3's pre holds t2 already)
      const float after = wave == 3 ? 1.f : wave == 2 ? t3 : wave == 1 ? t2 * t3 : t2 * t3;  // (wave 0's suf holds t1 already)
      __syncthreads();
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        qs[(tok0 + x) * kRow + lane] = q[x] * (before * pre[x]);
        if (DELTA) ks[(tok0 + x) * kRow + lane] = k[x] * (before * pre[x]);
      }
      write_rows(cb);
#pragma unroll
      for (int x = 0; x < 16; x += 4) {
        const f32x4_t v = {k[x] * (suf[x] * after), k[x + 1] * (suf[x + 1] * after), k[x + 2] * (suf[x + 2] * after), k[x + 3] * (suf[x + 3] * after)};
        *reinterpret_cast<f32x4_t*>(part + P::KE + at<4>(ch / 16, wave, ch % 16 + 4 * x)) = v;
      }
      if (wave == 0) part[P::DEC + ch] = whole;
    } else {
      own_rows();
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        qs[(tok0 + x) * kRow + lane] = q[x];
        ks[(tok0 + x) * kRow + lane] = k[x];
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j <= wave) low_b[j] = tile64(qs, ks, wave, j, low_b[j]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (DELTA && j <= 3 - wave) low_a[j] = tile(ks, ks, 3 - wave, j, low_a[j]);
      __syncthreads();
#pragma unroll
      for (int x = 0; x < 16; ++x) {
        const float m = total[0][tok0 + x];
        qs[(tok0 + x) * kRow + lane] = q[x] * m;
        if (DELTA) ks[(tok0 + x) * kRow + lane] = k[x] * m;
      }
      write_rows(cb);
#pragma unroll
      for (int x = 0; x < 16; x += 4) {
        f32x4_t v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = k[x + e] * (dm[63 * (kTok + 1) + tok0 + x + e] * (DELTA ? 1.f : b_s[tok0 + x + e]));
        *reinterpret_cast<f32x4_t*>(part + P::KE + at<4>(ch / 16, wave, ch % 16 + 4 * x)) = v;
      }
      if (wave == 0) part[P::DEC + ch] = total[0][63];
    }
  }
  __syncthreads();
  // A and B whole, in LDS: A in ks, B in qs (rows of kRow), zeros above their diagonals
  for (int i = tid; i < kTok * kRow; i += 256) ks[i] = qs[i] = 0.f;
  __syncthreads();
  auto put = [&](float* m, int i, int j, const f32x4_t& v, bool diagonal) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = 16 * i + 4 * lg + e, at = 16 * j + r;
      if (at < t || (diagonal && at == t)) m[t * kRow + at] = v[e];
    }
  };
  if (CH) {
    const int tok16 = 16 * wave;
    if (lg == 0) qs[(tok16 + r) * kRow + tok16 + r] = diag;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int e = 0; e < 4; ++e) {  // place 4 lg + e of the rows, r of the columns (see above)
        const int size = 2 * half + (r >= 8), w = 1 << size, row = (4 * lg + e) % 8, col = r % 8;
        const int at = (tok16 + (row >> size << (size + 1)) + w + row % w) * kRow + tok16 + (col >> size << (size + 1)) + col % w;
        if ((4 * lg + e >= 8) == (r >= 8) && row >> size == col >> size) {
          qs[at] = near_b[half][e];
          if (DELTA) ks[at] = near_a[half][e];
        }
      }
    const int i = wave % 2 * 2 + 1;
    if (wave >= 2) put(qs, i, i - 1, mid, true);
    else if (DELTA) put(ks, i, i - 1, mid, false);
    put(qs, 2 + wave / 2, wave % 2, far_b, true);
    if (DELTA) put(ks, 2 + wave / 2, wave % 2, far_a, false);
  } else {
    const float skip = g.skip != nullptr ? g.skip[h] : 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j <= wave) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = 16 * wave + 4 * lg + e, at = 16 * j + r;
          const float d = at <= t ? dm[t * (kTok + 1) + at] : 0.f;
          low_b[j][e] *= DELTA ? d : d * b_s[at];
          if (at == t && group == 0) low_b[j][e] += skip;
        }
        put(qs, wave, j, low_b[j], true);
      }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (DELTA && j <= 3 - wave) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = 16 * (3 - wave) + 4 * lg + e, at = 16 * j + r;
          low_a[j][e] *= at <= t ? dm[t * (kTok + 1) + at] : 0.f;
        }
        put(ks, 3 - wave, j, low_a[j], false);
      }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kTok * kTok / 4; i += 256 * G) {
    const int row = (i / 256 * 16 + i % 16) * kRow + i / 64 % 4 * 16 + i / 16 % 4 * 4;  // (see at)
    f32x4_t v = *reinterpret_cast<const f32x4_t*>(&qs_all[0][row]);
    if (G > 1) v += *reinterpret_cast<const f32x4_t*>(&qs_all[G - 1][row]);
    *reinterpret_cast<f32x4_t*>(part + P::B + 4 * i) = v;
  }
  if (!DELTA) return;
  // T = (I + diag(beta) A)^-1 diag(beta) in blocks of 16 x 16.  On the diagonal a wave solves its block, a column a lane: x_t =
  // (1 where t is the column) - beta_t (sum over j < t of A[t][j] x_j); below it, block by block away from the diagonal,
  // X_ij = -X_ii (sum over j <= k < i of beta A_ik X_kj).  X goes to qs (B has been written), with beta's rows in A.
  __syncthreads();
  for (int i = threadIdx.x; i < kTok * kTok / 4; i += 256) {
    f32x4_t* at = reinterpret_cast<f32x4_t*>(&ks[i / 16 * kRow + i % 16 * 4]);
    *at *= b_s[i / 16];
    *reinterpret_cast<f32x4_t*>(&qs[i / 16 * kRow + i % 16 * 4]) = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  __syncthreads();
  {
    const float* m = ks + 16 * wave * kRow + 16 * wave;
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float s[2] = {t == r ? 1.f : 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < t; ++j) s[j % 2] = fmaf(-m[t * kRow + j], x[j], s[j % 2]);
      x[t] = s[0] + s[1];
      if (lg == 0) qs[(16 * wave + t) * kRow + 16 * wave + r] = x[t];
    }
  }
  // (second operand of a product as rows of X: element 16 k + 4 lg + e of column 16 j + r)
  auto column = [&](const float* m, int k, int j) {
    f32x4_t v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = m[(16 * k + 4 * lg + e) * kRow + 16 * j + r];
    return v;
  };
#pragma unroll
  for (int away = 1; away < 4; ++away) {
    __syncthreads();
    const int j = wave, i = wave + away;
    if (i < 4) {
      f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
      for (int k = j; k < i; ++k) sum = mma16(*reinterpret_cast<const f32x4_t*>(&ks[(16 * i + r) * kRow + 16 * k + 4 * lg]), column(qs, k, j), sum);
      // (a product's result, lane (r, lg) with rows 4 lg .. of column r, is the second operand of the next as it stands)
      const f32x4_t x = triangle16(*reinterpret_cast<const f32x4_t*>(&qs[(16 * i + r) * kRow + 16 * i + 4 * lg]), sum, f32x4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int e = 0; e < 4; ++e) qs[(16 * i + 4 * lg + e) * kRow + 16 * j + r] = -x[e];
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kTok * kTok / 4; i += 256) {
    const int col = i / 64 % 4 * 16 + i / 16 % 4 * 4;
    f32x4_t v = *reinterpret_cast<const f32x4_t*>(&qs[(i / 256 * 16 + i % 16) * kRow + col]);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] *= b_s[col + e];
    *reinterpret_cast<f32x4_t*>(part + P::T + 4 * i) = v;
  }
}

// ---------------------------------------------------------------------------------------------- walk
// A workgroup of eight waves a (head, 16 columns of S, request).  Four of them carry S on: a wave owns a quarter of its rows, as the
// products that update it leave them (lane (r, g): rows 4g .. 4g + 3 of a tile of 16, column r), which is also how the other products take
// S, v and u as their second operand; through LDS every wave gets all of them.  The other four make the read-outs, 16 tokens each, of S
// and u in LDS while the first are at the update (a wave of each kind a SIMD; the waves with the most tiles up to the diagonal of T and of
// B are not neighbours).
template <typename T, int D, int KIND>
__global__ __launch_bounds__(512, 2) void chunk_walk_kernel(const T* __restrict__ qkv, float* __restrict__ state, float* __restrict__ out, ChunkArgs g) {
  constexpr bool DELTA = KIND & kDelta;
  constexpr int M = D / 16, MT = D / 64;
  using P = Part<D, KIND>;
  // (two of what a chunk's read-outs may still read while the next chunk's is written)
  __shared__ __attribute__((aligned(16))) f32x4_t s_lds[2][M][64], x_lds[DELTA ? 4 : 1][64], u_lds[2][4][64];
  const int hl = blockIdx.x, h = g.head0 + hl, col0 = 16 * blockIdx.y, seq = blockIdx.z, vdim = g.vdim;
  const int q0 = g.seq_qstart[seq], ql = g.seq_qlen[seq], chunks = (ql + kTok - 1) / kTok;
  if (ql <= 0) return;  // (a request without tokens leaves its memory alone: its slot may be another's by now)
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), r = lane % 16, lg = lane / 16;
  // (the last chunk asks for itself once more, unread)
  auto part = [&](int c) {
    return __builtin_amdgcn_make_buffer_rsrc(g.ws + part_of(seq, gridDim.z, q0, min(c, chunks - 1), gridDim.x, hl) * P::SIZE, 0, P::SIZE * 4, 0x00027000);
  };
  // (a scalar base and place: addresses of their own would take the registers that the loads on their way need)
  using Source = __amdgpu_buffer_rsrc_t;
  auto piece = [](Source p, int lane_bytes, int at) {
    return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(p, lane_bytes, 4 * at, 0));
  };
  auto lower = [&](int row, const f32x4_t* a, const f32x4_t* b, f32x4_t c) {
    return row == 0 ? lower_row<0>(a, b, c) : row == 1 ? lower_row<1>(a, b, c) : row == 2 ? lower_row<2>(a, b, c) : lower_row<3>(a, b, c);
  };

  if (wave >= 4) {
    const int tile = 7 - wave;
    f32x4_t q[M], b[4];
    auto ask_q = [&](Source p, int m) {
#pragma unroll
      for (int x = 0; x < 4; ++x) q[m + x] = piece(p, 16 * lane, P::Q + at<M>(tile, m + x, 0));
    };
    auto ask_b = [&](Source p) {
#pragma unroll
      for (int m = 0; m < 4; ++m) b[m] = piece(p, 16 * lane, P::B + at<4>(tile, m, 0));
    };
#pragma unroll
    for (int m = 0; m < M; m += 4) ask_q(part(0), m);
    ask_b(part(0));
    for (int c = 0; c < chunks; ++c) {
      const Source next = part(c + 1);
      __syncthreads();  // S is in LDS (and u, where it is v)
      f32x4_t o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < M; m += 4) {
        if (DELTA && m == M / 2) __syncthreads();  // (the writers': v - K' S is in LDS)
        f32x4_t s4[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) s4[x] = s_lds[c % 2][m + x][lane];
        o += mma64(&q[m], s4);
        ask_q(next, m);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (DELTA && M == 4) __syncthreads();
      if (DELTA) __syncthreads();  // u is in LDS
      f32x4_t u[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) u[m] = u_lds[c % 2][m][lane];
      o = lower(tile, b, u, o);
      ask_b(next);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = c * kTok + 16 * tile + 4 * lg + i;
        if (t < ql) out[(static_cast<size_t>(q0 + t) * g.n_heads + h) * vdim + col0 + r] = o[i];
      }
    }
    return;
  }

  float* S_head = state + (static_cast<size_t>(g.state_slots[seq]) * g.n_heads + h) * D * vdim + col0 + r;
  f32x4_t S[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) S[m][i] = S_head[static_cast<size_t>(16 * (wave * MT + m) + 4 * lg + i) * vdim];

  // (waited for here: a load from before the loop that may still be on its way inside it makes every turn wait for its own)
  __builtin_amdgcn_s_waitcnt(0);

  f32x4_t k[DELTA ? M : 1], ke[MT][4], tm[DELTA ? 4 : 1], dec[MT];
  uint32_t raw_v[4];  // (as they lie there: a conversion where they are asked for would wait for them)
  auto ask_k = [&](Source p, int m) {
#pragma unroll
    for (int x = 0; x < 4; ++x) k[m + x] = piece(p, 16 * lane, P::K + at<M>(wave, m + x, 0));
  };
  auto ask_v = [&](int c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = c * kTok + 16 * wave + 4 * lg + i;
      raw_v[i] = raw_bits(qkv[static_cast<size_t>(q0 + min(t, ql - 1)) * g.qkv_stride + g.v_col + h * vdim + col0 + r]);
    }
  };
  auto ask_t = [&](Source p) {
    if (DELTA) {
#pragma unroll
      for (int m = 0; m < 4; ++m) tm[m] = piece(p, 16 * lane, P::T + at<4>(wave, m, 0));
    }
  };
  auto ask_ke = [&](Source p, int m) {
    dec[m] = piece(p, 16 * lg, P::DEC + 16 * (wave * MT + m));
#pragma unroll
    for (int x = 0; x < 4; ++x) ke[m][x] = piece(p, 16 * lane, P::KE + at<4>(wave * MT + m, x, 0));
  };
  if (DELTA) {
#pragma unroll
    for (int m = 0; m < M; m += 4) ask_k(part(0), m);
  }
  ask_v(0);
  ask_t(part(0));
#pragma unroll
  for (int m = 0; m < MT; ++m) ask_ke(part(0), m);
  auto turn = [&](int c, auto last) {
    const Source next = part(c + 1);
#pragma unroll
    for (int m = 0; m < MT; ++m) s_lds[c % 2][wave * MT + m][lane] = S[m];
    f32x4_t v;
    auto take_v = [&] {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = c * kTok + 16 * wave + 4 * lg + i < ql ? from_raw<T>(raw_v[i]) : 0.f;
      ask_v(min(c + 1, chunks - 1));
    };
    if (!DELTA) {
      take_v();
      u_lds[c % 2][wave][lane] = v;
    }
    __syncthreads();
    if (DELTA) {
      f32x4_t p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < M; m += 4) {
        f32x4_t s4[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) s4[x] = s_lds[c % 2][m + x][lane];
        p += mma64(&k[m], s4);
        ask_k(next, m);
        __builtin_amdgcn_sched_barrier(0);
      }
      take_v();
      x_lds[wave][lane] = v - p;
      __syncthreads();
      f32x4_t x4[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) x4[m] = x_lds[m][lane];
      u_lds[c % 2][wave][lane] = lower(wave, tm, x4, f32x4_t{0.f, 0.f, 0.f, 0.f});
      ask_t(next);
      __syncthreads();
    }
    f32x4_t u[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) u[m] = u_lds[c % 2][m][lane];
    if (!decltype(last)::value) {
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const f32x4_t sum = mma64(ke[m], u);
#pragma unroll
        for (int i = 0; i < 4; ++i) S[m][i] = fmaf(S[m][i], dec[m][i], sum[i]);
        ask_ke(next, m);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // the memory that is kept: in float64, rounded once.  Its last tokens weigh the most and 64 products in float32 round them oftener than
      // the walk does: time mixing 0.57e-7 -> 0.40e-7 of its size (walked 0.44e-7), delta rule 1.00e-7 -> 0.85e-7 (0.83e-7).  A product in
      // float64 leaves row lg + 4 i in lane (r, lg), so the keys' rows are handed over in that order.
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        f64x4_t sum;
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] = static_cast<double>(S[m][i]) * static_cast<double>(dec[m][i]);
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            sum = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(__shfl(ke[m][x][e], 4 * (r % 4) + r / 4 + 16 * lg, 64)),
                                                       static_cast<double>(u[x][e]), sum, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) S[m][i] = static_cast<float>(sum[i]);
      }
    }
  };
  for (int c = 0; c + 1 < chunks; ++c) turn(c, std::false_type{});
  turn(chunks - 1, std::true_type{});
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) S_head[static_cast<size_t>(16 * (wave * MT + m) + 4 * lg + i) * vdim] = S[m][i];
}

template <typename T, int D, int KIND>
int launch(const T* qkv, const T* beta_rows, float* state, float* out, ChunkArgs g, int n_seqs, int n_tokens, int max_qlen, size_t ws_floats,
           hipStream_t stream) {
  // as many heads at a time as the workspace holds
  const size_t a_head = (static_cast<size_t>(n_tokens / kTok) + n_seqs) * Part<D, KIND>::SIZE;
  const int heads = static_cast<int>(std::min<size_t>(g.n_heads, ws_floats / a_head));
  YK_REQUIRE(heads > 0, "state_scan_chunks: the workspace is too small");
  for (g.head0 = 0; g.head0 < g.n_heads; g.head0 += heads) {
    const int here = std::min(heads, g.n_heads - g.head0);
    chunk_prepare_kernel<T, D, KIND><<<dim3((max_qlen + kTok - 1) / kTok, here, n_seqs), 256 * prepare_groups(D), 0, stream>>>(qkv, beta_rows, g);
    if (yk_check_launch("chunk_prepare")) return -1;
    chunk_walk_kernel<T, D, KIND><<<dim3(here, g.vdim / 16, n_seqs), 512, 0, stream>>>(qkv, state, out, g);
    if (yk_check_launch("chunk_walk")) return -1;
  }
  return 0;
}

// the kinds of a decay, write and read-out that state_scan.hip's fast form has
int kind_of(int decay_mode, int write_mode, int with_bonus) {
  return (decay_mode >= 1 && decay_mode <= 3 ? kChannel : 0) + (write_mode == 1 ? kDelta : 0) + (with_bonus ? kReadFirst : 0);
}

}  // namespace

// Floats of workspace for one head (0: sizes or a kind that the chunked form is not built for); the more heads fit in
// what the caller gives, the fewer launches.
extern "C" size_t yk_state_scan_chunks_floats(int n_tokens, int n_seqs, int dim, int vdim, int decay_mode, int write_mode, int with_bonus, int with_skip) {
  const int kind = kind_of(decay_mode, write_mode, with_bonus);
  if ((dim != 64 && dim != 128 && dim != 256) || vdim % 16 != 0 || decay_mode < 0 || decay_mode > 3 || kind == kReadFirst || (with_skip && kind != 0) ||
      kind > (kChannel | kReadFirst) || (dim == 256 && (kind & kDelta)))  // (the delta rule's operands of 256 channels do not fit in registers)
    return 0;
  const size_t delta = kind & kDelta ? 1 : 0;
  return (static_cast<size_t>(n_tokens / kTok) + n_seqs) * ((2 + delta) * kTok * dim + dim + (1 + delta) * kTok * kTok);
}

// yk_linear_state_scan's arguments (see there), for rows whose queries and keys start at multiples of 16 bytes; max_qlen: the
// longest span.
extern "C" int yk_state_scan_chunks(const void* qkv, int qkv_stride, int dtype, int n_heads, int n_kv, int dim, int vdim, float* state,
                                    const int32_t* seq_qstart, const int32_t* seq_qlen, const int32_t* state_slots, int n_seqs, int n_tokens,
                                    int max_qlen, float q_scale, float unit_eps, int decay_mode, const float* decay, int decay_stride, int decay_col,
                                    const float* decay_p0, const float* decay_p1, float tau, const float* beta, int beta_stride, int beta_col,
                                    float* out, int q_col, int k_col, int v_col, int write_mode, const float* skip, const void* beta_rows,
                                    const float* bonus, float* workspace, size_t workspace_floats, hipStream_t stream) {
  YK_REQUIRE(n_seqs >= 0 && n_heads > 0 && n_kv > 0 && n_heads % n_kv == 0 && dim > 0 && vdim > 0 && max_qlen >= 0, "state_scan_chunks: bad sizes");
  YK_REQUIRE(q_col >= 0 && k_col >= 0 && v_col >= 0 && qkv_stride >= std::max(std::max(q_col, k_col) + n_kv * dim, v_col + n_heads * vdim),
             "state_scan_chunks: rows shorter than q, k and v");
  YK_REQUIRE(write_mode == 0 || (write_mode == 1 && (beta != nullptr || beta_rows != nullptr)) || (write_mode == 2 && decay_mode == 0),
             "state_scan_chunks: the delta rule needs beta, a write by the step the decay per head");
  YK_REQUIRE(bonus == nullptr || (write_mode == 0 && skip == nullptr), "state_scan_chunks: a bonus goes with plain writes and no skip");
  YK_REQUIRE(yk_state_scan_chunks_floats(n_tokens, n_seqs, dim, vdim, decay_mode, write_mode, bonus != nullptr, skip != nullptr) > 0 || n_seqs == 0,
             "state_scan_chunks: sizes or a kind it is not built for");
  YK_REQUIRE(decay != nullptr && decay_p0 != nullptr && (decay_mode == 1 || decay_mode == 3 || decay_p1 != nullptr), "state_scan_chunks: the decay's inputs are missing");
  YK_REQUIRE(decay_mode != 1 || tau > 0.f, "state_scan_chunks: tau must be positive");
  YK_REQUIRE(qkv_stride % 8 == 0 && q_col % 8 == 0 && k_col % 8 == 0 && reinterpret_cast<uintptr_t>(qkv) % 16 == 0,
             "state_scan_chunks: the rows of queries and keys must be 16-byte aligned");
  YK_REQUIRE(workspace != nullptr && reinterpret_cast<uintptr_t>(workspace) % 16 == 0, "state_scan_chunks: the workspace must be 16-byte aligned");
  YK_REQUIRE(n_seqs <= 65535 && n_heads <= 65535 && vdim / 16 <= 65535, "state_scan_chunks: too many requests or heads for one launch");
  if (n_seqs == 0 || max_qlen == 0) return 0;
  const ChunkArgs g{seq_qstart, seq_qlen, state_slots, qkv_stride, n_heads, n_kv, vdim, q_col, k_col, v_col, 0, q_scale, unit_eps, decay_mode, decay,
                    decay_stride, decay_col, decay_p0, decay_p1, tau, beta, beta_stride, beta_col, write_mode == 2, skip, bonus, workspace};
#define YK_CASE(T, DIM, KIND)                                                                                                      \
  if (dim == DIM && kind == KIND)                                                                                                  \
    return launch<T, DIM, KIND>(static_cast<const T*>(qkv), static_cast<const T*>(beta_rows), state, out, g, n_seqs, n_tokens, max_qlen, \
                                workspace_floats, stream);
#define YK_KINDS(T, DIM) YK_CASE(T, DIM, 0) YK_CASE(T, DIM, 1) YK_CASE(T, DIM, 2) YK_CASE(T, DIM, 3) YK_CASE(T, DIM, 5)
  const int kind = kind_of(decay_mode, write_mode, bonus != nullptr);
  if (dtype == YK_BF16) {
    YK_KINDS(bf16_t, 64)
    YK_KINDS(bf16_t, 128)
    YK_CASE(bf16_t, 256, 0) YK_CASE(bf16_t, 256, 1) YK_CASE(bf16_t, 256, 5)
  }
  if (dtype == YK_F32) {
    YK_KINDS(float, 64)
    YK_KINDS(float, 128)
    YK_CASE(float, 256, 0) YK_CASE(float, 256, 1) YK_CASE(float, 256, 5)
  }
#undef YK_KINDS
#undef YK_CASE
  return yk_fail("state_scan_chunks: unsupported dtype");
}
