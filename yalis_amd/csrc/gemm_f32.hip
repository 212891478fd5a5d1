// Products y[M, N] = x[M, K] . w[N, K]^T with float32 arithmetic on the matrix cores
// (v_mfma_f32_32x32x2_f32 and v_mfma_f32_16x16x4_f32: float32 inputs, products and sums, no
// narrower mode), for operands whose rows can be read four elements at a time.  gemm_fma in
// gemm.hip takes what these do not: K or strides that are no multiple of four, unaligned rows.  Of more than 32 rows, all float32,
// most are made by gemm_split.hip instead (its rule has both sides' times).
//
// As there, every 16 products along K are summed on their own and then added to the running sum:
// a sum of K terms carries the rounding of about sqrt(K / 16) + 4 additions instead of sqrt(K).
#include <algorithm>

#include <type_traits>

#include "common.h"

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// four elements of a row as float32
__device__ __forceinline__ f32x4_t load4(const float* p) { return *reinterpret_cast<const f32x4_t*>(p); }
__device__ __forceinline__ f32x4_t load4(const bf16_t* p) {
  const u32x2_t u = *reinterpret_cast<const u32x2_t*>(p);
  return f32x4_t{__uint_as_float(u[0] << 16), __uint_as_float(u[0] & 0xffff0000u), __uint_as_float(u[1] << 16),
                 __uint_as_float(u[1] & 0xffff0000u)};
}
// the same of a weight, which is read once
__device__ __forceinline__ f32x4_t stream4(const float* p) { return __builtin_nontemporal_load(reinterpret_cast<const f32x4_t*>(p)); }
__device__ __forceinline__ f32x4_t stream4(const bf16_t* p) {
  const u32x2_t u = __builtin_nontemporal_load(reinterpret_cast<const u32x2_t*>(p));
  return f32x4_t{__uint_as_float(u[0] << 16), __uint_as_float(u[0] & 0xffff0000u), __uint_as_float(u[1] << 16),
                 __uint_as_float(u[1] & 0xffff0000u)};
}

// ------------------------------------------------------------------------------- tiles, many rows
// A workgroup makes a tile of 64 x 64 outputs with KS groups of 2 x 2 waves, a wave one product of
// 32 x 32; the groups share K (their sums meet in LDS at the end, in their order), so that a product
// with few tiles still has several waves a SIMD to hide its loads behind.  A group walks its part of
// K 32 at a time through two LDS buffers, the next step's rows in flight in registers while the matrix
// cores work: one barrier a step.  Rows are 36 floats apart in LDS, which spreads the 16-byte reads of
// 16 neighbouring lanes over all banks.  Lane l of a wave reads elements 8j + 4 (l / 32) .. + 3 of row
// l % 32 and feeds them to four products one after another, so every LDS read is 16 bytes wide; both
// operands take K in that same order.
// Bound by the matrix cores (256 flops a clock and compute unit in float32).
constexpr int BT = 64;
constexpr int BK = 32;
constexpr int ROW = BK + 4;

template <typename TX, typename TW, typename TO, int KS>
__global__ __launch_bounds__(256 * KS) void gemm_f32_tile_kernel(const TX* __restrict__ x, const TW* __restrict__ w,
                                                                 TO* __restrict__ y, int M, int N, int K, int ldx, int ldw,
                                                                 int ldy) {
  __shared__ __attribute__((aligned(16))) float staged[KS][2][2][BT * ROW];  // group, buffer, operand
  const int m0 = blockIdx.y * BT, n0 = blockIdx.x * BT;
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / 256), tid = threadIdx.x % 256;
  const int lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wm = wave / 2 * 32, wn = wave % 2 * 32;
  const int lr = tid / 8, lk = tid % 8 * 4;  // this thread's row (of 32) and place in a staged step
  const TX* xp[2];
  const TW* wp[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    xp[i] = x + static_cast<size_t>(min(m0 + lr + 32 * i, M - 1)) * ldx;
    wp[i] = w + static_cast<size_t>(min(n0 + lr + 32 * i, N - 1)) * ldw;
  }
  f32x4_t xr[2], wr[2];
  auto fetch = [&](int k0) {
    const int k = k0 + lk;
    const bool in = k < K;  // K is a multiple of four: four elements are all inside or all outside
    const f32x4_t none = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      xr[i] = in ? load4(xp[i] + k) : none;
      wr[i] = in ? load4(wp[i] + k) : none;
    }
  };
  auto park = [&](int buf) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      *reinterpret_cast<f32x4_t*>(&staged[group][buf][0][(lr + 32 * i) * ROW + lk]) = xr[i];
      *reinterpret_cast<f32x4_t*>(&staged[group][buf][1][(lr + 32 * i) * ROW + lk]) = wr[i];
    }
  };
  f32x16_t acc = {};
  const int at = lane % 32 * ROW + lane / 32 * 4;
  // every group takes as many steps (the barriers are the workgroup's); steps beyond K meet zeros
  const int steps = ((K + BK - 1) / BK + KS - 1) / KS, first = group * steps;
  fetch(first * BK);
  park(0);
  for (int s = 0; s < steps; ++s) {
    if (s + 1 < steps) fetch((first + s + 1) * BK);
    __syncthreads();  // step s is parked, and every wave is done with step s - 1, whose buffer is written below
    const float* xb = &staged[group][s & 1][0][wm * ROW + at];
    const float* wb = &staged[group][s & 1][1][wn * ROW + at];
#pragma unroll
    for (int h = 0; h < BK; h += 16) {
      f32x16_t part = {};
#pragma unroll
      for (int kb = h; kb < h + 16; kb += 8) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(xb + kb);
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(wb + kb);
#pragma unroll
        for (int e = 0; e < 4; ++e) part = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], part, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] += part[r];
    }
    if (s + 1 < steps) park((s + 1) & 1);
  }
  {
    // a group's sums go into its own buffers (64 x 64 floats of the 4 x 64 x 36 there), lane by lane
    __syncthreads();
    float* mine = &staged[group][0][0][0];
    if (group > 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) mine[r * 256 + tid] = acc[r];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 1; g < KS; ++g)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] += (&staged[g][0][0][0])[r * 256 + tid];
  }
  // lane l holds outputs [8 (r / 4) + 4 (l / 32) + r % 4][l % 32] of its wave's product
  const int n = n0 + wn + lane % 32;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = m0 + wm + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
    if (m < M && n < N) y[static_cast<size_t>(m) * ldy + n] = from_f32<TO>(acc[r]);
  }
}

// ------------------------------------------------------------------------- one to four rows, no tile
// A wave makes R outputs for every row of x: its lanes read the weight's rows 1 KiB at a time (256
// consecutive elements), eight loads in flight, and every lane sums its own products in four chains a
// row (one of the four elements each) that meet at the end.  A row of the weight is one wave's, so that
// a matrix of 2,000 rows still occupies every compute unit, which tiles of 16 rows do not.
// Bound by the reading of the weight.
template <typename TX, typename TW, typename TO, int MR, int R>
__global__ __launch_bounds__(256) void gemm_f32_dot_kernel(const TX* __restrict__ x, const TW* __restrict__ w, TO* __restrict__ y,
                                                           int N, int K, int ldx, int ldw, int ldy) {
  constexpr int AHEAD = 8 / R;  // pieces of a row in flight
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int n0 = (blockIdx.x * 4 + wave) * R;
  if (n0 >= N) return;
  const TW* wp[R];
#pragma unroll
  for (int i = 0; i < R; ++i) wp[i] = w + static_cast<size_t>(min(n0 + i, N - 1)) * ldw + 4 * lane;
  const TX* xp = x + 4 * lane;
  f32x4_t acc[R][MR] = {};
  auto add = [&](const f32x4_t (&a)[R], const f32x4_t (&b)[MR]) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][m][e] = fmaf(a[i][e], b[m][e], acc[i][m][e]);
  };
  int k0 = 0;
  // What is left of a row is asked for by four and two pieces at once too, or a wave waits for each (2 rows, bfloat16 x,
  // N 4,096, K 1,536 8.4 -> 6.7 us, 4 rows, N 2,048 9.2 -> 5.4; two float32 rows are faster than tiles without that); and with three rows (float32 weights) and four, whose sums
  // take long enough, x beside the weight (4 rows, bfloat16 x, 4,096 x 4,096 18.1 -> 15.1; with fewer that only costs registers).
  constexpr bool X_AHEAD = MR == 4 || (MR == 3 && sizeof(TW) == 4);
  auto pieces = [&](auto count) {
    constexpr int P = decltype(count)::value;
    f32x4_t a[P][R], b[P][MR];
#pragma unroll
    for (int c = 0; c < P; ++c)
#pragma unroll
      for (int i = 0; i < R; ++i) a[c][i] = stream4(wp[i] + k0 + 256 * c);
#pragma unroll
    for (int c = 0; c < P; ++c)
#pragma unroll
      for (int m = 0; m < MR; ++m) b[c][m] = load4(xp + static_cast<size_t>(m) * ldx + k0 + 256 * c);
#pragma unroll
    for (int c = 0; c < P; ++c) add(a[c], b[c]);
    k0 += 256 * P;
  };
  if constexpr (X_AHEAD) {
    while (k0 + 256 * AHEAD <= K) pieces(std::integral_constant<int, AHEAD>());
  } else {
    for (; k0 + 256 * AHEAD <= K; k0 += 256 * AHEAD) {
      f32x4_t a[AHEAD][R];
#pragma unroll
      for (int c = 0; c < AHEAD; ++c)
#pragma unroll
        for (int i = 0; i < R; ++i) a[c][i] = stream4(wp[i] + k0 + 256 * c);
#pragma unroll
      for (int c = 0; c < AHEAD; ++c) {
        f32x4_t b[MR];
#pragma unroll
        for (int m = 0; m < MR; ++m) b[m] = load4(xp + static_cast<size_t>(m) * ldx + k0 + 256 * c);
        add(a[c], b);
      }
    }
  }
  if constexpr (MR > 2 || (MR == 2 && sizeof(TX) + sizeof(TW) < 8)) {
    if (AHEAD > 4 && k0 + 1024 <= K) pieces(std::integral_constant<int, 4>());
    if (k0 + 512 <= K) pieces(std::integral_constant<int, 2>());
  }
  for (; k0 < K; k0 += 256) {
    const bool in = k0 + 4 * lane < K;  // K is a multiple of four
    const f32x4_t none = {0.f, 0.f, 0.f, 0.f};
    f32x4_t a[R], b[MR];
#pragma unroll
    for (int i = 0; i < R; ++i) a[i] = in ? stream4(wp[i] + k0) : none;
#pragma unroll
    for (int m = 0; m < MR; ++m) b[m] = in ? load4(xp + static_cast<size_t>(m) * ldx + k0) : none;
    add(a, b);
  }
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int m = 0; m < MR; ++m) {
      const float v = wave_sum((acc[i][m][0] + acc[i][m][1]) + (acc[i][m][2] + acc[i][m][3]));
      if (lane == 0 && n0 + i < N) y[static_cast<size_t>(m) * ldy + n0 + i] = from_f32<TO>(v);
    }
}

// ------------------------------------------------------------------------------ few rows, one pass
// A workgroup of W waves makes 16 outputs for up to 16 MT rows of x (blockIdx.y: which of them); its
// waves walk K by turns, 64 elements each, and their sums meet in LDS at the end, wave by wave.  A
// wave's load covers 16 rows x 64 consecutive bytes of the weight, four of them in flight; many waves a
// compute unit keep the memory busy, so nothing is staged.  The rows of x come from the caches.
// Bound by the reading of the weight.
template <typename TX, typename TW, typename TO, int MT, int W>
__global__ __launch_bounds__(64 * W) void gemm_f32_rows_kernel(const TX* __restrict__ x, const TW* __restrict__ w,
                                                               TO* __restrict__ y, int M, int N, int K, int ldx, int ldw,
                                                               int ldy) {
  __shared__ float sums[W][MT][16][17];
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int r = lane % 16, g = lane / 16;
  const TW* wp = w + static_cast<size_t>(min(n0 + r, N - 1)) * ldw + 4 * g;
  const TX* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xp[t] = x + static_cast<size_t>(min(m0 + 16 * t + r, M - 1)) * ldx + 4 * g;
  f32x4_t acc[MT] = {};
  auto sixteen = [&](const f32x4_t& a, const f32x4_t (&b)[MT]) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      f32x4_t part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e) part = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[t][e], part, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[t][i] += part[i];
    }
  };
  int k0 = wave * 64;
  for (; k0 + 64 <= K; k0 += W * 64) {
    f32x4_t a[4], b[4][MT];
#pragma unroll
    for (int c = 0; c < 4; ++c) a[c] = stream4(wp + k0 + 16 * c);
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int t = 0; t < MT; ++t) b[c][t] = load4(xp[t] + k0 + 16 * c);
#pragma unroll
    for (int c = 0; c < 4; ++c) sixteen(a[c], b[c]);
  }
  for (int k = k0; k < K && k < k0 + 64; k += 16) {  // the last, short piece of K: one wave's
    const bool in = k + 4 * g < K;  // K is a multiple of four
    const f32x4_t none = {0.f, 0.f, 0.f, 0.f};
    const f32x4_t a = in ? load4(wp + k) : none;
    f32x4_t b[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) b[t] = in ? load4(xp[t] + k) : none;
    sixteen(a, b);
  }
  // lane l holds outputs 4 (l / 16) .. + 3 of row l % 16
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[wave][t][r][4 * g + i] = acc[t][i];
  __syncthreads();
  for (int o = threadIdx.x; o < MT * 256; o += 64 * W) {
    const int t = o / 256, row = o / 16 % 16, col = o % 16;
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < W; ++v) s += sums[v][t][row][col];
    const int m = m0 + 16 * t + row, n = n0 + col;
    if (m < M && n < N) y[static_cast<size_t>(m) * ldy + n] = from_f32<TO>(s);
  }
}

// Which form.  Up to 32 rows of x every weight is read once and the few-row form runs at the memory's rate; beyond, its
// reading of x through the caches holds it at 50 TFLOP/s, where tiles reach 110, so tiles win as soon as there are about
// a hundred of them.  Four groups of waves a tile while the tiles are no more than the 256 compute units, two beyond (one
// group is nowhere faster than two).  Measured (us, few rows / tiles with one, two, four groups; the kernel of gemm.hip):
//   N 3,072, K 2,048   64 rows 27 / 55 / 45 / 42   100 rows 42 / 57 / 46 / 43    511 rows 131 / 84 / 80 / 84   (321, 306, 358)
//   N 2,048, K 8,192   64 rows 102 / 218 / 176 / 160   311 rows 266 / 218 / 176 / 162   511 rows 339 / 222 / 178 / 164   (1,488, 1,404, 1,423)
//   N 16,384, K 2,048   32 rows 48 / 61 / 48 / 47   64 rows 90 / 61 / 50 / 47   511 rows 696 / 334 / 330 / 340   (351, 391, 932)
//   N 6,144, K 4,096   48 rows 79 / 112 / 89 / 84   1,024 rows 1,032 / 481 / 462 / 486
// Up to four rows no tile at all: a wave a row of the weight, or two rows, which share the reads of x: from 8,192 rows of the
// weight on, with three rows of x (float32 weights) and four from 4,096 (4 rows, N 8,191, K 4,096, one / two rows a wave 37 / 30 us).
// Measured (us, tiles of 16 rows / this), 1, 2, 3 and 4 rows of x:
//   N 2,048, K 8,192   25.9 / 12.2   27.1 / 14.0   27.8 / 14.9   28.2 / 17.0 (128 tiles leave half of the compute units idle)
//   N 3,072, K 2,048   8.5 / 5.9   8.6 / 6.8   8.8 / 7.5   8.9 / 8.4
//   N 16,384, K 2,048   28.4 / 22.5   28.6 / 25.4   29.2 / 26.8   29.6 / 29.6
//   N 128,256, K 2,048   186 / 149   190 / 157   198 / 181   204 / 211
//   N 128,256, K 2,048, bfloat16 weights   170 / 85   174 / 104   180 / 122   183 / 140
// Not where the tiles are faster (the same way round, over N 64 to 128,256 and K 128 to 14,336):
//   four float32 rows against a float32 table: 65,536 x 4,096 209 / 217, 128,256 x 2,048 above (32,768 x 3,072 88 / 85);
//   rows too short for the loads of several pieces to overlap (bfloat16 x, N 65,536): 2 rows, K 128 10.3 / 12.2, 3 rows, K 256
//   14.9 / 20.3, (K 512 26.7 / 22.5); both float32, 3 rows, K 128 11.7 / 13.5, (K 256 16.8 / 15.5).
// Its sums are closer to 64 bits than the tiles' (0.9 to 1.3e-7 of the result, 1.2 to 1.5e-7).
template <typename TX, typename TW>
bool takes_dot(int M, int N, int K) {
  constexpr bool both_float32 = sizeof(TX) == 4 && sizeof(TW) == 4;
  if (M == 1) return true;
  if (M == 2) return both_float32 || K >= 256;
  if (M == 3) return K >= (both_float32 ? 256 : 512);
  return M == 4 && K >= 512 && !(both_float32 && N >= 65536 && K >= 2048);
}
static int g_force_form = 0;  // 0: the rule; 1: few rows; 2, 4: tiles with that many groups of waves

template <typename TX, typename TW, typename TO, int MR>
void launch_dot(const TX* x, const TW* w, TO* y, int N, int K, int ldx, int ldw, int ldy, hipStream_t stream) {
  if (N < (MR == 4 || (MR == 3 && sizeof(TW) == 4) ? 4096 : 8192))
    gemm_f32_dot_kernel<TX, TW, TO, MR, 1><<<(N + 3) / 4, 256, 0, stream>>>(x, w, y, N, K, ldx, ldw, ldy);
  else
    gemm_f32_dot_kernel<TX, TW, TO, MR, 2><<<(N + 7) / 8, 256, 0, stream>>>(x, w, y, N, K, ldx, ldw, ldy);
}

template <typename TX, typename TW, typename TO>
int launch(const TX* x, const TW* w, TO* y, int M, int N, int K, int ldx, int ldw, int ldy, hipStream_t stream) {
  const dim3 tiles((N + BT - 1) / BT, (M + BT - 1) / BT);
  const long long n_tiles = static_cast<long long>(tiles.x) * tiles.y;
  const int form = g_force_form ? g_force_form : M <= 32 || n_tiles < 96 ? 1 : n_tiles <= 256 ? 4 : 2;
  if (form == 4) {
    gemm_f32_tile_kernel<TX, TW, TO, 4><<<tiles, 1024, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy);
  } else if (form == 2) {
    gemm_f32_tile_kernel<TX, TW, TO, 2><<<tiles, 512, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy);
  } else if (g_force_form != 1 && takes_dot<TX, TW>(M, N, K)) {
    if (M == 1)
      launch_dot<TX, TW, TO, 1>(x, w, y, N, K, ldx, ldw, ldy, stream);
    else if (M == 2)
      launch_dot<TX, TW, TO, 2>(x, w, y, N, K, ldx, ldw, ldy, stream);
    else if (M == 3)
      launch_dot<TX, TW, TO, 3>(x, w, y, N, K, ldx, ldw, ldy, stream);
    else
      launch_dot<TX, TW, TO, 4>(x, w, y, N, K, ldx, ldw, ldy, stream);
  } else {
    const int cols = (N + 15) / 16;
    if (M <= 16 && cols <= 512 && K >= 1024)
      gemm_f32_rows_kernel<TX, TW, TO, 1, 16><<<dim3(cols, 1), 1024, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy);
    else if (M <= 16)
      gemm_f32_rows_kernel<TX, TW, TO, 1, 8><<<dim3(cols, 1), 512, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy);
    else if (M <= 32)
      gemm_f32_rows_kernel<TX, TW, TO, 2, 8><<<dim3(cols, 1), 512, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy);
    else
      gemm_f32_rows_kernel<TX, TW, TO, 4, 8><<<dim3(cols, (M + 63) / 64), 512, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy);
  }
  return yk_check_launch("gemm_f32");
}

template <typename TX, typename TW>
int launch_out(const void* x, const void* w, void* y, int y_dtype, int M, int N, int K, int ldx, int ldw, int ldy, hipStream_t stream) {
  if (y_dtype == YK_F32)
    return launch(static_cast<const TX*>(x), static_cast<const TW*>(w), static_cast<float*>(y), M, N, K, ldx, ldw, ldy, stream);
  return launch(static_cast<const TX*>(x), static_cast<const TW*>(w), static_cast<bf16_t*>(y), M, N, K, ldx, ldw, ldy, stream);
}

}  // namespace

// For tests and measurements: which form a product takes (0: the library decides; 1: tiles of 16 rows).
extern "C" int yk_gemm_f32_force(int form) {
  YK_REQUIRE(form == 0 || form == 1 || form == 2 || form == 4, "gemm_f32_force: 0 the rule, 1 few rows in tiles of 16, 2 / 4 tiles with that many groups of waves");
  g_force_form = form;
  return 0;
}

// Whether the operands' rows can be read four elements at a time (sizes and addresses as the entry
// point gemm_fma takes them; two bfloat16 operands stay there).
bool gemm_f32_takes(const void* x, int x_dtype, const void* w, int w_dtype, int y_dtype, int M, int K, int ldx, int ldw) {
  auto aligned = [](const void* p, int dtype) { return reinterpret_cast<uintptr_t>(p) % (dtype == YK_F32 ? 16 : 8) == 0; };
  return (x_dtype == YK_F32 || w_dtype == YK_F32) && (y_dtype == YK_F32 || y_dtype == YK_BF16) && (x_dtype == YK_F32 || x_dtype == YK_BF16) &&
         (w_dtype == YK_F32 || w_dtype == YK_BF16) && K % 4 == 0 && ldx % 4 == 0 && ldw % 4 == 0 && aligned(x, x_dtype) && aligned(w, w_dtype) &&
         (M + 63) / 64 <= 65535;
}

int gemm_f32(const void* x, int x_dtype, const void* w, int w_dtype, void* y, int y_dtype, int M, int N, int K, int ldx, int ldw, int ldy,
             hipStream_t stream) {
  if (x_dtype == YK_F32 && w_dtype == YK_F32) return launch_out<float, float>(x, w, y, y_dtype, M, N, K, ldx, ldw, ldy, stream);
  if (x_dtype == YK_BF16) return launch_out<bf16_t, float>(x, w, y, y_dtype, M, N, K, ldx, ldw, ldy, stream);
  return launch_out<float, bf16_t>(x, w, y, y_dtype, M, N, K, ldx, ldw, ldy, stream);
}
