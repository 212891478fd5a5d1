// Products y[M, N] = x[M, K] . w[N, K]^T of float32 operands on the bfloat16 matrix cores: every float32 is the exact sum of three bfloat16
// (its rounding, the rounding of what is left, and the rest), and of the nine products of parts the six are made whose terms reach the last
// places of the float32 product.  The float32 matrix instructions reach 1/16 of the bfloat16 rate, and the kernel on them about 110 TFLOP/s;
// six products of parts leave 2.7 times theirs.
//
// What is lost: parts smaller than 2^-24 of a product, three terms of nine, each below 2^-25 of it.  What is gained: a matrix instruction adds
// 32 products of one element of y, not four, so that sums are rounded less often.  Error against 64 bits (root mean square, of normal numbers;
// the float32 instructions in brackets): K 516 0.8e-7 (1.0e-7), 2,048 0.9e-7 to 1.0e-7 (1.2e-7 to 1.7e-7), 4,096 1.0e-7 to 1.3e-7 (1.4e-7 to
// 2.2e-7), 8,192 1.1e-7 to 1.6e-7 (1.7e-7 to 3.0e-7).
//
// us, before (float32 instructions) / now: 511 x 16,384 x 2,048 314 / 209 (164 TFLOP/s), 511 x 3,072 x 2,048 78 / 52, 511 x 2,048 x 2,048
// 42.6 / 36.7, 511 x 2,048 x 8,192 160 / 115, 2,000 x 6,144 x 4,096 915 / 547 (184), 200 x 16,384 x 2,048 160 / 94, 64 x 2,048 x 8,192
// 101 / 29, 33 x 3,072 x 2,048 28 / 17.  With one row of x that makes infinities, NaN or sums beyond 2^80 (below): 511 x 16,384 x 2,048 317, 511 x
// 2,048 x 8,192 183, 200 x 3,072 x 2,048 59 (34 without); with all of them so 10.0, 5.0 and 1.5 ms, by a lane for each element 30, 15 and 3.8.
// What bounds it: the largest is held by the matrix cores (50% busy) and the vector instructions that take w apart (30%) at 2.0 GHz, which
// is what power leaves; LDS reads are 25%.  Splitting both operands in the kernel through LDS took 200 to 250 us there and 66 to 94 on 511 x
// 3,072 x 2,048.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// Operands are taken 2^24 times as large, so that the parts of the smallest float32 are no subnormal numbers, which the bfloat16 products
// take for zeros; what grows beyond float32 on the way is made again without (below).
constexpr float SCALE = 16777216.f;

// two elements into their parts, two bfloat16 a word
__device__ __forceinline__ void apart(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  a *= SCALE;
  b *= SCALE;
  h = pack_bf16x2(a, b);
  a -= __uint_as_float(h << 16);
  b -= __uint_as_float(h & 0xffff0000u);
  m = pack_bf16x2(a, b);
  a -= __uint_as_float(m << 16);
  b -= __uint_as_float(m & 0xffff0000u);
  l = pack_bf16x2(a, b);
}

// x [M, K] into its parts [3][M][kp], zeros from K on (kp a multiple of 128).  Of every 32 elements along K the parts hold 4 q .. + 3 and
// 16 + 4 q .. + 3 at 8 q .. + 7: what one lane of a matrix instruction multiplies are two pieces of 16 bytes of a row of w, and the first
// pieces of a row's four lanes lie side by side.
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ x, bf16_t* __restrict__ parts, int M, int K, int ldx, int kp) {
  const int64_t at = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
  if (at >= static_cast<int64_t>(M) * kp) return;
  const int m = static_cast<int>(at / kp), p = static_cast<int>(at % kp), k = p / 32 * 32 + p % 32 / 2;
  const float* const row = x + static_cast<size_t>(m) * ldx + k;
  const f32x4_t none = {0.f, 0.f, 0.f, 0.f};
  const f32x4_t u = k < K ? *reinterpret_cast<const f32x4_t*>(row) : none, v = k + 16 < K ? *reinterpret_cast<const f32x4_t*>(row + 16) : none;
  uint32_t h[4], mid[4], l[4];
  apart(u[0], u[1], h[0], mid[0], l[0]);
  apart(u[2], u[3], h[1], mid[1], l[1]);
  apart(v[0], v[1], h[2], mid[2], l[2]);
  apart(v[2], v[3], h[3], mid[3], l[3]);
  const size_t plane = static_cast<size_t>(M) * kp;
  *reinterpret_cast<u32x4_t*>(parts + at) = u32x4_t{h[0], h[1], h[2], h[3]};
  *reinterpret_cast<u32x4_t*>(parts + plane + at) = u32x4_t{mid[0], mid[1], mid[2], mid[3]};
  *reinterpret_cast<u32x4_t*>(parts + 2 * plane + at) = u32x4_t{l[0], l[1], l[2], l[3]};
}

// f(0) .. f(N - 1), each number a constant
template <int N, int I = 0, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>());
    each<N, I + 1>(f);
  }
}

// A workgroup of four waves makes 128 columns (rows of w) x 64 rows of y over one slice of K, a wave 32 x 64, 32 along K a step.  x comes in
// parts and goes to LDS as it is, three steps ahead in a ring of four; each wave takes its own rows of w apart in registers, where the matrix
// instructions need them, between the instructions of the step before: w does not pass LDS, and of x a step reads 12 KiB a wave for 48
// instructions.  The parts' planes of x are read in the order of their last use, so that one set of registers holds them: a step's instructions
// begin with x's third part and end with its first.  The products of both first parts and all others have sums of their own: the others
// are at most 2^-7 of the first, and so is what rounding their sums costs.  250 registers: two workgroups a compute unit.
constexpr int BN = 128, BM = 64, RING = 4, PLANE = BM * 64, STAGE = 3 * PLANE;

__global__ __launch_bounds__(256, 2) void gemm_split_kernel(const bf16_t* __restrict__ parts, int kp, const float* __restrict__ w,
                                                            float* __restrict__ y, int M, int N, int K, int ldw, int ldy, int slice_steps,
                                                            int vector, const float* __restrict__ x, int ldx) {
  constexpr int LX = STAGE / 1024 / 4;
  __shared__ __attribute__((aligned(1024))) unsigned char lds[RING * STAGE];
  // the dies take turns with workgroups: each gets a run of tiles, eight tiles of rows to a band
  const int tn = (N + BN - 1) / BN, tm = (M + BM - 1) / BM, tiles = tn * tm, total = gridDim.x, die = blockIdx.x % 8;
  const int u = die * (total / 8) + min(die, total % 8) + blockIdx.x / 8, z = u / tiles, t = u % tiles;
  const int first = t / (8 * tn) * 8, high = min(8, tm - first), r0 = t - first * tn;
  const int m0 = (first + r0 % high) * BM, n0 = r0 / high * BN;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), row = lane % 16, quarter = lane / 16;
  const int s0 = z * slice_steps, steps = min(slice_steps, kp / 32 - s0);  // a multiple of four
  y += static_cast<size_t>(z) * M * ldy;

  // x: KiB l * 4 + wave of a step's three planes, 16 rows each; rows beyond M lie beyond a plane's end
  const size_t plane = static_cast<size_t>(M) * kp;
  const bf16_t* const xbase = parts + static_cast<size_t>(m0) * kp;
  const int xbytes = min(BM, M - m0) * kp * 2;
  // LDS: rows of 64 bytes, piece c of row r at place c ^ swap(r / 4)
  auto swap = [](int i) { return (i & 1) << 1 ^ (i >> 1) * 3; };
  const int xlane = (lane / 4 * kp + 8 * ((lane % 4) ^ swap(lane / 16))) * 2;
  auto load_x = [&](int s, int l) {
    const int g = l * 4 + wave, r = g % (BM / 16) * 16;
    load_to_lds(xbase + g / (BM / 16) * plane, s < steps ? xbytes : 0, lds + s % RING * STAGE + g * 1024, xlane, r * kp * 2 + (s0 + s) * 64);
  };
  // w: what is read beyond a row's K meets zeros of x
  const float* const wbase = w + static_cast<size_t>(n0) * ldw;
  const auto wsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(wbase), 0, ((min(BN, N - n0) - 1) * ldw + K) * 4, 0x00027000);
  const int wlane = ((wave * 32 + row) * ldw + 4 * quarter) * 4;
  u32x4_t raw[2][2][2];  // [step % 2][i][half]
  auto fetch = [&](int s, int set, int i, int half) {
    raw[set][i][half] = __builtin_amdgcn_raw_buffer_load_b128(wsrc, wlane, i * 16 * ldw * 4 + (s0 + s) * 128 + half * 64, 0);
  };
  uint32_t a[2][3][2][4];  // [step % 2][part][i]: operands
  // a third of the taking apart of pair p (0 .. 7) of raw[set]
  float va, vb;
  auto take = [&](int set, int to, int p, int third) {
    const int i = p / 4, half = p / 2 % 2, e = p % 2;
    if (third == 0) {
      va = __uint_as_float(raw[set][i][half][2 * e]) * SCALE;
      vb = __uint_as_float(raw[set][i][half][2 * e + 1]) * SCALE;
    } else {
      const uint32_t before = a[to][third - 1][i][p % 4];
      va -= __uint_as_float(before << 16);
      vb -= __uint_as_float(before & 0xffff0000u);
    }
    a[to][third][i][p % 4] = pack_bf16x2(va, vb);
  };
  const unsigned char* const from = lds + row * 64 + (quarter ^ swap(row / 4)) * 16;
  bf16x8_t b[3][4];
  auto read = [&](int s, int p, int j) { b[p][j] = *reinterpret_cast<const bf16x8_t*>(from + s % RING * STAGE + p * PLANE + j * 1024); };
  f32x4_t acc[2][4] = {}, part[2][4] = {}, rest[2][4] = {};

  auto step = [&](int s, auto dc) {
    constexpr int d = decltype(dc)::value, Q = 48;  // d = s % 4
    each<Q>([&](auto qc) {
      constexpr int q = decltype(qc)::value, term = q / 8, i = q / 4 % 2, j = q % 4;
      constexpr int px = term < 1 ? 2 : term < 3 ? 1 : 0, pw = term == 0 ? 0 : term == 1 ? 1 : term == 2 ? 0 : 5 - term;
      f32x4_t& to = term < 5 ? rest[i][j] : part[i][j];
      const u32x4_t av = {a[d % 2][pw][i][0], a[d % 2][pw][i][1], a[d % 2][pw][i][2], a[d % 2][pw][i][3]};
      to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av), b[px][j], to, 0, 0, 0);
      if constexpr (q < 8 && q % 2 == 0) read(d, 0, q / 2);
      if constexpr (q >= 10 && q < 18 && q % 2 == 0) read(d + 1, 2, (q - 10) / 2);
      if constexpr (q >= 26 && q < 34 && q % 2 == 0) read(d + 1, 1, (q - 26) / 2);
      if constexpr (q < 2 * LX && q % 2 == 1) load_x(s + 3, q / 2);
      if constexpr (q < 36 && q % 3 != 2) {
        constexpr int c = q / 3 * 2 + q % 3;
        take((d + 1) % 2, (d + 1) % 2, c / 3, c % 3);
      }
      if constexpr (q >= 38 && q < 46 && q % 2 == 0) fetch(s + 3, (d + 1) % 2, (q - 38) / 4, (q - 38) / 2 % 2);
      __builtin_amdgcn_sched_barrier(0);
    });
    // x of step s + 2 has landed: four loads of w, three of x and four of w were asked for after it
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(((4 + LX + 4) & 15) | (4 + LX + 4) >> 4 << 14 | 7 << 4 | 0 << 8);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int l = 0; l < LX; ++l) load_x(s, l);
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      fetch(s, s, i, 0);
      fetch(s, s, i, 1);
    }
#pragma unroll
  for (int c = 0; c < 24; ++c) take(0, 0, c / 3, c % 3);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    fetch(2, 0, i, 0);
    fetch(2, 0, i, 1);
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    read(0, 2, j);
    read(0, 1, j);
  }
  for (int s = 0; s < steps; s += 4) {
    each<4>([&](auto dc) { step(s + decltype(dc)::value, dc); });
    // Sums of 128 products start from nothing: a running sum is rounded K / 128 times.
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[i][j] += part[i][j];
        part[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
  }
  __builtin_amdgcn_s_waitcnt(0);  // no load may still be on its way into LDS
  // lane l holds columns 4 (l / 16) .. + 3 of row l % 16
  uint32_t again = 0;  // bit 16 i + 4 j + e
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int mi = m0 + j * 16 + row, n = n0 + wave * 32 + i * 16 + 4 * quarter;
      if (mi >= M) continue;
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[e] = (acc[i][j][e] + rest[i][j][e]) * (1.f / SCALE) * (1.f / SCALE);
        if (!(fabsf(o[e]) <= 3.402823466e38f) && n + e < N) again |= 1u << (16 * i + 4 * j + e);
      }
      float* const to = y + static_cast<size_t>(mi) * ldy + n;
      if (vector && n + 3 < N) {
        *reinterpret_cast<f32x4_t*>(to) = f32x4_t{o[0], o[1], o[2], o[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) to[e] = o[e];
      }
    }
  // An infinity has no rest, and neither has a number that is one when scaled or rounded: what such operands give is made of them as they
  // are, an element at a time by the whole wave: sums of 16 products, added up along K by each lane and then over the lanes.
  const int k0 = s0 * 32, k1 = min(K, k0 + steps * 32);
  for (uint64_t lanes = __ballot(again != 0); lanes != 0; lanes = __ballot(again != 0)) {
    const int from = __builtin_ctzll(lanes);
    const int which = __builtin_ctz(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(again), from)));
    const int mi = m0 + which / 4 % 4 * 16 + from % 16, n = n0 + wave * 32 + which / 16 * 16 + from / 16 * 4 + which % 4;
    const float* const xm = x + static_cast<size_t>(mi) * ldx;
    const float* const wv = w + static_cast<size_t>(n) * ldw;
    float v = 0.f;
    for (int k = k0 + 16 * lane; k < k1; k += 16 * 64) {
      float sum = 0.f;
#pragma unroll
      for (int p = 0; p < 16; p += 4) {
        if (k + p >= k1) break;  // (K is a multiple of four)
        const f32x4_t a4 = *reinterpret_cast<const f32x4_t*>(xm + k + p), b4 = *reinterpret_cast<const f32x4_t*>(wv + k + p);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum = fmaf(a4[e], b4[e], sum);
      }
      v += sum;
    }
    v = wave_sum(v);
    if (lane == from) {
      y[static_cast<size_t>(mi) * ldy + n] = v;
      again &= again - 1;
    }
  }
}

// y [M, N] of slices [slices][M][N], added in order; four elements a thread (count = M N of a multiple of four, y rows N apart)
__global__ __launch_bounds__(256) void add_slices_kernel(const f32x4_t* __restrict__ part, f32x4_t* __restrict__ y, int slices, int64_t count) {
  const int64_t at = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (at >= count) return;
  f32x4_t v = part[at];
  for (int z = 1; z < slices; ++z) v += part[z * count + at];
  y[at] = v;
}

// rows of x that are taken apart at a time: their parts take up to 64 MiB
int pass_rows(int kp) { return std::max(64, (64 << 20) / (6 * kp) / 64 * 64); }
int padded(int K) { return (K + 127) / 128 * 128; }

// The rule: what a product takes here and in gemm_f32, us, fitted to what 104 products of 33 to 2,000 rows, 64 to 16,384 columns and K of
// 4 to 8,192 took (nowhere 2% slower than gemm_f32 there; the largest gain left is 2,000 x 128 x 2,048, 34 where 25 us would do).  Here: the split of x; the compute
// units work through their workgroups' steps in turn, however many are resident, and w comes at 4 TB/s; slices are written, and read by a
// kernel of their own; rows beyond a pass walk along K again, which takes a tenth less than the passes apart (us, there / here: 5,677 x 632 x 6,592, four
// passes, 501 / 677, 1,681 x 916 x 7,264, two, 288 / 324, 2,009 x 7,724 x 5,428 1,702 / 1,105; 63 of 120 such products are taken, the slowest in 1.02 times
// its time there).  There: few tiles of 64 x 64 run as tiles of 16 rows, in the time of one walk along K, more in rounds of 256.
double split_us(int M, int N, int K, int slices) {
  const int kp = padded(K), per = (kp / 128 + slices - 1) / slices * 4, rows = pass_rows(kp);
  if (M > rows) return .9 * (M / rows * split_us(rows, N, K, slices) + (M % rows ? split_us(M % rows, N, K, slices) : 0.));
  const double rounds = std::ceil(static_cast<double>((N + BN - 1) / BN) * ((M + BM - 1) / BM) * ((kp / 32 + per - 1) / per) / 256.);
  return 8. + std::max((rounds > 1. ? .7 : .75) * per * rounds, 1e-6 * N * K) + 1.5e-6 * M * kp + (slices > 1 ? 4. + 2e-6 * slices * M * N : 0.);
}

double f32_us(int M, int N, int K) {
  const double tiles = static_cast<double>((M + 63) / 64) * ((N + 63) / 64);
  return tiles < 96. ? 3. + .0102 * K : 4. + .019 * K * std::ceil(tiles / 256.);
}

}  // namespace

// The K slices in which a product of float32 (rows of aligned pieces of 16 bytes) is best made here, or 0 where gemm_f32 is faster.
extern "C" int yk_gemm_split_plan(int M, int N, int K) {
  if (M <= 32 || N <= 0 || K <= 0 || K % 4 || K > 1 << 22) return 0;
  int best = 1;
  if (N % 4 == 0 && M <= pass_rows(padded(K)))
    for (int slices = 2; slices <= 16 && slices <= padded(K) / 128; ++slices)
      if (split_us(M, N, K, slices) < split_us(M, N, K, best)) best = slices;
  return split_us(M, N, K, best) < f32_us(M, N, K) ? best : 0;
}

// Floats of scratch that the product takes.
extern "C" int64_t yk_gemm_split_floats(int M, int N, int K, int slices) {
  const int kp = padded(K);
  return (static_cast<int64_t>(3) * std::min(M, pass_rows(kp)) * kp + 1) / 2 + (slices > 1 ? static_cast<int64_t>(slices) * M * N : 0);
}

extern "C" int yk_gemm_split(const float* x, const float* w, float* y, float* ws, int64_t ws_floats, int M, int N, int K, int ldx, int ldw, int ldy,
                             int slices, hipStream_t stream) {
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  YK_REQUIRE(M > 0 && N > 0 && K > 0 && K % 4 == 0 && K <= 1 << 22, "gemm_split: bad sizes");
  YK_REQUIRE(ldx >= K && ldw >= K && ldy >= N && ldx % 4 == 0 && ldw % 4 == 0 && ldw <= 1 << 21 && aligned(x) && aligned(w) && aligned(ws),
             "gemm_split: rows of x and w are read in aligned pieces of 16 bytes");
  const int kp = padded(K), rows = pass_rows(kp);
  YK_REQUIRE(slices >= 1 && slices <= kp / 128, "gemm_split: slices are 128 along K and longer");
  YK_REQUIRE(slices == 1 || (M <= rows && N % 4 == 0 && ldy == N && aligned(y)), "gemm_split: these rows are not for slices");
  YK_REQUIRE(ws_floats >= yk_gemm_split_floats(M, N, K, slices), "gemm_split: scratch too small");
  const int64_t tiles = static_cast<int64_t>((N + BN - 1) / BN) * ((std::min(M, rows) + BM - 1) / BM);
  YK_REQUIRE(tiles * slices < 1 << 30, "gemm_split: too many tiles");
  bf16_t* const parts = reinterpret_cast<bf16_t*>(ws);
  float* const sums = ws + (static_cast<int64_t>(3) * std::min(M, rows) * kp + 1) / 2;
  const int per = (kp / 128 + slices - 1) / slices * 4, made = (kp / 32 + per - 1) / per;
  for (int at = 0; at < M; at += rows) {
    const int m = std::min(rows, M - at);
    const float* const xm = x + static_cast<size_t>(at) * ldx;
    float* const to = made > 1 ? sums : y + static_cast<size_t>(at) * ldy;
    const int vector = ldy % 4 == 0 && aligned(to);
    split_rows_kernel<<<static_cast<int>((static_cast<int64_t>(m) * kp / 8 + 255) / 256), 256, 0, stream>>>(xm, parts, m, K, ldx, kp);
    const int groups = ((N + BN - 1) / BN) * ((m + BM - 1) / BM) * made;
    gemm_split_kernel<<<groups, 256, 0, stream>>>(parts, kp, w, to, m, N, K, ldw, ldy, per, vector, xm, ldx);
  }
  if (made > 1) {
    const int64_t count = static_cast<int64_t>(M) * N / 4;
    add_slices_kernel<<<static_cast<int>((count + 255) / 256), 256, 0, stream>>>(reinterpret_cast<const f32x4_t*>(sums), reinterpret_cast<f32x4_t*>(y),
                                                                                 made, count);
  }
  return yk_check_launch("gemm_split");
}
