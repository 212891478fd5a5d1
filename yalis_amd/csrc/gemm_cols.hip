// Few-row products y[M, N] = x[M, K] . w[N, K]^T that finish what they begin: up to 16 rows of
// bfloat16 x, K shared among the waves of a workgroup instead of among workgroups, so that the sums
// meet in LDS and the product's own epilogue (a bias, a gated pair, the rounding) runs
// on them.  The few-row product of gemm.hip divides K among workgroups and leaves slices, which a
// consumer that reads rows anyway (a norm, attention) adds on its way, but which elsewhere cost a
// kernel that does nothing else.
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

union Frag8 {
  u32x4_t u;
  bf16x8_t v;
};

constexpr int KC = 256;      // K elements a wave takes at a time
constexpr int ROW = KC + 8;  // an LDS row (16-byte reads of 16 neighbouring lanes meet no bank twice)
constexpr int STEPS = KC / 32;
constexpr int CHAINS = 2;    // running sums a wave keeps of one output, which its products join by turns

// what becomes of the sums
struct Finish {
  int gated, kind;  // pairs, as gated_pair makes them
  float p0, p1;
  const void* bias;  // [N] or null
  int bias_f32;
};

// a register from N lanes further on in the lane's row of 16 (which it wraps round)
template <int N>
__device__ __forceinline__ u32x4_t from_lanes_on(u32x4_t v) {
  if constexpr (N == 0) return v;
  u32x4_t o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = __builtin_amdgcn_update_dpp(0, v[i], 0x120 + (16 - N) % 16, 0xf, 0xf, false);  // row_ror:(16 - N)
  return o;
}

// A workgroup of W waves makes 16 columns (16 rows of the weight) for all rows of x; its waves walk K
// by turns, 256 elements at a time, the next chunk's loads in flight while the current one is
// multiplied.  As in gemm.hip: a load covers two rows x 512 bytes of the weight, the chunk is parked
// in a wave-private piece of LDS and read back as the matrix cores' A operand (v_mfma_f32_16x16x32_bf16:
// lane holds w[lane % 16][8 (lane / 16) ..]).  x comes from the caches straight into the B operand, since
// no other wave of the workgroup wants the same piece: of MR rows (the least of 2, 4, 8 and 16 that M fits) a load brings
// 16 / MR steps of 32, one in each MR lanes of a row of 16, and the lanes that hold the operand's columns get theirs by moves
// between registers (what the other lanes hold makes columns that nobody stores): a load of 1 KiB
// keeps the caches' path busy for 16 clocks whatever is in it, and eight a chunk for x took as long as the weight's own.
// Rows beyond N are read from the last row and
// never stored, K beyond the end is read from valid places and meets zeros of x.  Workgroups start at
// different chunks, so that they do not ask for addresses a whole number of rows apart at every moment,
// and those of one die (every eighth) at different ones too: against starting at the workgroup's number, when
// this was chosen, 4,096 x 4,096 11.1 -> 8.3 us, 8,192 x 4,096 19.2 -> 15.5, 4,672 x 2,048 8.9 -> 8.4.
// gated: the 16 rows are eight gate rows, then the eight up rows that belong to them.
// FIN: a bias or pairs; without, nothing but the sums is looked at.
// A wave's products join two running sums by turns: every addition rounds the sum it joins, and from a K of about
// 5,000 on one sum a wave met more of them than the slices of the other form do.  Distance from 64 bits in parts of
// 10^-7 of the result's norm (slices / one sum a wave / two): 1,024 x 5,632 1.41 / 1.62 / 1.22, 1,500 x 8,192
// 1.46 / 1.92 / 1.40, 1,024 x 12,288 1.76 / 2.38 / 1.68, 2,048 x 2,048 1.32 / 1.02 / 0.86; the same time.
// Bound by the reading of the weight, and in small matrices by the chain of it, LDS, the products and the meeting of the waves.  At 1, 4 and
// 8 rows, before x came in loads of several steps, the start was found without a division and the sums alone had a form of their own / now:
// 2,048 x 2,048 4.3, 4.6, 4.9 / 3.5, 4.2, 4.3 us; 11,264 x 2,048 9.9, 9.9, 10.5 / 9.4, 9.4, 9.7; 4,096 x 4,096 8.3, 8.3, 8.5 / 6.9, 7.1, 7.8.
template <typename TO, int MR, bool FIN, int W>
__global__ __launch_bounds__(64 * W) void gemm_cols_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                           TO* __restrict__ y, int M, int N, int K, int ldx, int ldw, int ldy,
                                                           uint32_t chunks_inverse, Finish f) {
  constexpr int GROUP = 16 / MR, XL = STEPS / GROUP;  // steps a load of x brings; loads a chunk
  __shared__ __attribute__((aligned(16))) bf16_t parked[W][16][ROW];
  __shared__ float sums[W][16][17];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int r = lane % 16, g = lane / 16, half = lane / 32, l32 = lane % 32;
  const int n0 = blockIdx.x * 16;
  const int n_chunks = (K + KC - 1) / KC, k_last = K - 8;
  // the rows of a load as bytes from the workgroup's first (they leave registers for a second workgroup on the compute unit)
  const bf16_t* w0 = w + static_cast<size_t>(n0) * ldw;
  uint32_t wrow[STEPS];
#pragma unroll
  for (int j = 0; j < STEPS; ++j) wrow[j] = 2u * static_cast<uint32_t>(min(2 * j + half, N - 1 - n0)) * static_cast<uint32_t>(ldw);
  const uint32_t xrow = static_cast<uint32_t>(min(r % MR, M - 1)) * static_cast<uint32_t>(ldx);
  const int turn = 5 * blockIdx.x + blockIdx.x / 8;
  const int start = n_chunks > 1 ? turn - n_chunks * divide_by(turn, n_chunks, chunks_inverse) : 0;
  auto chunk_at = [&](int i) {
    const int j = i + start;
    return (j >= n_chunks ? j - n_chunks : j) * KC;
  };
  u32x4_t wr[STEPS], xr[XL];
  auto fetch_w = [&](int kc) {
    const uint32_t k = 2u * static_cast<uint32_t>(min(kc + 8 * l32, k_last));
#pragma unroll
    for (int j = 0; j < STEPS; ++j)
      wr[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(reinterpret_cast<const char*>(w0) + (wrow[j] + k)));
  };
  auto fetch_x = [&](int kc) {
#pragma unroll
    for (int u = 0; u < XL; ++u) xr[u] = *reinterpret_cast<const u32x4_t*>(x + (xrow + min(kc + 32 * (GROUP * u + r / MR) + 8 * g, k_last)));
  };
  f32x4_t acc[CHAINS] = {};
  if (wave < n_chunks) {
    fetch_w(chunk_at(wave));
    fetch_x(chunk_at(wave));
  }
  for (int i = wave; i < n_chunks; i += W) {
    const int kc = chunk_at(i);
#pragma unroll
    for (int j = 0; j < STEPS; ++j) *reinterpret_cast<u32x4_t*>(&parked[wave][2 * j + half][8 * l32]) = wr[j];
    if (i + W < n_chunks) fetch_w(chunk_at(i + W));
    Frag8 a[STEPS];
#pragma unroll
    for (int u = 0; u < STEPS; ++u) a[u].u = *reinterpret_cast<const u32x4_t*>(&parked[wave][r][32 * u + 8 * g]);
    const bool whole = kc + KC <= K;
    auto multiply = [&](auto step) {
      constexpr int U = decltype(step)::value;
      Frag8 b;
      b.u = from_lanes_on<(U % GROUP) * MR>(xr[U / GROUP]);
      if (!whole) b.u = kc + 32 * U + 8 * g < K ? b.u : u32x4_t{0u, 0u, 0u, 0u};
      acc[U % CHAINS] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[U].v, b.v, acc[U % CHAINS], 0, 0, 0);
    };
    multiply(std::integral_constant<int, 0>{});
    multiply(std::integral_constant<int, 1>{});
    multiply(std::integral_constant<int, 2>{});
    multiply(std::integral_constant<int, 3>{});
    multiply(std::integral_constant<int, 4>{});
    multiply(std::integral_constant<int, 5>{});
    multiply(std::integral_constant<int, 6>{});
    multiply(std::integral_constant<int, 7>{});
    if (i + W < n_chunks) fetch_x(chunk_at(i + W));
  }
  // lane holds columns 4g .. 4g + 3 of row r of x
#pragma unroll
  for (int e = 0; e < 4; ++e) sums[wave][r][4 * g + e] = acc[0][e] + acc[1][e];
  __syncthreads();
  auto total = [&](int m, int c) {
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < W; ++v) s += sums[v][m][c];
    if (FIN && f.bias && n0 + c < N)
      s += f.bias_f32 ? static_cast<const float*>(f.bias)[n0 + c] : to_f32<bf16_t>(static_cast<const bf16_t*>(f.bias)[n0 + c]);
    return s;
  };
  if (FIN && f.gated) {
    for (int o = threadIdx.x; o < 8 * M; o += 64 * W) {
      const int m = o / 8, c = o % 8;
      const float v = gated_pair(as_output(total(m, c), 1), as_output(total(m, c + 8), 1), f.kind, f.p0, f.p1);
      y[static_cast<size_t>(m) * ldy + n0 / 2 + c] = from_f32<TO>(v);
    }
    return;
  }
  const int o = threadIdx.x, m = o / 16, c = o % 16;  // (at most 256 outputs)
  if (o < 16 * M && n0 + c < N) y[static_cast<size_t>(m) * ldy + n0 + c] = from_f32<TO>(total(m, c));
}

static int g_mode = 0;

}  // namespace

// Whether a product of these sizes goes this way; slices_do: the other form would need no kernel of its own
// after it (its consumer adds the slices, or there is one slice only).
// Measured in replayed graphs with a copy of x before and the residual's norm after (us: slices added by the norm (by a kernel of their own) / this):
//            1 row                        8 rows                       16 rows
//   1,024 x 2,048    8.4 (10.0) / 7.2     9.0 (10.6) / 8.2     9.4 (11.0) / 9.1
//   1,024 x 4,096    9.0 (10.7) / 8.4     9.5 (10.9) / 10.0    9.9 (11.4) / 11.9
//   2,048 x 2,048    9.1 (10.6) / 7.8     9.6 (11.2) / 8.5     9.9 (11.6) / 9.5
//   2,048 x 5,632   11.3 (12.8) / 10.4   12.1 (13.8) / 12.5   13.0 (14.5) / 14.9
//   2,048 x 8,192   12.7 (13.6) / 12.3   13.2 (14.5) / 14.2   13.9 (15.1) / 17.6
//   3,072 x 3,072   11.0 (12.6) / 8.9    11.5 (13.3) / 10.5   12.1 (13.9) / 11.6
//   3,072 x 8,192   14.8 (15.9) / 13.9   15.4 (16.7) / 15.4   16.4 (17.8) / 18.6
//   4,096 x 2,048    9.9 (11.4) / 8.8    10.5 (11.9) / 9.5    11.0 (12.7) / 10.4
//   4,096 x 4,096   12.6 (13.6) / 11.0   13.0 (14.4) / 12.1   13.9 (14.8) / 13.5
//   4,096 x 11,008  22.2 (23.0) / 19.8   22.9 (24.0) / 21.1   23.8 (25.2) / 24.9
//   4,096 x 14,336  24.4 (25.4) / 23.4   24.8 (26.0) / 25.1   25.9 (27.3) / 29.9
//   5,120 x 4,096   15.0 (15.1) / 14.5   15.5 (15.9) / 16.5   16.3 (16.7) / 20.5
//   6,144 x 4,096   16.8 (16.2) / 14.9   17.0 (17.6) / 16.9   18.0 (18.0) / 20.6
//   8,192 x 4,096   18.4 (19.3) / 16.6   18.9 (20.2) / 17.9   19.4 (20.3) / 22.1
//   8,192 x 5,632   21.0 (22.3) / 20.8   21.8 (23.0) / 22.7   22.6 (23.8) / 25.9
// (gated, with a copy of x before, fused or slices and the activation's kernel / this) 8,192 x 2,048 11.3 / 9.1, 11.7 / 10.1, 12.3 / 11.5; 8,192 x
// 4,096 16.1 / 14.5, 16.3 / 15.4, 16.8 / 19.7; 16,384 x 2,048 14.7 / 14.2, 15.0 / 15.4, 15.5 / 17.7; 28,672 x 4,096 37.4 / 38.4, 37.1 / 40.8, 37.9 / 53.8
// A workgroup of 16 columns reads x once for them, four times as often a column as the other form, and
// ends with a barrier and a few sums: both count the more, the more rows x has and the more workgroups a compute unit runs one
// after another; few columns are few workgroups, whose walk over a long K nothing divides further; and a second round that fills a part of
// the units waits for the first.  So, where slices would do (handed_on), up to eight rows:
//   - matrices of up to 6.5 M elements whose K and columns are not far apart (1,024 x 4,096 at eight rows 9.5 / 10.0; one slice: 8,192 x 512
//     5.3 / 4.3, 12,288 x 512 5.5 / 5.7, 25,344 x 256 4.8 / 8.2);
//   - larger ones whose workgroups make one or two rounds of the compute units with an eighth of them idle or fewer (as above, slices / this: 4,112 x
//     8,192 19.2 / 23.6, 8,208 x 4,096 20.2 / 21.6; 3,584 and 3,600 x 8,192 16.8 / 16.5 and 17.2 / 17.2, 7,168 and 7,680 x 4,096 17.2 / 17.5 and 18.1 / 17.8),
//     up to where the two meet (4,096 x 11,008 22.9 / 21.2, 12,288 22.6 / 22.9, 13,312 23.7 / 23.8; 8,192 x 4,096 18.9 / 18.2, 4,864 20.1 / 20.7);
//   - up to four rows as far as that line lies then (4,096 x 14,336 24.6 / 23.8, 16,384 26.8 / 27.0; 2,048 x 5,120 11.3 / 11.1, 5,888 11.7 / 11.7; between 2,560 and
//     2,816 columns, and with five rows, it is 3 to 8 % ahead some way beyond); up to two rows (2,048 x 8,192 12.7 / 12.5, 9,216 13.6 / 13.6;
//     1,024 x 4,096 9.1 / 8.7, 5,120 9.6 / 10.1; 16,384 x 2,048 20.2 / 18.4, 2,304 21.3 / 20.7);
//   - of the larger ones only those with one side half as long again as the other.  That is no line of speed: square ones are ahead here too (one, four and
//     eight rows: 3,072 x 3,072 11.0, 11.2, 11.4 / 9.1, 9.9, 10.4; 4,096 x 4,096 12.2, 12.7, 13.2 / 11.2, 11.6, 12.0; 4,096 x 6,136 16.4, 17.0, 17.4 / 14.0, 14.8, 15.7).
//     It is the price of an interface: products of this shape come as slices in the library's workspace, and a program that holds them while
//     it launches the next product is told so.
// At 16 rows the two are about even, and a product that takes attention's
// unmerged splits (which this form does not) has the bits of the one that takes them merged there.
// Where a kernel would have to add the slices: also up to 13 M elements (36 M with up to 8 rows and a K of one round of eight waves) with a K
// of up to 8,192 (6,144 from 13 rows on; any with up to four), but not a short K against many columns (with a
// bias 16,384 x 256 6.1 / 5.2, 22,016 x 256 7.0 / 7.2 at 8 rows; 16,384 x 1,024 9.8 / 9.3, 22,016 x 1,024 11.7 / 12.4).
// Narrow products, of fewer than 1,024 columns, would gain too (256 x 2,048 7.2 / 4.0) and stay where they are:
// there a product has the same bits whether it comes as slices or reduced, which programs that compare the two
// may count on; here its sums run in another order.
static bool handed_on(int M, int N, int K) {
  const long long elements = static_cast<long long>(N) * K;
  if (M <= 8 && elements <= 6500000 && K >= KC && (K <= 8 * KC || 2LL * K <= 3LL * N) && (N <= 8192 || N <= 16LL * K)) return true;
  if (M > 8 || K < 8 * KC || (2LL * K < 3LL * N && 2LL * N < 3LL * K)) return false;
  constexpr int UNITS = 256;  // compute units, a workgroup of 16 columns each
  const int tiles = (N + 15) / 16;
  auto rounds = [&](int r) { return tiles > r * UNITS - r * UNITS / 8 && tiles <= r * UNITS; };
  const bool one_round = rounds(1), two_rounds = rounds(2);
  if ((one_round && K <= 12288) || (two_rounds && K <= 4096)) return true;
  if (M <= 4 && (((N >= 2816 && N <= 4096) || two_rounds) && K <= 14336)) return true;
  if (M <= 4 && N >= 2048 && N < 2816 && K <= 5632) return true;
  return M <= 2 && ((N <= 2048 && K <= 4LL * N) || (rounds(4) && K <= 8 * KC));
}

extern "C" int yk_gemm_cols_ok(int M, int N, int K, int slices_do) {
  if (M < 1 || M > 16 || K < 8 || K % 8 || N < 1) return 0;
  if (g_mode) return g_mode == 2;
  if (N < 1024) return 0;
  if (handed_on(M, N, K)) return 1;
  const long long elements = static_cast<long long>(N) * K;
  if (slices_do || (M > 4 && K > (M <= 12 ? 8192 : 6144))) return 0;
  if (elements <= 13000000) return N <= 64LL * K;
  return M <= 8 && elements <= 36000000 && K <= 8 * KC && N <= 16LL * K;
}

// For tests and measurements: 0 the rule, 1 never, 2 wherever it can.
extern "C" int yk_gemm_cols_force(int mode) {
  YK_REQUIRE(mode >= 0 && mode <= 2, "gemm_cols_force: 0 the rule, 1 never, 2 wherever it can");
  g_mode = mode;
  return 0;
}

// y [M, N] = the product (+ bias); gated: the rows of w alternate in groups of eight gate rows and their
// eight up rows, y [M, N / 2] bfloat16 = gated_pair of them (kind, p0, p1).
extern "C" int yk_gemm_cols(const void* x, const void* w, void* y, int y_dtype, int M, int N, int K, int ldx, int ldw, int ldy,
                            const void* bias, int bias_dtype, int gated, int kind, float p0, float p1, hipStream_t stream) {
  YK_REQUIRE(M >= 0 && M <= 16 && N > 0 && K > 0 && K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0,
             "gemm_cols: up to 16 rows; K and the leading dimensions must be multiples of 8");
  YK_REQUIRE(ldw < 1 << 27, "gemm_cols: a workgroup's rows of the weight must lie within 4 GiB");
  YK_REQUIRE(ldx >= K && ldw >= K && ldy >= (gated ? N / 2 : N), "gemm_cols: leading dimensions too small");
  YK_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0, "gemm_cols: operands must be 16-byte aligned");
  YK_REQUIRE(y_dtype == YK_BF16 || (y_dtype == YK_F32 && !gated), "gemm_cols: unsupported output dtype");
  YK_REQUIRE(!gated || (N % 16 == 0 && kind >= 0 && kind < YK_GATED_KINDS), "gemm_cols: a gated product needs N % 16 == 0 and a known pair");
  YK_REQUIRE(!bias || bias_dtype == YK_F32 || bias_dtype == YK_BF16, "gemm_cols: unsupported bias dtype");
  if (M == 0) return 0;
  if (static_cast<long long>(M - 1) * ldx + K >= 1ll << 31) {  // the kernel's offsets into x have 32 bits: rows that far apart go one by one (the same sums)
    for (int m = 0; m < M; ++m) {
      const int rc = yk_gemm_cols(static_cast<const bf16_t*>(x) + static_cast<size_t>(m) * ldx, w,
                                  static_cast<char*>(y) + static_cast<size_t>(m) * ldy * (y_dtype == YK_F32 ? 4 : 2), y_dtype, 1, N, K, ldx, ldw, ldy, bias,
                                  bias_dtype, gated, kind, p0, p1, stream);
      if (rc) return rc;
    }
    return 0;
  }
  const Finish f{gated, kind, p0, p1, bias, bias_dtype == YK_F32};
  const unsigned tiles = (N + 15) / 16;
  const int n_chunks = (K + KC - 1) / KC;
#define YK_COLS(TO, MR, FIN, W)                                                                                               \
  gemm_cols_kernel<TO, MR, FIN, W><<<tiles, 64 * W, 0, stream>>>(static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), \
                                                                     static_cast<TO*>(y), M, N, K, ldx, ldw, ldy,             \
                                                                     n_chunks > 1 ? inverse_of(n_chunks) : 0u, f)
#define YK_COLS_WAVES(TO, MR, FIN)          \
  if (sixteen) YK_COLS(TO, MR, FIN, 16);         \
  else YK_COLS(TO, MR, FIN, 8)
#define YK_COLS_ROWS(TO, FIN)               \
  if (M <= 2) { YK_COLS_WAVES(TO, 2, FIN); } \
  else if (M <= 4) { YK_COLS_WAVES(TO, 4, FIN); } \
  else if (M <= 8) { YK_COLS_WAVES(TO, 8, FIN); } \
  else { YK_COLS_WAVES(TO, 16, FIN); }
  const bool sixteen = tiles <= 256 && n_chunks > 8 && n_chunks <= 24;
  const bool fin = gated || bias;
  if (y_dtype == YK_F32 && fin) { YK_COLS_ROWS(float, true); }
  else if (y_dtype == YK_F32) { YK_COLS_ROWS(float, false); }
  else if (fin) { YK_COLS_ROWS(bf16_t, true); }
  else { YK_COLS_ROWS(bf16_t, false); }
#undef YK_COLS_ROWS
#undef YK_COLS_WAVES
#undef YK_COLS
  return yk_check_launch("gemm_cols");
}
