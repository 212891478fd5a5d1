// Few-row products y[M, N] = x[M, K] . w[N, K]^T that finish what they begin: up to 16 rows of
// bfloat16 x, K shared among the waves of a workgroup instead of among workgroups, so that the sums
// meet in LDS and the product's own epilogue (a bias, a gated pair, the rounding) runs
// on them.  The few-row product of gemm.hip divides K among workgroups and leaves slices, which a
// consumer that reads rows anyway (a norm, attention) adds on its way, but which elsewhere cost a
// kernel that does nothing else.
#include <algorithm>

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
constexpr int W = 8;         // waves a workgroup
constexpr int CHAINS = 2;    // running sums a wave keeps of one output, which its products join by turns

// what becomes of the sums
struct Finish {
  int gated, kind;  // pairs, as gated_pair makes them
  float p0, p1;
  const void* bias;  // [N] or null
  int bias_f32;
};

// A workgroup of eight waves makes 16 columns (16 rows of the weight) for all rows of x; its waves walk K
// by turns, 256 elements at a time, the next chunk's loads in flight while the current one is
// multiplied.  As in gemm.hip: a load covers two rows x 512 bytes of the weight, the chunk is parked
// in a wave-private piece of LDS and read back as the matrix cores' A operand (v_mfma_f32_16x16x32_bf16:
// lane holds w[lane % 16][8 (lane / 16) ..]); x comes from the caches straight into the B operand, since
// no other wave of the workgroup wants the same piece.  Rows beyond N are read from the last row and
// never stored, K beyond the end is read from valid places and meets zeros of x.  Workgroups start at
// different chunks, so that they do not ask for addresses a whole number of rows apart at every moment,
// and those of one die (every eighth) at different ones too: against starting at the workgroup's number, when
// this was chosen, 4,096 x 4,096 11.1 -> 8.3 us, 8,192 x 4,096 19.2 -> 15.5, 4,672 x 2,048 8.9 -> 8.4.
// gated: the 16 rows are eight gate rows, then the eight up rows that belong to them.
// A wave's products join two running sums by turns: every addition rounds the sum it joins, and from a K of about
// 5,000 on one sum a wave met more of them than the slices of the other form do.  Distance from 64 bits in parts of
// 10^-7 of the result's norm (slices / one sum a wave / two): 1,024 x 5,632 1.41 / 1.62 / 1.22, 1,500 x 8,192
// 1.46 / 1.92 / 1.40, 1,024 x 12,288 1.76 / 2.38 / 1.68, 2,048 x 2,048 1.32 / 1.02 / 0.86; the same time.
// Bound by the reading of the weight.
template <typename TO>
__global__ __launch_bounds__(64 * W) void gemm_cols_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                           TO* __restrict__ y, int M, int N, int K, int ldx, int ldw, int ldy,
                                                           Finish f) {
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
  const bf16_t* xrow = x + static_cast<size_t>(min(r, M - 1)) * ldx;
  const int start = (5 * blockIdx.x + blockIdx.x / 8) % n_chunks;
  auto chunk_at = [&](int i) {
    const int j = i + start;
    return (j >= n_chunks ? j - n_chunks : j) * KC;
  };
  u32x4_t wr[STEPS], xr[STEPS];
  auto fetch_w = [&](int kc) {
    const uint32_t k = 2u * static_cast<uint32_t>(min(kc + 8 * l32, k_last));
#pragma unroll
    for (int j = 0; j < STEPS; ++j)
      wr[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(reinterpret_cast<const char*>(w0) + (wrow[j] + k)));
  };
  auto fetch_x = [&](int kc) {
#pragma unroll
    for (int u = 0; u < STEPS; ++u) xr[u] = *reinterpret_cast<const u32x4_t*>(xrow + min(kc + 32 * u + 8 * g, k_last));
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
#pragma unroll
    for (int u = 0; u < STEPS; ++u) {
      Frag8 b;
      b.u = whole || kc + 32 * u + 8 * g < K ? xr[u] : u32x4_t{0u, 0u, 0u, 0u};
      acc[u % CHAINS] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u].v, b.v, acc[u % CHAINS], 0, 0, 0);
    }
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
    if (f.bias && n0 + c < N)
      s += f.bias_f32 ? static_cast<const float*>(f.bias)[n0 + c] : to_f32<bf16_t>(static_cast<const bf16_t*>(f.bias)[n0 + c]);
    return s;
  };
  if (f.gated) {
    for (int o = threadIdx.x; o < 8 * M; o += 64 * W) {
      const int m = o / 8, c = o % 8;
      const float v = gated_pair(as_output(total(m, c), 1), as_output(total(m, c + 8), 1), f.kind, f.p0, f.p1);
      y[static_cast<size_t>(m) * ldy + n0 / 2 + c] = from_f32<TO>(v);
    }
    return;
  }
  for (int o = threadIdx.x; o < 16 * M; o += 64 * W) {
    const int m = o / 16, c = o % 16;
    if (n0 + c < N) y[static_cast<size_t>(m) * ldy + n0 + c] = from_f32<TO>(total(m, c));
  }
}

static int g_mode = 0;

}  // namespace

// Whether a product of these sizes goes this way; slices_do: the other form would need no kernel of its own
// after it (its consumer adds the slices, or there is one slice only).
// Measured in replayed graphs (us, slices and the kernel that adds them (without it) / this, at 1, 8 and 16 rows of x):
//   plain  1,024 x 1,024    6.8 (4.7) / 3.3    6.9 (4.8) / 3.5    7.3 (5.2) / 3.9
//          2,048 x 2,048    7.4 (5.0) / 4.4    7.8 (5.2) / 4.8    8.4 (5.5) / 5.5
//          3,072 x 2,048    7.8 (5.3) / 4.7    8.2 (5.4) / 5.1    8.7 (5.8) / 6.0
//          4,672 x 2,048    9.9 (6.9) / 6.6    9.5 (7.0) / 7.5   10.1 (7.5) / 8.9
//          2,048 x 5,632   10.5 (7.1) / 7.8   11.2 (7.3) / 9.1   11.9 (7.8) / 10.9
//          3,072 x 4,096   10.1 (6.3) / 7.1   10.5 (6.6) / 7.7   11.2 (7.1) / 9.1
//          6,144 x 2,048    9.3 (6.4) / 7.0    9.5 (6.6) / 7.6   10.3 (7.1) / 9.2
//          4,096 x 4,096   11.4 (7.7) / 8.0   11.5 (7.4) / 8.4   12.1 (7.8) / 10.1
//          2,048 x 8,192   12.8 (7.6) / 9.4   13.9 (7.7) / 11.2  14.4 (7.9) / 13.8
//          8,320 x 2,048   10.8 (8.4) / 8.9   10.6 (8.2) / 10.0  11.4 (8.7) / 12.2
//         16,384 x 2,048   15.3 (13.1) / 13.6 14.8 (12.3) / 13.5 15.5 (12.6) / 16.4
//          8,192 x 4,096   17.4 (14.8) / 13.7 17.4 (14.5) / 14.3 18.0 (14.9) / 17.7
//         12,352 x 4,096   21.1 (18.9) / 20.7 21.1 (18.9) / 23.7 22.0 (19.4) / 30.2
//   gated  4,096 x 2,048    8.4 / 5.5    8.9 / 5.8    9.5 / 6.6     11,264 x 2,048  12.7 / 11.0  12.7 / 11.5  13.4 / 13.5
//         16,384 x 2,048   15.3 / 14.1  15.8 / 15.2  15.5 / 16.6    22,016 x 4,096  33.4 / 33.0  34.1 / 37.2  33.8 / 45.7
// A workgroup of 16 columns reads x once for them, four times as often a column as the other form, and
// ends with a barrier and a few sums: both count the more, the more workgroups a compute unit runs one
// after another, and the first with the rows of x.  So: matrices of up to 13 M elements, and with up to
// 8 rows of x those of up to 36 M whose K is one round of the eight waves.  (These two lines were drawn when a die's
// workgroups still started at few places, which cost the larger matrices most; since then this form is also faster some way
// beyond them, as the table shows.  Four or sixteen waves a workgroup, then too: 4,672 x 2,048 8.0 and 8.7, 16,384 x 2,048
// 16.1 and 19.1, 4,096 x 2,048 6.6 and 6.3.)
// Nor where K and columns are far apart: few columns are few workgroups, whose walk over a long K is not divided any further
// (1,024 x 8,192 at 9 and 16 rows 12.5 / 10.8 and 12.6 / 13.3, 1,024 x 11,008 at 4, 8 and 16 12.7 / 11.4, 13.2 / 13.9 and 13.8 / 17.4); a short K leaves
// waves without a chunk, and from 8,192 columns on a second round of workgroups waits for the first, two a compute unit (with a
// bias 16,384 x 256 6.1 / 5.2, 22,016 x 256 7.0 / 7.2 at 8 rows; 16,384 x 1,024 9.8 / 9.3, 22,016 x 1,024 11.7 / 12.4).
// Where slices would do, this form still saves what starting a second round of workgroups and adding the
// slices cost, in small matrices: a decode step of the 1B shape (qkv 3,072 x 2,048, o-proj 2,048 x 2,048)
// went from 0.84 to 0.80 ms with up to 6.5 M elements; with up to 13 M the delta-rule design's step at eight
// rows (down-proj 2,048 x 5,632) lost what it had gained (12.65 -> 12.82 ms for 16 steps and their prompts).
// Only up to eight rows: at 16 the two are even, and a product that takes attention's
// unmerged splits (which this form does not) has the bits of the one that takes them merged there.
// The lines for K and columns are narrower here (8 rows, with the norm that follows, slices / this: 1,024 x 4,096 8.2 / 9.4,
// 1,536 x 3,072 8.6 / 8.9, 1,024 x 5,632 9.4 / 11.2; one slice: 8,192 x 512 5.3 / 4.3, 12,288 x 512 5.5 / 5.7, 25,344 x 256 4.8 / 8.2,
// 8,208 x 768 6.7 / 5.7).
// Narrow products, of fewer than 1,024 columns, would gain too (256 x 2,048 7.2 / 4.0) and stay where they are:
// there a product has the same bits whether it comes as slices or reduced, which programs that compare the two
// may count on; here its sums run in another order.
extern "C" int yk_gemm_cols_ok(int M, int N, int K, int slices_do) {
  if (M < 1 || M > 16 || K < 8 || K % 8 || N < 1) return 0;
  if (g_mode) return g_mode == 2;
  if (N < 1024) return 0;
  const long long elements = static_cast<long long>(N) * K;
  if (slices_do)
    return M <= 8 && elements <= 6500000 && K >= KC && (K <= W * KC || 2LL * K <= 3LL * N) && (N <= 8192 || N <= 16LL * K);
  if (M > 4 && K > (M <= 12 ? 8192 : 6144)) return 0;
  if (elements <= 13000000) return N <= 64LL * K;
  return M <= 8 && elements <= 36000000 && K <= W * KC && N <= 16LL * K;
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
  const Finish f{gated, kind, p0, p1, bias, bias_dtype == YK_F32};
  const unsigned tiles = (N + 15) / 16;
  if (y_dtype == YK_F32)
    gemm_cols_kernel<float><<<tiles, 64 * W, 0, stream>>>(static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w),
                                                          static_cast<float*>(y), M, N, K, ldx, ldw, ldy, f);
  else
    gemm_cols_kernel<bf16_t><<<tiles, 64 * W, 0, stream>>>(static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w),
                                                           static_cast<bf16_t*>(y), M, N, K, ldx, ldw, ldy, f);
  return yk_check_launch("gemm_cols");
}
