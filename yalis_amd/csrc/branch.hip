// A branch's output joins the residual stream through a norm of its own:
//   residual[n, :] += branch[n, :] / sqrt(mean(branch[n, :]^2) + eps) * w'      (w' = w or 1 + w)
// and, where the engine's activations are narrower than the float32 residual, the new residual
// rounded to the activation dtype is written beside it: the next branch reads the stream itself,
// not a normed copy, so this is the only pass over the row between two branches.
//
// The branch may come as
//   * a tensor [rows, width] in the activation dtype or float32,
//   * the unreduced K slices of a product (float32 [slices, rows, width]; summed in the order of
//     the slices and, with round_sum, rounded as the product's own output would have been),
//   * and / or the rows of a mixture of experts before they are combined: float32
//     [rows * top, width], of which row n takes pair_weight * (the sum of its `top` rows, in
//     order).
// Everything is float32 arithmetic; one workgroup a row, the row parked in LDS between the
// sum of squares and the update.
//
// Beside it: the other arrangement, the stream itself normed after a branch has joined it (yk_sum_norm).
#include <algorithm>
#include <type_traits>

#include "common.h"

// General form: any width, a column a thread, the row parked in LDS.
template <typename TS, typename TW, typename TO>
__global__ __launch_bounds__(256) void norm_add_kernel(
    float* __restrict__ residual, const TS* __restrict__ src, int n_splits, size_t split_stride, int round_sum,
    const float* __restrict__ pairs, int top, float pair_weight, const TW* __restrict__ w, int unit_offset,
    float eps, TO* __restrict__ out, int width) {
  extern __shared__ float row[];  // [width], then 17 floats of scratch
  float* scratch = row + width;
  const size_t n = blockIdx.x;
  float ss = 0.f;
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    float v = 0.f;
    if (src != nullptr) {
      for (int s = 0; s < n_splits; ++s) v += to_f32<TS>(src[s * split_stride + n * width + c]);
      v = as_output(v, round_sum);
    }
    if (pairs != nullptr) {
      float e = 0.f;
      for (int k = 0; k < top; ++k) e += pairs[(n * top + k) * width + c];
      v = fmaf(pair_weight, e, v);
    }
    row[c] = v;
    ss = fmaf(v, v, ss);
  }
  const float total = block_sum(ss, scratch);
  const float inv = 1.f / sqrtf(total / static_cast<float>(width) + eps);
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    const float wv = to_f32<TW>(w[c]) + (unit_offset ? 1.f : 0.f);
    const float r = residual[n * width + c] + row[c] * inv * wv;
    residual[n * width + c] = r;
    if (out != nullptr) out[n * width + c] = from_f32<TO>(r);
  }
}

// Fast form: P pieces of four columns a thread, in registers throughout; the branch's slices, the token's expert rows, the residual and
// the weight are all asked for before any is used (ask_slices in common.h says why that takes care).  Bound by the launch and one trip
// to memory and back each way.  Behind copies of 16 MB and of its input in a replayed graph, four rows of 2,048 in bfloat16 alone / with two expert
// rows, us: with 256 threads whose loads waited one for another 3.6 / 4.6, now 2.0 / 2.3.
constexpr uint32_t ROW_ROUND = 1u << 16, ROW_UNIT = 1u << 17;  // `how`: bits 0-15 slices; 19-23 waves
template <typename TS, typename TW, int P, SlicesAtOnce HOW>
__global__ __launch_bounds__(1024) void norm_add_vec_kernel(float* __restrict__ residual, const TS* __restrict__ src,
                                                            const float* __restrict__ pairs, const TW* __restrict__ w,
                                                            bf16_t* __restrict__ out, int width, uint32_t how, int top,
                                                            uint32_t split_stride, float pair_weight, float eps) {
  __shared__ float scratch[16];
  constexpr int G = P == 4 ? 1 : HOW == kFewRows ? 8 / P : slices_at_once<HOW, P>, GS = sizeof(TS) == 2 ? 1 : G;  // expert rows and slices asked for at once
  const int n_splits = how & 0xffffu, waves = (how >> 19) & 31, round_sum = (how & ROW_ROUND) != 0;
  const size_t n = blockIdx.x;
  float4 rs[P];
  typename Four<TW>::raw wr[P];
  uint32_t at[P];
#pragma unroll
  for (int k = 0; k < P; ++k) at[k] = min(4 * (static_cast<int>(threadIdx.x) + 64 * waves * k), width - 4);
  const TS* p = src + n * width;
  const float* q = pairs + n * top * width;
  typename Four<TS>::raw d[GS][P];
  float4 e[G][P];
  if (src != nullptr) ask_slices<GS, P, TS>(p, at, n_splits, split_stride, d);
  if (pairs != nullptr) ask_slices<G, P, float>(q, at, top, width, e);
#pragma unroll
  for (int k = 0; k < P; ++k) {
    rs[k] = four_at<float>(residual + n * width + at[k]);
    wr[k] = Four<TW>::at(w + at[k]);
  }
  float4 v[P], es[P];
#pragma unroll
  for (int k = 0; k < P; ++k) v[k] = es[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (src != nullptr) {
    join_slices<GS, P, TS>(d, n_splits, v);
    if constexpr (HOW != kOneSlice || P == 4) join_rest<GS, P, TS>(p, at, n_splits, split_stride, v);
#pragma unroll
    for (int k = 0; k < P; ++k)
      v[k] = make_float4(as_output(v[k].x, round_sum), as_output(v[k].y, round_sum), as_output(v[k].z, round_sum), as_output(v[k].w, round_sum));
  }
  if (pairs != nullptr) {
    join_slices<G, P, float>(e, top, es);
    if constexpr (HOW != kOneSlice || P == 4) join_rest<G, P, float>(q, at, top, width, es);
#pragma unroll
    for (int k = 0; k < P; ++k)
      v[k] = make_float4(fmaf(pair_weight, es[k].x, v[k].x), fmaf(pair_weight, es[k].y, v[k].y), fmaf(pair_weight, es[k].z, v[k].z),
                         fmaf(pair_weight, es[k].w, v[k].w));
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < P; ++k) {
    const bool in = 4 * (static_cast<int>(threadIdx.x) + 64 * waves * k) < width;
    ss = in ? fmaf(v[k].x, v[k].x, fmaf(v[k].y, v[k].y, fmaf(v[k].z, v[k].z, fmaf(v[k].w, v[k].w, ss)))) : ss;
  }
  const float total = block_sum_first(ss, scratch, waves);
  const float inv = 1.f / sqrtf(total / static_cast<float>(width) + eps), off = how & ROW_UNIT ? 1.f : 0.f;
#pragma unroll
  for (int k = 0; k < P; ++k) {
    const float4 wv = Four<TW>::wide(wr[k]);
    const float4 r = make_float4(fmaf(v[k].x * inv, wv.x + off, rs[k].x), fmaf(v[k].y * inv, wv.y + off, rs[k].y),
                                 fmaf(v[k].z * inv, wv.z + off, rs[k].z), fmaf(v[k].w * inv, wv.w + off, rs[k].w));
    if (4 * (static_cast<int>(threadIdx.x) + 64 * waves * k) >= width) continue;
    put_four<float>(residual + n * width + at[k], r);
    if (out != nullptr) put_four<bf16_t>(out + n * width + at[k], r);
  }
}

// rows of a float32 stream rounded to the activation dtype (what the first branch of a model reads)
template <typename TO>
__global__ void round_rows_kernel(const float* __restrict__ x, TO* __restrict__ out, size_t total) {
  for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < total;
       i += static_cast<size_t>(gridDim.x) * blockDim.x)
    out[i] = from_f32<TO>(x[i]);
}

extern "C" int yk_round_rows(const float* x, void* out, int out_dtype, size_t total, hipStream_t stream) {
  if (total == 0) return 0;
  YK_REQUIRE(out_dtype == YK_BF16, "round_rows: the narrow dtype is bfloat16");
  const int grid = static_cast<int>(std::min<size_t>((total + 255) / 256, 65535));
  round_rows_kernel<bf16_t><<<grid, 256, 0, stream>>>(x, static_cast<bf16_t*>(out), total);
  return yk_check_launch("round_rows");
}

extern "C" int yk_norm_add(float* residual, const void* src, int src_dtype, int n_splits, int round_sum,
                           const float* pairs, int top, float pair_weight, const void* w, int w_dtype,
                           int unit_offset, float eps, void* out, int out_dtype, int n_rows, int width,
                           hipStream_t stream) {
  YK_REQUIRE(n_rows >= 0 && width > 0, "norm_add: bad sizes");
  YK_REQUIRE(src != nullptr || pairs != nullptr, "norm_add: no branch given");
  YK_REQUIRE(n_splits >= 1 && (n_splits == 1 || src_dtype == YK_F32), "norm_add: unreduced slices must be float32");
  YK_REQUIRE(pairs == nullptr || top >= 1, "norm_add: expert rows need a count per token");
  YK_REQUIRE(width <= 15 * 1024, "norm_add: rows of more than 15,360 elements do not fit the row buffer");
  YK_REQUIRE(out == nullptr || out_dtype == YK_BF16, "norm_add: the rounded copy is bfloat16");
  if (n_rows == 0) return 0;
  const size_t stride = static_cast<size_t>(n_rows) * width;
  const size_t lds = (static_cast<size_t>(width) + 17) * sizeof(float);
  auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool vec = width % 4 == 0 && al(residual) && al(src) && al(pairs) && al(w) && al(out) && n_splits < 1 << 16 && stride < size_t{1} << 32;
  // a piece a thread where rows are few, two where they fill the chip (as add_rmsnorm), never more than 1,024 threads
  const int threads = std::max(64, std::min(1024, ((n_rows >= 1024 ? width / 8 : width / 4) + 63) / 64 * 64));
  const int pieces = (width / 4 + threads - 1) / threads;
  const uint32_t how = static_cast<uint32_t>(n_splits & 0xffff) | (round_sum ? ROW_ROUND : 0u) | (unit_offset ? ROW_UNIT : 0u) |
                       static_cast<uint32_t>(threads / 64) << 19;
  const SlicesAtOnce at_once = slices_how(std::max(n_splits, pairs ? top : 0), n_rows);
#define YK_VEC(TS, TW, P, HOW)                                                                               \
  norm_add_vec_kernel<TS, TW, P, HOW><<<n_rows, threads, 0, stream>>>(                                            \
      residual, static_cast<const TS*>(src), pairs, static_cast<const TW*>(w), static_cast<bf16_t*>(out), width, how, top, \
      static_cast<uint32_t>(stride), pair_weight, eps)
#define YK_CASE(SD, TS, WD, TW)                                                                            \
  if ((src == nullptr || src_dtype == SD) && w_dtype == WD) {                                                \
    if (vec && pieces <= 1 && at_once == kOneSlice) YK_VEC(TS, TW, 1, kOneSlice);                            \
    else if (vec && pieces <= 1 && at_once == kManyRows) YK_VEC(TS, TW, 1, kManyRows);                       \
    else if (vec && pieces <= 1) YK_VEC(TS, TW, 1, kFewRows);                                                \
    else if (vec && pieces <= 2 && at_once == kOneSlice) YK_VEC(TS, TW, 2, kOneSlice);                       \
    else if (vec && pieces <= 2 && at_once == kManyRows) YK_VEC(TS, TW, 2, kManyRows);                       \
    else if (vec && pieces <= 2) YK_VEC(TS, TW, 2, kFewRows);                                                \
    else if (vec) YK_VEC(TS, TW, 4, kOneSlice); /* (one at a time: what the registers hold) */               \
    else                                                                                                     \
      norm_add_kernel<TS, TW, bf16_t><<<n_rows, 256, lds, stream>>>(                                         \
          residual, static_cast<const TS*>(src), n_splits, stride, round_sum, pairs, top, pair_weight,       \
          static_cast<const TW*>(w), unit_offset, eps, static_cast<bf16_t*>(out), width);                    \
    return yk_check_launch("norm_add");                                                                      \
  }
  YK_CASE(YK_F32, float, YK_F32, float)
  YK_CASE(YK_F32, float, YK_BF16, bf16_t)
  YK_CASE(YK_BF16, bf16_t, YK_F32, float)
  YK_CASE(YK_BF16, bf16_t, YK_BF16, bf16_t)
#undef YK_CASE
#undef YK_VEC
  return yk_fail("norm_add: unsupported dtype combination");
}

// ------------------------------------------------------------- the stream normed after the sum
//   b        = branch_scale * (a-term + b-term) * channel weight
//   r        = residual_scale * residual[n, :] + b
//   residual = r / sqrt(mean(r^2) + eps) * w'           (w' = w or 1 + w), and its rounded copy beside it
// A term is a branch's rows (activation dtype, float32, or a product's unreduced slices), as they are or first divided
// by their own root mean square and multiplied by a weight; the second term and the channel weight may be absent.  Both
// terms' sums of squares are reduced together.  One workgroup a row; rows of up to 4,096 elements stay in registers
// between the reductions (VEC: four columns a thread and piece, everything asked for before the first reduction), longer
// or odd ones in LDS.
struct SumTerm {
  const void* src;
  int bf16;  // 1: bfloat16 rows; 0: float32 rows or slices
  int n_splits;
  int round_sum;
  float eps;
  const void* w;  // null: added as it is
};

__device__ __forceinline__ void block_sum2(float& a, float& b, float* scratch) {
  a = wave_sum(a);
  b = wave_sum(b);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, n_waves = blockDim.x / kWave;
  __syncthreads();  // scratch may still be read from an earlier call
  if (lane == 0) scratch[wave] = a, scratch[16 + wave] = b;
  __syncthreads();
  a = row_sum(lane % 16 < n_waves ? scratch[lane % 16] : 0.f);
  b = row_sum(lane % 16 < n_waves ? scratch[16 + lane % 16] : 0.f);
}

__device__ __forceinline__ float sum_term1(const SumTerm& t, size_t at, size_t stride) {
  if (t.bf16) return to_f32<bf16_t>(static_cast<const bf16_t*>(t.src)[at]);
  float v = 0.f;
  for (int s = 0; s < t.n_splits; ++s) v += static_cast<const float*>(t.src)[at + s * stride];
  return as_output(v, t.round_sum);
}

__device__ __forceinline__ float dot4(float4 v) { return fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, v.w * v.w))); }
__device__ __forceinline__ float4 mul4(float4 a, float4 b) { return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w); }
__device__ __forceinline__ float4 scaled4(float4 a, float s) { return make_float4(a.x * s, a.y * s, a.z * s, a.w * s); }

// P: pieces of 4 columns a thread holds; A16: the first term is bfloat16 rows; B: 0 no second term, 1 float32 rows or slices, 2 bfloat16
// rows.  What a row needs is asked for before any of it is used.  Behind copies of 16 MB and of its input, eight rows of 2,048, one bfloat16 term / one of
// eight slices / two bfloat16 terms with their own norms, us: with loads that waited one for another 2.3 / 3.3 / 3.9, now 2.2 / 3.1 / 3.1.
// `how`: bits 0-7 and 8-15 the terms' slices; 19-23 waves; and the bits below
constexpr uint32_t SUM_ROUND_A = 1u << 16, SUM_ROUND_B = 1u << 17, SUM_UNIT = 1u << 18, SUM_AW = 1u << 24, SUM_BW = 1u << 25, SUM_CW = 1u << 26;
template <typename TW, bool A16, int B, int P, SlicesAtOnce HOW>
__global__ __launch_bounds__(1024) void sum_norm_vec_kernel(float* __restrict__ residual, const void* __restrict__ a_src,
                                                            const void* __restrict__ b_src, const TW* __restrict__ w,
                                                            bf16_t* __restrict__ out, int width, uint32_t how, uint32_t stride,
                                                            float residual_scale, const TW* __restrict__ aw, const TW* __restrict__ bw,
                                                            const TW* __restrict__ cw, float branch_scale, float eps, float a_eps,
                                                            float b_eps) {
  using TA = std::conditional_t<A16, bf16_t, float>;
  using TB = std::conditional_t<B == 2, bf16_t, float>;
  constexpr int G = HOW == kFewRows ? 8 : HOW == kManyRows ? 4 : 1, GA = A16 ? 1 : G, GB = B != 1 ? 1 : G;  // slices asked for at once
  __shared__ float scratch[3][16];
  const int na = how & 0xff, nb = (how >> 8) & 0xff, waves = (how >> 19) & 31;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const size_t n = blockIdx.x;
  uint32_t at[P];
  float4 rs[P];
  typename Four<TW>::raw wn[P], wc[P], wa[P], wb[P];
  const TA* pa = static_cast<const TA*>(a_src) + n * width;
  const TB* pb = static_cast<const TB*>(b_src) + n * width;
  typename Four<TA>::raw da[GA][P];
  typename Four<TB>::raw db[GB][P];
#pragma unroll
  for (int k = 0; k < P; ++k) at[k] = min(4 * (static_cast<int>(threadIdx.x) + 64 * waves * k), width - 4);
  ask_slices<GA, P, TA>(pa, at, na, stride, da);
  if (B) ask_slices<GB, P, TB>(pb, at, nb, stride, db);
#pragma unroll
  for (int k = 0; k < P; ++k) {
    rs[k] = four_at<float>(residual + n * width + at[k]);
    wn[k] = Four<TW>::at(w + at[k]);
    wc[k] = wa[k] = wb[k] = Four<TW>::all(1.f);
  }
  arguments_now(aw, bw, cw);
  if (how & SUM_AW) {
#pragma unroll
    for (int k = 0; k < P; ++k) wa[k] = Four<TW>::at(aw + at[k]);
  }
  if (B && (how & SUM_BW)) {
#pragma unroll
    for (int k = 0; k < P; ++k) wb[k] = Four<TW>::at(bw + at[k]);
  }
  if (how & SUM_CW) {
#pragma unroll
    for (int k = 0; k < P; ++k) wc[k] = Four<TW>::at(cw + at[k]);
  }
  float4 a[P], b[P];
  auto term = [&](auto& d, auto p, int slices, int round_sum, float4 (&s)[P], auto type, auto group) {
    using T = decltype(type);
    constexpr int G = decltype(group)::value;
#pragma unroll
    for (int k = 0; k < P; ++k) s[k] = make_float4(0.f, 0.f, 0.f, 0.f);
    join_slices<G, P, T>(d, slices, s);
    if constexpr (HOW != kOneSlice) join_rest<G, P, T>(p, at, slices, stride, s);
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int k = 0; k < P; ++k)
        s[k] = make_float4(as_output(s[k].x, round_sum), as_output(s[k].y, round_sum), as_output(s[k].z, round_sum), as_output(s[k].w, round_sum));
    }
  };
  term(da, pa, na, (how & SUM_ROUND_A) != 0, a, TA{}, std::integral_constant<int, GA>{});
  if (B) term(db, pb, nb, (how & SUM_ROUND_B) != 0, b, TB{}, std::integral_constant<int, GB>{});
  float ia = 1.f, ib = 1.f;
  if (how & (SUM_AW | SUM_BW)) {
    float sa = 0.f, sb = 0.f;
#pragma unroll
    for (int k = 0; k < P; ++k) {
      const bool in = 4 * (static_cast<int>(threadIdx.x) + 64 * waves * k) < width;
      sa += in ? dot4(a[k]) : 0.f;
      if (B) sb += in ? dot4(b[k]) : 0.f;
    }
    sa = wave_sum(sa);
    if (B) sb = wave_sum(sb);
    if (lane == 0) scratch[0][wave] = sa, scratch[1][wave] = sb;
    __syncthreads();
    sa = row_sum(lane % 16 < waves ? scratch[0][lane % 16] : 0.f);
    sb = row_sum(lane % 16 < waves ? scratch[1][lane % 16] : 0.f);
    if (how & SUM_AW) ia = 1.f / sqrtf(sa / static_cast<float>(width) + a_eps);
    if (B && (how & SUM_BW)) ib = 1.f / sqrtf(sb / static_cast<float>(width) + b_eps);
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < P; ++k) {
    float4 v = scaled4(mul4(a[k], Four<TW>::wide(wa[k])), ia);
    if (B) {
      const float4 u = mul4(b[k], Four<TW>::wide(wb[k]));
      v = make_float4(fmaf(u.x, ib, v.x), fmaf(u.y, ib, v.y), fmaf(u.z, ib, v.z), fmaf(u.w, ib, v.w));
    }
    v = mul4(scaled4(v, branch_scale), Four<TW>::wide(wc[k]));
    rs[k] = make_float4(fmaf(residual_scale, rs[k].x, v.x), fmaf(residual_scale, rs[k].y, v.y), fmaf(residual_scale, rs[k].z, v.z),
                        fmaf(residual_scale, rs[k].w, v.w));
    ss += 4 * (static_cast<int>(threadIdx.x) + 64 * waves * k) < width ? dot4(rs[k]) : 0.f;
  }
  ss = block_sum_first(ss, scratch[2], waves);
  const float inv = 1.f / sqrtf(ss / static_cast<float>(width) + eps);
  const float off = how & SUM_UNIT ? 1.f : 0.f;
#pragma unroll
  for (int k = 0; k < P; ++k) {
    const float4 wv = Four<TW>::wide(wn[k]);
    const float4 r = make_float4(rs[k].x * inv * (wv.x + off), rs[k].y * inv * (wv.y + off), rs[k].z * inv * (wv.z + off),
                                 rs[k].w * inv * (wv.w + off));
    if (4 * (static_cast<int>(threadIdx.x) + 64 * waves * k) >= width) continue;
    put_four<float>(residual + n * width + at[k], r);
    if (out != nullptr) put_four<bf16_t>(out + n * width + at[k], r);
  }
}

template <typename TW>
__global__ __launch_bounds__(256) void sum_norm_kernel(float* __restrict__ residual, SumTerm ta, SumTerm tb, int has_b, size_t stride,
                                                       float branch_scale, const TW* __restrict__ cw, float residual_scale,
                                                       const TW* __restrict__ w, int unit_offset, float eps,
                                                       bf16_t* __restrict__ out, int width) {
  extern __shared__ float row[];  // [width] (and [width] for a second term), then 34 floats of scratch
  float* second = row + width;
  float* scratch = row + (has_b ? 2 : 1) * static_cast<size_t>(width);
  const size_t n = blockIdx.x;
  float sa = 0.f, sb = 0.f;
  for (int c = threadIdx.x; c < width; c += blockDim.x) {  // (every thread keeps to its own columns throughout)
    const float a = sum_term1(ta, n * width + c, stride);
    row[c] = a;
    sa = fmaf(a, a, sa);
    if (has_b) {
      const float b = sum_term1(tb, n * width + c, stride);
      second[c] = b;
      sb = fmaf(b, b, sb);
    }
  }
  block_sum2(sa, sb, scratch);
  const float ia = ta.w != nullptr ? 1.f / sqrtf(sa / static_cast<float>(width) + ta.eps) : 1.f;
  const float ib = has_b && tb.w != nullptr ? 1.f / sqrtf(sb / static_cast<float>(width) + tb.eps) : 1.f;
  float ss = 0.f, none = 0.f;
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    float v = row[c] * (ta.w != nullptr ? to_f32<TW>(static_cast<const TW*>(ta.w)[c]) : 1.f) * ia;
    if (has_b) v = fmaf(second[c] * (tb.w != nullptr ? to_f32<TW>(static_cast<const TW*>(tb.w)[c]) : 1.f), ib, v);
    v *= branch_scale;
    if (cw != nullptr) v *= to_f32<TW>(cw[c]);
    const float r = fmaf(residual_scale, residual[n * width + c], v);
    row[c] = r;
    ss = fmaf(r, r, ss);
  }
  block_sum2(ss, none, scratch);
  const float inv = 1.f / sqrtf(ss / static_cast<float>(width) + eps);
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    const float r = row[c] * inv * (to_f32<TW>(w[c]) + (unit_offset ? 1.f : 0.f));
    residual[n * width + c] = r;
    if (out != nullptr) out[n * width + c] = f32_to_bf16(r);
  }
}

// Terms a and b (b_src null: one term): dtype, slices, whether their sum is rounded, eps and weight (null: as it is).
// All weights share w_dtype.
extern "C" int yk_sum_norm(float* residual, const void* a_src, int a_dtype, int a_splits, int a_round, float a_eps, const void* a_w,
                           const void* b_src, int b_dtype, int b_splits, int b_round, float b_eps, const void* b_w,
                           float branch_scale, const void* channel_w, float residual_scale, const void* w, int w_dtype,
                           int unit_offset, float eps, void* out, int n_rows, int width, hipStream_t stream) {
  YK_REQUIRE(n_rows >= 0 && width > 0 && residual != nullptr && w != nullptr, "sum_norm: bad sizes");
  YK_REQUIRE(a_src != nullptr, "sum_norm: no branch given");
  YK_REQUIRE(a_splits >= 1 && (a_splits == 1 || a_dtype == YK_F32) && (b_src == nullptr || (b_splits >= 1 && (b_splits == 1 || b_dtype == YK_F32))),
             "sum_norm: unreduced slices must be float32");
  YK_REQUIRE((b_src != nullptr ? 2 : 1) * static_cast<long>(width) <= 15 * 1024, "sum_norm: the rows do not fit the row buffer");
  if (n_rows == 0) return 0;
  const size_t stride = static_cast<size_t>(n_rows) * width;
  const SumTerm ta{a_src, a_dtype == YK_BF16, a_splits, a_round, a_eps, a_w};
  const SumTerm tb{b_src, b_dtype == YK_BF16, b_splits, b_round, b_eps, b_w};
  const int has_b = b_src != nullptr;
  auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool vec = width % 4 == 0 && width <= 4096 && al(residual) && al(a_src) && al(b_src) && al(a_w) && al(b_w) && al(channel_w) &&
                   al(w) && al(out) && a_splits <= 255 && b_splits <= 255 && stride < size_t{1} << 32;
  // a piece a thread for few rows, two where rows fill the chip (eight rows of 2,048: 6.2 -> 4.2 us with twice the threads)
  const int threads = n_rows >= 1024 ? (width / 4 + 127) / 128 * 64 : (width / 4 + 63) / 64 * 64, pieces = 4 * threads < width ? 2 : 1;
  const uint32_t how = static_cast<uint32_t>(a_splits & 0xff) | static_cast<uint32_t>(b_splits & 0xff) << 8 | (a_round ? SUM_ROUND_A : 0u) |
                       (b_round ? SUM_ROUND_B : 0u) | (unit_offset ? SUM_UNIT : 0u) | static_cast<uint32_t>(threads / 64) << 19 |
                       (a_w ? SUM_AW : 0u) | (has_b && b_w ? SUM_BW : 0u) | (channel_w ? SUM_CW : 0u);
  const SlicesAtOnce at_once = slices_how(std::max(a_splits, has_b ? b_splits : 1), n_rows);
#define YK_VEC(TW, A16, B, P, HOW)                                                                                         \
  sum_norm_vec_kernel<TW, A16, B, P, (A16 && B != 1 ? kOneSlice : HOW)><<<n_rows, threads, 0, stream>>>(                   \
      residual, a_src, b_src, static_cast<const TW*>(w), static_cast<bf16_t*>(out), width, how, static_cast<uint32_t>(stride), residual_scale, \
      static_cast<const TW*>(a_w), static_cast<const TW*>(b_w), static_cast<const TW*>(channel_w), branch_scale, eps, a_eps, b_eps)
#define YK_VEC_P(TW, A16, B)                                                         \
  if (pieces == 1 && at_once == kOneSlice) YK_VEC(TW, A16, B, 1, kOneSlice);         \
  else if (pieces == 1 && at_once == kManyRows) YK_VEC(TW, A16, B, 1, kManyRows);    \
  else if (pieces == 1) YK_VEC(TW, A16, B, 1, kFewRows);                             \
  else if (at_once == kOneSlice) YK_VEC(TW, A16, B, 2, kOneSlice);                   \
  else YK_VEC(TW, A16, B, 2, kManyRows) /* (1,024 rows and more) */
#define YK_VEC_B(TW, A16)                 \
  if (!has_b) { YK_VEC_P(TW, A16, 0); }   \
  else if (tb.bf16) { YK_VEC_P(TW, A16, 2); } \
  else { YK_VEC_P(TW, A16, 1); }
#define YK_CASE(WD, TW)                                                                                                    \
  if (w_dtype == WD) {                                                                                                     \
    if (vec && ta.bf16) {                                                                                                  \
      YK_VEC_B(TW, true)                                                                                                   \
    } else if (vec) {                                                                                                      \
      YK_VEC_B(TW, false)                                                                                                  \
    } else {                                                                                                               \
      sum_norm_kernel<TW><<<n_rows, 256, ((has_b ? 2 : 1) * static_cast<size_t>(width) + 34) * sizeof(float), stream>>>(   \
          residual, ta, tb, has_b, stride, branch_scale, static_cast<const TW*>(channel_w), residual_scale,                \
          static_cast<const TW*>(w), unit_offset, eps, static_cast<bf16_t*>(out), width);                                  \
    }                                                                                                                      \
    return yk_check_launch("sum_norm");                                                                                    \
  }
  YK_CASE(YK_F32, float)
  YK_CASE(YK_BF16, bf16_t)
#undef YK_CASE
#undef YK_VEC_B
#undef YK_VEC_P
#undef YK_VEC
  return yk_fail("sum_norm: unsupported weight dtype");
}
