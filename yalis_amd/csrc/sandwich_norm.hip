// Norms on both sides of a branch, in one pass over a row of the residual stream:
//
//   t        = post(branch[n, :])            (or branch[n, :] itself without a post-norm)
//   r        = residual[row, :] + scale * t  (written back unless rows are gathered)
//   out[n,:] = pre(r)                        (left out when nobody reads the stream next)
//
// post and pre are norms with weight and optional bias:
//   centred:   (x - mean) / sqrt(mean((x - mean)^2) + eps) * w + b      (a layer norm)
//   otherwise:  x / sqrt(mean(x^2) + eps) * w + b                       (an RMS norm)
// Mean and variance are taken in two passes over the row, which is parked in LDS; everything is
// float32, the output rounded once.  The branch may be a tensor in the activation dtype or
// float32, or the unreduced K slices of a product (float32 [slices, rows, width], summed in
// order and, with round_sum, rounded as the product's own output would have been).  Without a
// residual the kernel is the plain norm of the branch's rows.  `rows` (one index per output
// row) picks rows of residual and branch and leaves the residual as it is: the final norm on
// the rows whose logits are wanted.
//
// Beside it: an elementwise activation of a product's output (relu squared, silu, gelu) and the
// multiplication of float32 rows by a constant, with an optional soft cap.
#include <algorithm>

#include "common.h"

struct NormStats {
  float mean, inv;
};

// mean (0 when not centred) and 1 / sqrt(variance + eps) of row[0 .. width), every thread its own columns
__device__ __forceinline__ NormStats row_stats(const float* row, int width, int center, float eps, float* scratch) {
  float mean = 0.f;
  if (center) {
    float s = 0.f;
    for (int c = threadIdx.x; c < width; c += blockDim.x) s += row[c];
    mean = block_sum(s, scratch) / static_cast<float>(width);
  }
  float ss = 0.f;
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    const float d = row[c] - mean;
    ss = fmaf(d, d, ss);
  }
  const float var = block_sum(ss, scratch) / static_cast<float>(width);
  return {mean, 1.f / sqrtf(var + eps)};
}

template <typename TS, typename TW, typename TO>
__global__ __launch_bounds__(256) void sandwich_norm_kernel(
    float* __restrict__ residual, const TS* __restrict__ src, int n_splits, size_t split_stride, int round_sum,
    const TW* __restrict__ wa, const TW* __restrict__ ba, float eps_a, int center_a, int has_post, float scale,
    const TW* __restrict__ wb, const TW* __restrict__ bb, float eps_b, int center_b, int has_pre,
    const int32_t* __restrict__ rows, TO* __restrict__ out, int width) {
  extern __shared__ float row[];  // [width], then 17 floats of scratch
  float* scratch = row + width;
  const size_t n = blockIdx.x;
  const size_t r = rows != nullptr ? static_cast<size_t>(rows[n]) : n;
  if (src != nullptr) {
    for (int c = threadIdx.x; c < width; c += blockDim.x) {
      float v = 0.f;
      for (int s = 0; s < n_splits; ++s) v += to_f32<TS>(src[s * split_stride + r * width + c]);
      row[c] = as_output(v, round_sum);
    }
    if (has_post) {
      const NormStats st = row_stats(row, width, center_a, eps_a, scratch);
      for (int c = threadIdx.x; c < width; c += blockDim.x) {
        float t = (row[c] - st.mean) * st.inv * to_f32<TW>(wa[c]);
        if (ba != nullptr) t += to_f32<TW>(ba[c]);
        row[c] = t;
      }
    }
  }
  if (residual != nullptr) {
    for (int c = threadIdx.x; c < width; c += blockDim.x) {
      float v = residual[r * width + c];
      if (src != nullptr) {
        v = fmaf(scale, row[c], v);
        if (rows == nullptr) residual[r * width + c] = v;
      }
      row[c] = v;
    }
  }
  if (!has_pre) return;
  const NormStats st = row_stats(row, width, center_b, eps_b, scratch);
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    float t = (row[c] - st.mean) * st.inv * to_f32<TW>(wb[c]);
    if (bb != nullptr) t += to_f32<TW>(bb[c]);
    out[n * width + c] = from_f32<TO>(t);
  }
}

// The same for rows of up to 4,096 elements in pieces of four, a thread holding P of them in registers: everything a thread reads (the
// branch's slices, the residual, both norms' weights and biases) is asked for before any of it is used, and every reduction has a scratch
// of its own and one barrier.  Behind copies of 16 MB and of its input, eight rows of 4,096 as eight slices / in bfloat16, a centred
// norm after and a plain one before, us: with loads that waited one for another 5.5 / 4.7, now 5.0 / 4.1.
template <int P>
__device__ __forceinline__ NormStats piece_stats(const float4* v, const bool* in, int width, bool center, float eps, float (*scratch)[16], int waves) {
  float mean = 0.f;
  if (center) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < P; ++k) s += in[k] ? (v[k].x + v[k].y) + (v[k].z + v[k].w) : 0.f;
    mean = block_sum_first(s, scratch[0], waves) / static_cast<float>(width);
  }
  float ss = 0.f;
#pragma unroll
  for (int k = 0; k < P; ++k) {
    const float a = v[k].x - mean, b = v[k].y - mean, c = v[k].z - mean, d = v[k].w - mean;
    ss = in[k] ? fmaf(a, a, fmaf(b, b, fmaf(c, c, fmaf(d, d, ss)))) : ss;
  }
  return {mean, 1.f / sqrtf(block_sum_first(ss, scratch[1], waves) / static_cast<float>(width) + eps)};
}

__device__ __forceinline__ float4 piece_norm(float4 v, NormStats st, float4 w, float4 b) {
  return make_float4(fmaf((v.x - st.mean) * st.inv, w.x, b.x), fmaf((v.y - st.mean) * st.inv, w.y, b.y),
                     fmaf((v.z - st.mean) * st.inv, w.z, b.z), fmaf((v.w - st.mean) * st.inv, w.w, b.w));
}

// `how`: bits 0-15 slices; 19-23 waves; and these
constexpr uint32_t SN_ROUND = 1u << 16, SN_CENTER_A = 1u << 17, SN_CENTER_B = 1u << 18, SN_ROWS = 1u << 24, SN_BIAS_A = 1u << 25,
                   SN_BIAS_B = 1u << 26;
template <typename TS, typename TW, typename TO, int P, SlicesAtOnce HOW>
__global__ __launch_bounds__(1024) void sandwich_norm_vec_kernel(float* __restrict__ residual, const TS* __restrict__ src,
                                                                 const TW* __restrict__ wa, const TW* __restrict__ wb,
                                                                 TO* __restrict__ out, int width, uint32_t how, uint32_t split_stride,
                                                                 float scale, const TW* __restrict__ ba, const TW* __restrict__ bb,
                                                                 const int32_t* __restrict__ rows, float eps_a, float eps_b) {
  constexpr int SL = HOW == kFewRows ? 8 / P : slices_at_once<HOW, P>;  // slices asked for at once
  __shared__ float scratch[4][16];
  const int n_splits = how & 0xffffu, waves = (how >> 19) & 31, round_sum = (how & SN_ROUND) != 0;
  const size_t n = blockIdx.x;
  size_t r = n;
  if (how & SN_ROWS) r = rows[n];
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 br[P], rs[P];
  typename Four<TW>::raw wra[P], bra[P], wrb[P], brb[P];
  typename Four<TS>::raw d[SL][P];
  uint32_t at[P];
  bool in[P];
#pragma unroll
  for (int k = 0; k < P; ++k) {
    const int c = 4 * (static_cast<int>(threadIdx.x) + 64 * waves * k);
    in[k] = c < width;
    at[k] = min(c, width - 4);
    rs[k] = br[k] = zero;
    wra[k] = bra[k] = wrb[k] = brb[k] = Four<TW>::all(0.f);
  }
  const TS* p = src + r * width;
  if (src != nullptr) ask_slices<SL, P, TS>(p, at, n_splits, split_stride, d);
  if (residual != nullptr) {
#pragma unroll
    for (int k = 0; k < P; ++k) rs[k] = four_at<float>(residual + r * width + at[k]);
  }
  if (wa != nullptr) {
#pragma unroll
    for (int k = 0; k < P; ++k) wra[k] = Four<TW>::at(wa + at[k]);
  }
  if (wb != nullptr) {
#pragma unroll
    for (int k = 0; k < P; ++k) wrb[k] = Four<TW>::at(wb + at[k]);
  }
  arguments_now(ba, bb);
  if (how & SN_BIAS_A) {
#pragma unroll
    for (int k = 0; k < P; ++k) bra[k] = Four<TW>::at(ba + at[k]);
  }
  if (how & SN_BIAS_B) {
#pragma unroll
    for (int k = 0; k < P; ++k) brb[k] = Four<TW>::at(bb + at[k]);
  }
  if (src != nullptr) {
    join_slices<SL, P, TS>(d, n_splits, br);
    if constexpr (HOW != kOneSlice) join_rest<SL, P, TS>(p, at, n_splits, split_stride, br);
#pragma unroll
    for (int k = 0; k < P; ++k)
      br[k] = make_float4(as_output(br[k].x, round_sum), as_output(br[k].y, round_sum), as_output(br[k].z, round_sum),
                          as_output(br[k].w, round_sum));
    if (wa != nullptr) {
      const NormStats st = piece_stats<P>(br, in, width, how & SN_CENTER_A, eps_a, scratch, waves);
#pragma unroll
      for (int k = 0; k < P; ++k) br[k] = piece_norm(br[k], st, Four<TW>::wide(wra[k]), Four<TW>::wide(bra[k]));
    }
  }
  if (residual != nullptr) {
    if (src != nullptr) {
#pragma unroll
      for (int k = 0; k < P; ++k) {
        rs[k] = make_float4(fmaf(scale, br[k].x, rs[k].x), fmaf(scale, br[k].y, rs[k].y), fmaf(scale, br[k].z, rs[k].z),
                            fmaf(scale, br[k].w, rs[k].w));
        if (!(how & SN_ROWS) && in[k]) put_four<float>(residual + r * width + at[k], rs[k]);
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < P; ++k) rs[k] = br[k];
  }
  if (wb == nullptr) return;
  const NormStats st = piece_stats<P>(rs, in, width, how & SN_CENTER_B, eps_b, scratch + 2, waves);
#pragma unroll
  for (int k = 0; k < P; ++k)
    if (in[k]) put_four<TO>(out + n * width + at[k], piece_norm(rs[k], st, Four<TW>::wide(wrb[k]), Four<TW>::wide(brb[k])));
}

// src_rows: rows of residual and of every slice of src (the stride between slices); n_rows: rows of out.
extern "C" int yk_sandwich_norm(float* residual, const void* src, int src_dtype, int n_splits, int round_sum, int src_rows,
                                const void* wa, const void* ba, float eps_a, int center_a, float scale, const void* wb,
                                const void* bb, float eps_b, int center_b, int w_dtype, const int32_t* rows, void* out,
                                int out_dtype, int n_rows, int width, hipStream_t stream) {
  YK_REQUIRE(n_rows >= 0 && width > 0 && src_rows >= 0, "sandwich_norm: bad sizes");
  YK_REQUIRE(residual != nullptr || src != nullptr, "sandwich_norm: neither a residual nor a branch");
  YK_REQUIRE(n_splits >= 1 && (n_splits == 1 || src_dtype == YK_F32), "sandwich_norm: unreduced slices must be float32");
  YK_REQUIRE(width <= 15 * 1024, "sandwich_norm: rows of more than 15,360 elements do not fit the row buffer");
  YK_REQUIRE((wb != nullptr) == (out != nullptr), "sandwich_norm: an output needs a norm, and a norm an output");
  YK_REQUIRE(wa == nullptr || src != nullptr, "sandwich_norm: a branch's norm needs the branch");
  if (n_rows == 0) return 0;
  const size_t stride = static_cast<size_t>(src_rows) * width;
  const size_t lds = (static_cast<size_t>(width) + 17) * sizeof(float);
  auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool vec = width % 4 == 0 && width <= 4096 && al(residual) && al(src) && al(wa) && al(ba) && al(wb) &&
                   al(bb) && al(out) && n_splits < 1 << 16 && stride < size_t{1} << 32;
  // a piece a thread for few rows, two where rows fill the chip: eight rows of 4,096 11.1 -> 6.2 us, 2,048 rows of 2,048 24 -> 15 us
  // against 256 threads with up to four pieces each (whose slices were then added one round trip after the other)
  const int threads = n_rows >= 1024 ? (width / 4 + 127) / 128 * 64 : (width / 4 + 63) / 64 * 64, pieces = 4 * threads < width ? 2 : 1;
  const uint32_t how = static_cast<uint32_t>(n_splits & 0xffff) | (round_sum ? SN_ROUND : 0u) | (center_a ? SN_CENTER_A : 0u) |
                       (center_b ? SN_CENTER_B : 0u) | static_cast<uint32_t>(threads / 64) << 19 | (rows ? SN_ROWS : 0u) |
                       (wa && ba ? SN_BIAS_A : 0u) | (wb && bb ? SN_BIAS_B : 0u);
  const SlicesAtOnce at_once = slices_how(n_splits, n_rows);
#define YK_VEC(TS, TW, TO, P, HOW)                                                                                \
  sandwich_norm_vec_kernel<TS, TW, TO, P, (sizeof(TS) == 2 ? kOneSlice : HOW)><<<n_rows, threads, 0, stream>>>(                                        \
      residual, static_cast<const TS*>(src), static_cast<const TW*>(wa), static_cast<const TW*>(wb), static_cast<TO*>(out), width, how, \
      static_cast<uint32_t>(stride), scale, static_cast<const TW*>(ba), static_cast<const TW*>(bb), rows, eps_a, eps_b)
#define YK_CASE(SD, TS, WD, TW, OD, TO)                                                                           \
  if ((src == nullptr || src_dtype == SD) && w_dtype == WD && (out == nullptr || out_dtype == OD)) {              \
    if (vec && pieces == 1 && at_once == kOneSlice) YK_VEC(TS, TW, TO, 1, kOneSlice);                             \
    else if (vec && pieces == 1 && at_once == kManyRows) YK_VEC(TS, TW, TO, 1, kManyRows);                        \
    else if (vec && pieces == 1) YK_VEC(TS, TW, TO, 1, kFewRows);                                                 \
    else if (vec && at_once == kOneSlice) YK_VEC(TS, TW, TO, 2, kOneSlice);                                       \
    else if (vec) YK_VEC(TS, TW, TO, 2, kManyRows); /* (1,024 rows and more) */                                   \
    else                                                                                                          \
    sandwich_norm_kernel<TS, TW, TO><<<n_rows, 256, lds, stream>>>(                                               \
        residual, static_cast<const TS*>(src), n_splits, stride, round_sum, static_cast<const TW*>(wa),           \
        static_cast<const TW*>(ba), eps_a, center_a, wa != nullptr, scale, static_cast<const TW*>(wb),            \
        static_cast<const TW*>(bb), eps_b, center_b, wb != nullptr, rows, static_cast<TO*>(out), width);          \
    return yk_check_launch("sandwich_norm");                                                                      \
  }
  YK_CASE(YK_F32, float, YK_F32, float, YK_F32, float)
  YK_CASE(YK_F32, float, YK_F32, float, YK_BF16, bf16_t)
  YK_CASE(YK_F32, float, YK_BF16, bf16_t, YK_BF16, bf16_t)
  YK_CASE(YK_BF16, bf16_t, YK_BF16, bf16_t, YK_BF16, bf16_t)
  YK_CASE(YK_BF16, bf16_t, YK_F32, float, YK_BF16, bf16_t)
  YK_CASE(YK_F32, float, YK_BF16, bf16_t, YK_F32, float)
#undef YK_CASE
#undef YK_VEC
  return yk_fail("sandwich_norm: unsupported dtype combination");
}

// ------------------------------------------------------------------------------ activation
// kinds: 0 silu, 1 gelu (tanh form), 2 the square of relu
template <typename TS, typename TO>
__global__ void activation_kernel(const TS* __restrict__ src, int n_splits, size_t split_stride, int round_sum, int kind,
                                  TO* __restrict__ out, size_t total) {
  for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < total;
       i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    float v = 0.f;
    for (int s = 0; s < n_splits; ++s) v += to_f32<TS>(src[s * split_stride + i]);
    v = as_output(v, round_sum);
    float y;
    if (kind == 2) {
      const float p = fmaxf(v, 0.f);
      y = p * p;
    } else {
      y = act_apply(v, kind);
    }
    out[i] = from_f32<TO>(y);
  }
}

// The same, four elements a thread; all its slices (up to 16) asked for at once where the launch is small (2,048 rows of 8,192: 39 -> 18 us).
template <typename TS, typename TO, SlicesAtOnce HOW>
__global__ __launch_bounds__(256) void activation_vec_kernel(const TS* __restrict__ src, int n_splits, size_t split_stride, int round_sum, int kind,
                                                             TO* __restrict__ out, size_t pieces) {
  const size_t first = blockIdx.x * static_cast<size_t>(256);
  const uint32_t at[1] = {4 * static_cast<uint32_t>(min(static_cast<size_t>(threadIdx.x), pieces - 1 - first))};
  float4 v[1];
  sum_slices<HOW, 1, TS>(src + 4 * first, at, n_splits, split_stride, v);
  if (first + threadIdx.x < pieces)
    put_four<TO>(out + 4 * first + at[0], make_float4(act_plain(as_output(v[0].x, round_sum), kind), act_plain(as_output(v[0].y, round_sum), kind),
                                                      act_plain(as_output(v[0].z, round_sum), kind), act_plain(as_output(v[0].w, round_sum), kind)));
}

extern "C" int yk_activation(const void* src, int src_dtype, int n_splits, int round_sum, int kind, void* out, int out_dtype,
                             size_t total, hipStream_t stream) {
  YK_REQUIRE(kind >= 0 && kind <= 2, "activation: unknown kind");
  YK_REQUIRE(n_splits >= 1 && (n_splits == 1 || src_dtype == YK_F32), "activation: unreduced slices must be float32");
  if (total == 0) return 0;
  const int grid = static_cast<int>(std::min<size_t>((total + 255) / 256, 1 << 20));
  const bool vec = total % 4 == 0 && total < (1ull << 40) && (reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
#define YK_VEC(TS, TO, HOW)                                                                                         \
  activation_vec_kernel<TS, TO, HOW><<<(total / 4 + 255) / 256, 256, 0, stream>>>(                                 \
      static_cast<const TS*>(src), n_splits, total, round_sum, kind, static_cast<TO*>(out), total / 4)
#define YK_CASE(SD, TS, OD, TO)                                                                                    \
  if (src_dtype == SD && out_dtype == OD) {                                                                        \
    if (vec && n_splits == 1) YK_VEC(TS, TO, kOneSlice);                                                           \
    else if (vec && total > 1 << 18) YK_VEC(TS, TO, (sizeof(TS) == 2 ? kOneSlice : kManyRows));                    \
    else if (vec) YK_VEC(TS, TO, (sizeof(TS) == 2 ? kOneSlice : kFewRows));                                        \
    else                                                                                                           \
      activation_kernel<TS, TO><<<grid, 256, 0, stream>>>(static_cast<const TS*>(src), n_splits, total, round_sum, kind, \
                                                          static_cast<TO*>(out), total);                           \
    return yk_check_launch("activation");                                                                          \
  }
  YK_CASE(YK_F32, float, YK_F32, float)
  YK_CASE(YK_F32, float, YK_BF16, bf16_t)
  YK_CASE(YK_BF16, bf16_t, YK_BF16, bf16_t)
#undef YK_CASE
#undef YK_VEC
  return yk_fail("activation: unsupported dtype combination");
}

// x *= s; with a cap, x = cap tanh(x s / cap)
__global__ void scale_rows_kernel(float* __restrict__ x, float s, float cap, size_t total) {
  for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < total;
       i += static_cast<size_t>(gridDim.x) * blockDim.x) {
    const float v = x[i] * s;
    x[i] = cap > 0.f ? cap * tanhf(v / cap) : v;
  }
}

extern "C" int yk_scale_rows(float* x, float s, float cap, size_t total, hipStream_t stream) {
  YK_REQUIRE(cap >= 0.f, "scale_rows: a cap is positive, 0 for none");
  if (total == 0) return 0;
  const int grid = static_cast<int>(std::min<size_t>((total + 255) / 256, 1 << 20));
  scale_rows_kernel<<<grid, 256, 0, stream>>>(x, s, cap, total);
  return yk_check_launch("scale_rows");
}
