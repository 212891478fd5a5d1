// Attention over one latent row per token.  A page row holds [c (kv_rank) | kr (rot_dim)]: the
// normed latent from which every head's keys and values are made, and one rotated key part
// shared by the heads.  The up-projections are applied to the queries and to the attention's
// result instead of to the cached rows:
//   score_h(i, j) = ([W_uk,h^T q_h,i | turn(qr_h,i)] . [c_j | kr_j]) * scale        (float32)
//   o_h,i         = W_uv,h (sum_j softmax_j(score_h(i, .)) c_j)
// so the pages are read as they are, all heads against the same rows.
//
// Three kernels:
//   * latent_prepare: from the stacked down-projection's rows, the normed query latent, and the
//     token's page row (normed latent, rotated key part);
//   * head_linear: per head x[n, h, :in] . W[h] (W [heads][in][out]), with optionally a tail of
//     every head copied behind the product turned by the token's position (queries into the
//     latent's space) or a sigmoid gate per head on the output (values out of it);
//   * latent_attention: a workgroup takes a tile of consecutive tokens of a request and a group
//     of heads (16 pairs at most, four to a wave), walks the keys in blocks staged once in LDS,
//     a lane to a key for the scores and a lane to a latent column for the weighted sum.
#include <algorithm>
#include <type_traits>

#include "common.h"

// --------------------------------------------------------------------------------- prepare
template <typename T, typename TW>
__global__ __launch_bounds__(512) void latent_prepare_kernel(
    const T* __restrict__ proj, int proj_stride, int q_rank, const TW* __restrict__ q_norm, float eps, T* __restrict__ c_q,
    int kv_col, int kv_rank, int rot_dim, const TW* __restrict__ kv_norm, const int32_t* __restrict__ positions,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, int interleaved, T* __restrict__ pages,
    T* __restrict__ pages_t, int page_size, const int32_t* __restrict__ slots) {
  __shared__ float scratch[17];
  const size_t n = blockIdx.x;
  const T* row = proj + n * proj_stride;
  float ss = 0.f, inv;
  if (blockIdx.y == 0) {
    for (int c = threadIdx.x; c < q_rank; c += blockDim.x) {
      const float v = to_f32<T>(row[c]);
      ss = fmaf(v, v, ss);
    }
    inv = 1.f / sqrtf(block_sum(ss, scratch) / static_cast<float>(q_rank) + eps);
    for (int c = threadIdx.x; c < q_rank; c += blockDim.x)
      c_q[n * q_rank + c] = from_f32<T>(to_f32<T>(row[c]) * inv * to_f32<TW>(q_norm[c]));
    return;
  }
  const T* kv = row + kv_col;
  for (int c = threadIdx.x; c < kv_rank; c += blockDim.x) {
    const float v = to_f32<T>(kv[c]);
    ss = fmaf(v, v, ss);
  }
  inv = 1.f / sqrtf(block_sum(ss, scratch) / static_cast<float>(kv_rank) + eps);
  T* dst = pages + static_cast<size_t>(slots[n]) * (kv_rank + rot_dim);
  // pages_t: the latent once more, transposed ([page][column][slot]), for readers that want a column's
  // slots side by side
  const size_t slot = static_cast<size_t>(slots[n]);
  T* dst_t = pages_t == nullptr ? nullptr : pages_t + (slot / page_size) * kv_rank * page_size + slot % page_size;
  for (int c = threadIdx.x; c < kv_rank; c += blockDim.x) {
    const T v = from_f32<T>(to_f32<T>(kv[c]) * inv * to_f32<TW>(kv_norm[c]));
    dst[c] = v;
    if (dst_t != nullptr) dst_t[static_cast<size_t>(c) * page_size] = v;
  }
  const int half = rot_dim / 2;
  const size_t p = static_cast<size_t>(positions[n]);
  for (int i = threadIdx.x; i < half; i += blockDim.x) {
    const int ia = interleaved ? 2 * i : i, ib = interleaved ? 2 * i + 1 : i + half;
    const float a = to_f32<T>(kv[kv_rank + ia]), b = to_f32<T>(kv[kv_rank + ib]);
    const float c = cos_t[p * half + i], s = sin_t[p * half + i];
    dst[kv_rank + ia] = from_f32<T>(rot_first(a, b, c, s));
    dst[kv_rank + ib] = from_f32<T>(rot_second(a, b, c, s));
  }
}

extern "C" int yk_latent_prepare(const void* proj, int proj_stride, int dtype, int q_rank, const void* q_norm, int w_dtype,
                                 float eps, void* c_q, int kv_col, int kv_rank, int rot_dim, const void* kv_norm,
                                 const int32_t* positions, const float* cos_t, const float* sin_t, int interleaved,
                                 int max_positions, void* pages, void* pages_t, int page_size, const int32_t* slots,
                                 int n_tokens, hipStream_t stream) {
  YK_REQUIRE(pages_t == nullptr || page_size > 0, "latent_prepare: transposed pages need the page size");
  YK_REQUIRE(n_tokens >= 0 && q_rank > 0 && kv_rank >= 0 && rot_dim >= 0 && rot_dim % 2 == 0, "latent_prepare: bad sizes");
  YK_REQUIRE(proj_stride >= q_rank && (kv_rank == 0 || proj_stride >= kv_col + kv_rank + rot_dim),
             "latent_prepare: the projection's rows are shorter than its sections");
  YK_REQUIRE(kv_rank == 0 || (kv_norm != nullptr && pages != nullptr && slots != nullptr && positions != nullptr),
             "latent_prepare: a layer that keeps a cache needs its norm, pages, slots and positions");
  YK_REQUIRE(kv_rank == 0 || rot_dim == 0 || (cos_t != nullptr && sin_t != nullptr && max_positions > 0),
             "latent_prepare: the rotated part needs its tables");
  if (n_tokens == 0) return 0;
  // queries and cache rows in workgroups of their own, of as many threads as leave one or two rounds of a row to read where tokens are
  // few (eight tokens of a width of 4,096: 13.0 -> 5.0 us)
  const int threads = n_tokens < 256 ? 512 : 128;
#define YK_CASE(D, T, WD, TW)                                                                                         \
  if (dtype == D && w_dtype == WD) {                                                                                  \
    latent_prepare_kernel<T, TW><<<dim3(n_tokens, kv_rank > 0 ? 2 : 1), threads, 0, stream>>>(                                                       \
        static_cast<const T*>(proj), proj_stride, q_rank, static_cast<const TW*>(q_norm), eps, static_cast<T*>(c_q),  \
        kv_col, kv_rank, rot_dim, static_cast<const TW*>(kv_norm), positions, cos_t, sin_t, interleaved,              \
        static_cast<T*>(pages), static_cast<T*>(pages_t), page_size, slots);                                          \
    return yk_check_launch("latent_prepare");                                                                         \
  }
  YK_CASE(YK_F32, float, YK_F32, float)
  YK_CASE(YK_BF16, bf16_t, YK_BF16, bf16_t)
  YK_CASE(YK_BF16, bf16_t, YK_F32, float)
#undef YK_CASE
  return yk_fail("latent_prepare: unsupported dtype combination");
}

// ------------------------------------------------------------------------- per-head products
constexpr int kHeadTokens = 8;   // tokens a workgroup multiplies by one head's matrix
constexpr int kHeadOut = 64;     // output columns a workgroup makes
constexpr int kHeadSlices = 4;   // groups of 64 threads that divide the input elements among them

// out[n, h, o] = sum_i x[n, h, i] w[h][i][o] for a tile of kHeadTokens tokens, one head and kHeadOut
// columns; thread (slice, column) sums every fourth input element, the slices meet in LDS.  TX: the
// input's and TG the gate's element type.
template <typename TX, typename TW, typename TG, typename TO>
__global__ __launch_bounds__(kHeadOut * kHeadSlices) void head_linear_kernel(
    const TX* __restrict__ x, int x_stride, const TW* __restrict__ w, TO* __restrict__ out, int out_stride, int in_dim,
    int out_dim, int tail, const int32_t* __restrict__ positions, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, int interleaved, const TG* __restrict__ gate, int gate_stride, int gate_col,
    int gate_elems, int n_tokens) {
  extern __shared__ float xs[];  // [kHeadTokens][in_dim + tail], then [kHeadSlices][kHeadTokens][kHeadOut]
  const int n0 = blockIdx.x * kHeadTokens, h = blockIdx.y, o0 = blockIdx.z * kHeadOut;
  const int count = min(kHeadTokens, n_tokens - n0);
  const int xw = in_dim + tail;
  float* part = xs + kHeadTokens * xw;
  for (int i = threadIdx.x; i < kHeadTokens * xw; i += blockDim.x) {
    const int t = i / xw, c = i % xw;
    xs[i] = t < count ? to_f32<TX>(x[static_cast<size_t>(n0 + t) * x_stride + h * xw + c]) : 0.f;
  }
  __syncthreads();
  const TW* wh = w + static_cast<size_t>(h) * in_dim * out_dim;
  const int ow = out_dim + tail;
  const int slice = threadIdx.x / kHeadOut, o = o0 + threadIdx.x % kHeadOut;
  float acc[kHeadTokens];
#pragma unroll
  for (int t = 0; t < kHeadTokens; ++t) acc[t] = 0.f;
  if (o < out_dim) {
    for (int i0 = slice; i0 < in_dim; i0 += 4 * kHeadSlices) {
      float wv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = i0 + j * kHeadSlices;
        wv[j] = i < in_dim ? to_f32<TW>(wh[static_cast<size_t>(i) * out_dim + o]) : 0.f;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = min(i0 + j * kHeadSlices, in_dim - 1);
#pragma unroll
        for (int t = 0; t < kHeadTokens; ++t) acc[t] = fmaf(xs[t * xw + i], wv[j], acc[t]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < kHeadTokens; ++t) part[(slice * kHeadTokens + t) * kHeadOut + threadIdx.x % kHeadOut] = acc[t];
  __syncthreads();
  for (int i = threadIdx.x; i < count * kHeadOut; i += blockDim.x) {
    const int t = i / kHeadOut, oc = i % kHeadOut;
    if (o0 + oc >= out_dim) continue;
    float v = 0.f;
#pragma unroll
    for (int sl = 0; sl < kHeadSlices; ++sl) v += part[(sl * kHeadTokens + t) * kHeadOut + oc];
    if (gate != nullptr)
      v *= 1.f / (1.f + expf(-to_f32<TG>(gate[static_cast<size_t>(n0 + t) * gate_stride + gate_col + h * gate_elems +
                                                  (gate_elems > 1 ? o0 + oc : 0)])));
    out[static_cast<size_t>(n0 + t) * out_stride + h * ow + o0 + oc] = from_f32<TO>(v);
  }
  if (blockIdx.z != 0) return;
  const int half = tail / 2;
  for (int i = threadIdx.x; i < count * half; i += blockDim.x) {
    const int t = i / half, j = i % half;
    const int ia = interleaved ? 2 * j : j, ib = interleaved ? 2 * j + 1 : j + half;
    const float a = xs[t * xw + in_dim + ia], b = xs[t * xw + in_dim + ib];
    const size_t p = static_cast<size_t>(positions[n0 + t]);
    const float c = cos_t[p * half + j], s = sin_t[p * half + j];
    TO* dst = out + static_cast<size_t>(n0 + t) * out_stride + h * ow + out_dim;
    dst[ia] = from_f32<TO>(rot_first(a, b, c, s));
    dst[ib] = from_f32<TO>(rot_second(a, b, c, s));
  }
}

// The same for an even out_dim and a handful of tokens, where the product is all latency: 32 slices of 32 threads, a thread two
// columns; eight of its weights (of 4 or 8 bytes) are on their way at a time, the first before the input is staged; a token's inputs lie
// side by side in LDS, so that an input element of all eight tokens is two reads for sixteen multiplications.  Eight tokens of 32 heads,
// bfloat16: 512 -> 128 elements 42 -> 6.7 us in a replayed step, 128 -> 512 14 -> under 6 us against head_linear_kernel, whose loads wait for one
// another; errors against float64 9.6e-8 and 7.3e-8 of the size in float32 (2.1e-7 and 1.1e-7), the waves' sums being added pairwise.
constexpr int kPairSlices = 32, kPairBatch = 8;
__device__ __forceinline__ float2 pair_of(uint32_t w) { return make_float2(__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u)); }
__device__ __forceinline__ float2 pair_of(uint2 w) { return make_float2(__uint_as_float(w.x), __uint_as_float(w.y)); }
template <typename T>
struct PairBits;
template <>
struct PairBits<float> {
  typedef uint2 type;
};
template <>
struct PairBits<bf16_t> {
  typedef uint32_t type;
};

template <typename TX, typename TW, typename TG, typename TO>
__global__ __launch_bounds__(32 * kPairSlices) void head_linear_pair_kernel(
    const TX* __restrict__ x, int x_stride, const TW* __restrict__ w, TO* __restrict__ out, int out_stride, int in_dim,
    int out_dim, int tail, const int32_t* __restrict__ positions, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, int interleaved, const TG* __restrict__ gate, int gate_stride, int gate_col,
    int gate_elems, int n_tokens) {
  static_assert(kHeadTokens == 8 && kHeadOut == 64, "thread (slice, pair) and two 16-byte reads a row");
  extern __shared__ __attribute__((aligned(16))) float xs[];  // [in_dim + tail][8], then [16 waves][8][64]
  const int n0 = blockIdx.x * kHeadTokens, h = blockIdx.y, o0 = blockIdx.z * kHeadOut;
  const int count = min(kHeadTokens, n_tokens - n0), xw = in_dim + tail, ow = out_dim + tail;
  float* part = xs + kHeadTokens * xw;
  const int slice = threadIdx.x / 32, o = o0 + 2 * (threadIdx.x % 32);
  typedef typename PairBits<TW>::type bits_t;
  const TW* wh = w + static_cast<size_t>(h) * in_dim * out_dim + min(o, out_dim - 2);
  bits_t wv[kPairBatch];
  auto ask = [&](int i0) {
#pragma unroll
    for (int j = 0; j < kPairBatch; ++j)
      wv[j] = *reinterpret_cast<const bits_t*>(wh + static_cast<size_t>(min(i0 + j * kPairSlices, in_dim - 1)) * out_dim);
  };
  ask(slice);
  for (int i = threadIdx.x; i < kHeadTokens * xw; i += blockDim.x) {
    const int t = i % kHeadTokens, c = i / kHeadTokens;
    xs[i] = t < count ? to_f32<TX>(x[static_cast<size_t>(n0 + t) * x_stride + h * xw + c]) : 0.f;
  }
  __syncthreads();
  float acc[kHeadTokens][2] = {};
  for (int i0 = slice; i0 < in_dim; i0 += kPairBatch * kPairSlices) {
#pragma unroll
    for (int j = 0; j < kPairBatch; ++j) {
      const int i = i0 + j * kPairSlices;
      if (i >= in_dim) continue;
      const float2 p = pair_of(wv[j]);
      const float4 a = *reinterpret_cast<const float4*>(&xs[i * kHeadTokens]), b = *reinterpret_cast<const float4*>(&xs[i * kHeadTokens + 4]);
      const float v[kHeadTokens] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
      for (int t = 0; t < kHeadTokens; ++t) {
        acc[t][0] = fmaf(v[t], p.x, acc[t][0]);
        acc[t][1] = fmaf(v[t], p.y, acc[t][1]);
      }
    }
    if (i0 + kPairBatch * kPairSlices < in_dim) ask(i0 + kPairBatch * kPairSlices);
  }
  // a wave's two slices meet in registers, the waves in LDS
#pragma unroll
  for (int t = 0; t < kHeadTokens; ++t) {
    float sum[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const auto half = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[t][e]), __float_as_uint(acc[t][e]), false, false);
      sum[e] = __uint_as_float(half[0]) + __uint_as_float(half[1]);
    }
    if (threadIdx.x % 64 < 32)
      *reinterpret_cast<float2*>(&part[(threadIdx.x / 64 * kHeadTokens + t) * kHeadOut + 2 * (threadIdx.x % 32)]) = make_float2(sum[0], sum[1]);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < count * kHeadOut; i += blockDim.x) {
    const int t = i / kHeadOut, oc = i % kHeadOut;
    if (o0 + oc >= out_dim) continue;
    float q[kPairSlices / 2];
#pragma unroll
    for (int sl = 0; sl < kPairSlices / 2; ++sl) q[sl] = part[(sl * kHeadTokens + t) * kHeadOut + oc];
#pragma unroll
    for (int d = kPairSlices / 4; d > 0; d /= 2)
#pragma unroll
      for (int sl = 0; sl < d; ++sl) q[sl] += q[sl + d];
    float v = q[0];
    if (gate != nullptr)
      v *= 1.f / (1.f + expf(-to_f32<TG>(gate[static_cast<size_t>(n0 + t) * gate_stride + gate_col + h * gate_elems +
                                                  (gate_elems > 1 ? o0 + oc : 0)])));
    out[static_cast<size_t>(n0 + t) * out_stride + h * ow + o0 + oc] = from_f32<TO>(v);
  }
  if (blockIdx.z != 0) return;
  const int half = tail / 2;
  for (int i = threadIdx.x; i < count * half; i += blockDim.x) {
    const int t = i / half, j = i % half;
    const int ia = interleaved ? 2 * j : j, ib = interleaved ? 2 * j + 1 : j + half;
    const float a = xs[(in_dim + ia) * kHeadTokens + t], b = xs[(in_dim + ib) * kHeadTokens + t];
    const size_t p = static_cast<size_t>(positions[n0 + t]);
    const float c = cos_t[p * half + j], s = sin_t[p * half + j];
    TO* dst = out + static_cast<size_t>(n0 + t) * out_stride + h * ow + out_dim;
    dst[ia] = from_f32<TO>(rot_first(a, b, c, s));
    dst[ib] = from_f32<TO>(rot_second(a, b, c, s));
  }
}

// x, w, gate and out each float32 or bfloat16 (the gate in the output's dtype where the input is float32:
// the way out of the latent; else in the input's)
extern "C" int yk_head_linear(const void* x, int x_stride, int x_dtype, const void* w, int w_dtype, void* out, int out_dtype,
                              int n_heads, int in_dim, int out_dim, int tail, const int32_t* positions, const float* cos_t,
                              const float* sin_t, int interleaved, const void* gate, int gate_dtype, int gate_stride,
                              int gate_col, int gate_elems, int n_tokens, hipStream_t stream) {
  YK_REQUIRE(n_tokens >= 0 && n_heads > 0 && in_dim > 0 && out_dim > 0 && tail >= 0 && tail % 2 == 0, "head_linear: bad sizes");
  YK_REQUIRE(gate == nullptr || gate_elems == 1 || gate_elems == out_dim, "head_linear: a gate per head or per output element");
  YK_REQUIRE(x_stride >= n_heads * (in_dim + tail), "head_linear: the input's rows are shorter than its heads");
  YK_REQUIRE(tail == 0 || (positions != nullptr && cos_t != nullptr && sin_t != nullptr), "head_linear: a turned tail needs positions and tables");
  const size_t lds = sizeof(float) * (static_cast<size_t>(kHeadTokens) * (in_dim + tail) + kHeadSlices * kHeadTokens * kHeadOut);
  const size_t pair_lds = sizeof(float) * (static_cast<size_t>(kHeadTokens) * (in_dim + tail) + kPairSlices / 2 * kHeadTokens * kHeadOut);
  // Pairs win by how long a thread's chain of weights is, and lose by their larger workgroups, of which a compute unit runs one.  Up to 32
  // tokens, time over head_linear_kernel's by workgroups (256 / 512 / 1,024 / 2,048): float32 weights, 32 input elements 1.15 / 1.35 / 1.75 /
  // 2.1, 64 0.94 / 1.11 / 1.3 / 1.55, 96 0.81 / 0.96 / 1.2 / 1.3, 128 0.71 / 0.8 / 0.98 / 1.13, 192 0.58 / 0.65 / 0.85 / 0.97; bfloat16 ones are about
  // as those of twice the elements (32 0.93 / 1.1 / 1.5 / 1.8, 64 0.73 / 0.87 / 1.13 / 1.35, 96 0.6 / 0.71 / 0.96 / 1.06, 128 0.51 / 0.63 / 0.75 / 0.87).  More tokens
  // (float32): 512 of 32 heads, 128 -> 512 93 us against 114, 512 -> 128 99 against 63.
  const dim3 grid((n_tokens + kHeadTokens - 1) / kHeadTokens, n_heads, (out_dim + kHeadOut - 1) / kHeadOut);
  const long long workgroups = static_cast<long long>(grid.x) * grid.y * grid.z;
  const int chain = w_dtype == YK_F32 ? in_dim : 2 * in_dim;
  const bool few = n_tokens <= 32 && (chain >= 192 || workgroups <= (chain >= 128 ? 1024 : chain >= 96 ? 512 : chain >= 64 ? 256 : 0));
  const bool pairs = (few || in_dim >= 256) && out_dim % 2 == 0 && reinterpret_cast<uintptr_t>(w) % 8 == 0 && pair_lds <= 64 * 1024;
  YK_REQUIRE(lds <= 64 * 1024, "head_linear: heads of more than 1,700 input elements do not fit");
  if (n_tokens == 0) return 0;
  const int out_stride = n_heads * (out_dim + tail);
  if (gate == nullptr) gate_dtype = out_dtype;
#define YK_CASE(XD, TX, WD, TW, GD, TG, OD, TO)                                                                      \
  if (x_dtype == XD && w_dtype == WD && gate_dtype == GD && out_dtype == OD) {                                       \
    if (pairs)                                                                                                       \
      head_linear_pair_kernel<TX, TW, TG, TO><<<grid, 32 * kPairSlices, pair_lds, stream>>>(                         \
          static_cast<const TX*>(x), x_stride, static_cast<const TW*>(w), static_cast<TO*>(out), out_stride, in_dim, \
          out_dim, tail, positions, cos_t, sin_t, interleaved, static_cast<const TG*>(gate), gate_stride, gate_col,  \
          gate_elems, n_tokens);                                                                                              \
    else                                                                                                             \
      head_linear_kernel<TX, TW, TG, TO><<<grid, kHeadOut * kHeadSlices, lds, stream>>>(                             \
          static_cast<const TX*>(x), x_stride, static_cast<const TW*>(w), static_cast<TO*>(out), out_stride, in_dim, \
          out_dim, tail, positions, cos_t, sin_t, interleaved, static_cast<const TG*>(gate), gate_stride, gate_col,  \
          gate_elems, n_tokens);                                                                                              \
    return yk_check_launch("head_linear");                                                                           \
  }
  YK_CASE(YK_F32, float, YK_F32, float, YK_F32, float, YK_F32, float)
  YK_CASE(YK_BF16, bf16_t, YK_BF16, bf16_t, YK_F32, float, YK_F32, float)
  YK_CASE(YK_BF16, bf16_t, YK_F32, float, YK_F32, float, YK_F32, float)
  YK_CASE(YK_F32, float, YK_BF16, bf16_t, YK_BF16, bf16_t, YK_BF16, bf16_t)
  YK_CASE(YK_F32, float, YK_F32, float, YK_BF16, bf16_t, YK_BF16, bf16_t)
#undef YK_CASE
  return yk_fail("head_linear: unsupported dtype combination");
}

// The same products on the matrix cores, for many tokens: bfloat16 weights kept [heads][out][in] (a row of
// the first operand is then 16 bytes of memory a lane), the input bfloat16 or float32 (as two bfloat16
// parts, the rounded value and what the rounding left over, each with its own product).  A wave makes
// 16 TT tokens x 64 columns of one head; the weight is the first operand, so that a lane ends with four
// consecutive columns of one token, a store of 16 bytes.  The next step's operands are in flight while
// the current ones are multiplied.  Four waves a workgroup take four runs of tokens.
// Bound by the float32 side (its reading or writing) and the reads of the weights from the caches, which
// every wave makes for its tokens: hence several token tiles a wave.  16 heads, us (one tile a wave,
// nothing in flight, 4-byte stores: before / 1 / 2 / 4 tiles a wave):
//   128 -> 512 in float32    100 tokens  5.6 / 5.0 / 5.7 / 5.5    512 14.7 / 14.2 / 11.0 / 9.5    2,048 45.8 / 43.4 / 32.6 / 27.1
//   512 -> 128 from float32  100 tokens 15.8 / 13.1 / 16.3 / 15.1  512 20.3 / 14.1 / 17.9 / 26.3  2,048 47.1 / 46.6 / 33.8 / 28.3
// (2,048 tokens: 83 MB, 17 us at what a copy reaches.  Twice the columns a wave: 30.1 and 27.7.)
// With a turned tail of 64 behind each head, which the head's workgroups share, 128 -> 512 (us, one tile / several, the tail
// left to the first workgroup / several, shared): 512 tokens 17.9 / 22.7 / 10.4, 1,000 27.7 / 30.2 / 16.6, 2,048 45.9 / 35.6 / 28.2
// (within a prompt, its inputs from memory, 46.8 -> 39.7).
typedef __bf16 hl_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float hl_f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t hl_u32x4_t __attribute__((ext_vector_type(4)));
union HlFrag {
  hl_u32x4_t u;
  hl_bf16x8_t v;
};

// eight consecutive elements of an input row as they lie there
template <typename TX>
struct HlRaw {
  hl_u32x4_t u[sizeof(TX) / 2];
};
template <typename TX>
__device__ __forceinline__ HlRaw<TX> hl_raw8(const TX* p) {
  HlRaw<TX> x;
#pragma unroll
  for (unsigned i = 0; i < sizeof(TX) / 2; ++i) x.u[i] = reinterpret_cast<const hl_u32x4_t*>(p)[i];
  return x;
}
__device__ __forceinline__ hl_u32x4_t hl_high8(const HlRaw<bf16_t>& x) { return x.u[0]; }
__device__ __forceinline__ hl_u32x4_t hl_high8(const HlRaw<float>& x) {
  hl_u32x4_t v;
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = pack_bf16x2(__uint_as_float(x.u[i / 2][2 * (i % 2)]), __uint_as_float(x.u[i / 2][2 * (i % 2) + 1]));
  return v;
}
// what the rounding of eight floats to bfloat16 left over, itself rounded to bfloat16: a float32 input goes
// through the matrix cores as the sum of the two, so the product sees it to 16 bits of fraction
__device__ __forceinline__ hl_u32x4_t hl_rest8(const HlRaw<bf16_t>&, hl_u32x4_t) { return hl_u32x4_t{0u, 0u, 0u, 0u}; }
__device__ __forceinline__ uint32_t hl_rest2(float x, float y, uint32_t hi) {
  return pack_bf16x2(x - __uint_as_float(hi << 16), y - __uint_as_float(hi & 0xffff0000u));
}
__device__ __forceinline__ hl_u32x4_t hl_rest8(const HlRaw<float>& x, hl_u32x4_t hi) {
  hl_u32x4_t v;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    v[i] = hl_rest2(__uint_as_float(x.u[i / 2][2 * (i % 2)]), __uint_as_float(x.u[i / 2][2 * (i % 2) + 1]), hi[i]);
  return v;
}
__device__ __forceinline__ void hl_store4(float* p, float a, float b, float c, float d) { *reinterpret_cast<float4*>(p) = make_float4(a, b, c, d); }
__device__ __forceinline__ void hl_store4(bf16_t* p, float a, float b, float c, float d) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(a, b), pack_bf16x2(c, d));
}

template <typename TX, typename TG, typename TO, int TT>
__global__ __launch_bounds__(256) void head_linear_mfma_kernel(
    const TX* __restrict__ x, int x_stride, const bf16_t* __restrict__ w_t, TO* __restrict__ out, int out_stride, int in_dim,
    int out_dim, int tail, const int32_t* __restrict__ positions, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, int interleaved, const TG* __restrict__ gate, int gate_stride, int gate_col,
    int gate_elems, int n_tokens) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  constexpr int NT = 4;
  const int r = lane % 16, g = lane / 16;
  const int n0 = (blockIdx.x * 4 + wave) * (16 * TT), h = blockIdx.y, o0 = blockIdx.z * (16 * NT);
  if (n0 >= n_tokens) return;
  const int xw = in_dim + tail, ow = out_dim + tail;
  const TX* xp[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t)  // (rows past the end repeat the last token and are not stored)
    xp[t] = x + static_cast<size_t>(min(n0 + 16 * t + r, n_tokens - 1)) * x_stride + h * xw + 8 * g;
  const int n_tiles = min(NT, (out_dim - o0) / 16);
  const bf16_t* wp[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)  // (tiles past the end repeat the last and are not stored)
    wp[j] = w_t + (static_cast<size_t>(h) * out_dim + o0 + 16 * min(j, n_tiles - 1) + r) * in_dim + 8 * g;
  hl_f32x4_t acc[TT][NT] = {};
  HlRaw<TX> xr[TT];
  HlFrag wr[NT];
  auto ask = [&](int k0) {
#pragma unroll
    for (int t = 0; t < TT; ++t) xr[t] = hl_raw8(xp[t] + k0);
#pragma unroll
    for (int j = 0; j < NT; ++j) wr[j].u = *reinterpret_cast<const hl_u32x4_t*>(wp[j] + k0);
  };
  ask(0);
  for (int k0 = 0; k0 < in_dim; k0 += 32) {
    HlFrag a[TT], rest[TT], b[NT];
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      a[t].u = hl_high8(xr[t]);
      rest[t].u = hl_rest8(xr[t], a[t].u);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j) b[j] = wr[j];
    ask(min(k0 + 32, in_dim - 32));  // (the last step asks for itself once more, unread)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j].v, a[t].v, acc[t][j], 0, 0, 0);
        if (sizeof(TX) == 4) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j].v, rest[t].v, acc[t][j], 0, 0, 0);
      }
  }
  // acc[t][j][i]: token n0 + 16 t + r, column o0 + 16 j + 4 g + i
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    const int n = n0 + 16 * t + r;
    if (n >= n_tokens) continue;
    float gv[4] = {1.f, 1.f, 1.f, 1.f};
    const TG* grow = gate == nullptr ? nullptr : gate + static_cast<size_t>(n) * gate_stride + gate_col + h * gate_elems;
    if (gate != nullptr && gate_elems == 1) gv[0] = gv[1] = gv[2] = gv[3] = 1.f / (1.f + expf(-to_f32<TG>(grow[0])));
#pragma unroll
    for (int j = 0; j < NT; ++j)
      if (j < n_tiles) {
        const int o = o0 + 16 * j + 4 * g;
        if (gate != nullptr && gate_elems > 1) {
#pragma unroll
          for (int i = 0; i < 4; ++i) gv[i] = 1.f / (1.f + expf(-to_f32<TG>(grow[o + i])));
        }
        hl_store4(out + static_cast<size_t>(n) * out_stride + h * ow + o, acc[t][j][0] * gv[0], acc[t][j][1] * gv[1], acc[t][j][2] * gv[2],
                  acc[t][j][3] * gv[3]);
      }
  }
  if (tail == 0) return;
  // the wave's tokens' tails are shared among the head's workgroups, which would otherwise end while the first still turns them
  const int half = tail / 2, pairs = min(16 * TT, n_tokens - n0) * half;
#pragma unroll 4
  for (int i = static_cast<int>(blockIdx.z) * kWave + lane; i < pairs; i += static_cast<int>(gridDim.z) * kWave) {
    const int t = i / half, j = i % half, n = n0 + t;
    const int ia = interleaved ? 2 * j : j, ib = interleaved ? 2 * j + 1 : j + half;
    const TX* src = x + static_cast<size_t>(n) * x_stride + h * xw + in_dim;
    const float a = to_f32<TX>(src[ia]), b = to_f32<TX>(src[ib]);
    const size_t p = static_cast<size_t>(positions[n]);
    const float c = cos_t[p * half + j], sn = sin_t[p * half + j];
    TO* dst = out + static_cast<size_t>(n) * out_stride + h * ow + out_dim;
    dst[ia] = from_f32<TO>(rot_first(a, b, c, sn));
    dst[ib] = from_f32<TO>(rot_second(a, b, c, sn));
  }
}

extern "C" int yk_head_linear_mfma_ok(int in_dim, int out_dim, int tail) { return in_dim % 32 == 0 && out_dim % 16 == 0 && tail % 8 == 0; }

// w_t: bfloat16 [heads][out_dim][in_dim]; x bfloat16 or float32 with 16-byte aligned rows and heads
extern "C" int yk_head_linear_mfma(const void* x, int x_stride, int x_dtype, const void* w_t, void* out, int out_dtype, int n_heads,
                                   int in_dim, int out_dim, int tail, const int32_t* positions, const float* cos_t,
                                   const float* sin_t, int interleaved, const void* gate, int gate_dtype, int gate_stride,
                                   int gate_col, int gate_elems, int n_tokens, hipStream_t stream) {
  YK_REQUIRE(gate == nullptr || gate_elems == 1 || gate_elems == out_dim, "head_linear_mfma: a gate per head or per output element");
  YK_REQUIRE(n_tokens >= 0 && n_heads > 0 && yk_head_linear_mfma_ok(in_dim, out_dim, tail), "head_linear_mfma: sizes it is not built for");
  YK_REQUIRE(x_stride >= n_heads * (in_dim + tail) && x_stride % 8 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 &&
                 reinterpret_cast<uintptr_t>(w_t) % 16 == 0,
             "head_linear_mfma: the input's rows must be 16-byte aligned");
  YK_REQUIRE(tail == 0 || (positions != nullptr && cos_t != nullptr && sin_t != nullptr), "head_linear_mfma: a turned tail needs positions and tables");
  if (n_tokens == 0) return 0;
  const int out_stride = n_heads * (out_dim + tail);
  if (gate == nullptr) gate_dtype = out_dtype;
  YK_REQUIRE(reinterpret_cast<uintptr_t>(out) % 16 == 0, "head_linear_mfma: the output must be 16-byte aligned");
  // as many token tiles a wave as still leave 896 waves (of the 1,024 that a wave for every SIMD would be); four only
  // where a wave's walk over the input is long enough to share what it read: us with a turned tail, one / two / four
  // tiles, 24 heads 96 -> 128 at 1,500 tokens 12.1 / 11.8 / 13.4, 32 heads 64 -> 128 14.0 / 12.4 / 13.8, 16 heads
  // 128 -> 512 at 1,000 26.6 / 19.4 / 16.6.  (At both lines more tiles are faster: 1,792 units, 32 heads 512 -> 128, 25.1 / 18.6 / 27.1,
  // 3,584 units, 16 heads 128 -> 512, 14.7 / 11.9 / 9.9; and already some way below them: 1,408 units 24.8 / 18.3, 2,816 units
  // 36.1 / 32.9 / 27.6.)
  const long long units = static_cast<long long>((n_tokens + 15) / 16) * n_heads * ((out_dim + 63) / 64);
  const int tiles = units >= 3584 && in_dim >= 128 ? 4 : units >= 1792 ? 2 : 1;
#define YK_TILES(TX, TG, TO, TT)                                                                                        \
  if (tiles == TT) {                                                                                                    \
    const dim3 grid((n_tokens + 64 * TT - 1) / (64 * TT), n_heads, (out_dim + 63) / 64);                                \
    head_linear_mfma_kernel<TX, TG, TO, TT><<<grid, 256, 0, stream>>>(                                                  \
        static_cast<const TX*>(x), x_stride, static_cast<const bf16_t*>(w_t), static_cast<TO*>(out), out_stride, in_dim, \
        out_dim, tail, positions, cos_t, sin_t, interleaved, static_cast<const TG*>(gate), gate_stride, gate_col,       \
        gate_elems, n_tokens);                                                                                          \
    return yk_check_launch("head_linear_mfma");                                                                         \
  }
#define YK_CASE(XD, TX, GD, TG, OD, TO)                                                                                 \
  if (x_dtype == XD && gate_dtype == GD && out_dtype == OD) {                                                           \
    YK_TILES(TX, TG, TO, 1) YK_TILES(TX, TG, TO, 2) YK_TILES(TX, TG, TO, 4)                                             \
  }
  YK_CASE(YK_BF16, bf16_t, YK_F32, float, YK_F32, float)
  YK_CASE(YK_F32, float, YK_BF16, bf16_t, YK_BF16, bf16_t)
#undef YK_CASE
#undef YK_TILES
  return yk_fail("head_linear_mfma: unsupported dtype combination");
}

// --------------------------------------------------------------------------------- attention
constexpr int kLatWaves = 4;       // waves of a workgroup
constexpr int kLatItems = 4;       // (token, head) pairs a wave carries
constexpr int kLatPairs = kLatWaves * kLatItems;

// tiles: rows of (request, first token index in the batch, token count, first position).  Workgroup
// (tile, head group): pair i of it is token i / heads_per_group of the tile and head
// group * heads_per_group + i % heads_per_group; wave w carries the pairs w, w + 4, w + 8, w + 12.
// KB keys are staged per block ([KB][width] in T, rows padded by `pad` elements); RPL latent columns a lane.
template <typename T, int RPL>
__global__ __launch_bounds__(64 * kLatWaves) void latent_attention_kernel(
    const float* __restrict__ q_lat, const T* __restrict__ pages, const int32_t* __restrict__ tiles,
    const int32_t* __restrict__ block_table, int table_width, int page_size, int n_heads, int heads_per_group, int kv_rank,
    int rot_dim, float scale, int KB, int pad, const float* __restrict__ sink, float* __restrict__ out) {
  extern __shared__ unsigned char lds_raw[];
  const int width = kv_rank + rot_dim, row_w = width + pad;
  T* kblock = reinterpret_cast<T*>(lds_raw);                                             // [KB][row_w]
  float* pbuf = reinterpret_cast<float*>(lds_raw + static_cast<size_t>(KB) * row_w * sizeof(T) + 16 -
                                         (static_cast<size_t>(KB) * row_w * sizeof(T)) % 16);  // [kLatPairs][KB]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int32_t* tile = tiles + 4 * blockIdx.x;
  const int seq = tile[0], tok0 = tile[1], count = tile[2], pos0 = tile[3];
  const int group = blockIdx.y;
  const int n_pairs = count * heads_per_group;
  const int last_pos = pos0 + count - 1;

  // this wave's pairs
  int tok[kLatItems], head[kLatItems], pos[kLatItems];
  bool live[kLatItems];
  float m[kLatItems], l[kLatItems], acc[kLatItems][RPL];
#pragma unroll
  for (int it = 0; it < kLatItems; ++it) {
    const int pair = wave + it * kLatWaves;
    const int t = pair / heads_per_group;
    head[it] = group * heads_per_group + pair % heads_per_group;
    live[it] = pair < n_pairs && head[it] < n_heads;
    tok[it] = tok0 + (live[it] ? t : 0);
    if (!live[it]) head[it] = 0;
    pos[it] = pos0 + (live[it] ? t : 0);
    // a sink is a score without a key: it starts the running maximum and counts once in the sum
    m[it] = sink != nullptr ? sink[head[it]] : -INFINITY;
    l[it] = sink != nullptr ? 1.f : 0.f;
#pragma unroll
    for (int r = 0; r < RPL; ++r) acc[it][r] = 0.f;
  }
  const int32_t* bt = block_table + static_cast<size_t>(seq) * table_width;

  for (int k0 = 0; k0 <= last_pos; k0 += KB) {
    const int nk = min(KB, last_pos + 1 - k0);
    __syncthreads();  // the block before has been read by every wave
    for (int i = threadIdx.x; i < nk * width; i += blockDim.x) {
      const int j = i / width, c = i % width;
      const int key = k0 + j;
      const size_t slot = static_cast<size_t>(bt[key / page_size]) * page_size + key % page_size;
      kblock[j * row_w + c] = pages[slot * width + c];
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kLatItems; ++it) {
      if (!live[it]) continue;  // (uniform over the wave)
      const float* q = q_lat + (static_cast<size_t>(tok[it]) * n_heads + head[it]) * width;
      float* pw = pbuf + (wave + it * kLatWaves) * KB;
      // scores: a lane to a key (KB may exceed 64 never: KB <= 64)
      float s = -INFINITY;
      if (lane < nk && k0 + lane <= pos[it]) {
        const T* kr = kblock + lane * row_w;
        float d = 0.f;
        for (int c = 0; c < width; ++c) d = fmaf(q[c], to_f32<T>(kr[c]), d);
        s = d * scale;
      }
      const float m_new = fmaxf(m[it], wave_max(s));
      const float p = s == -INFINITY ? 0.f : expf(s - m_new);
      const float corr = m[it] == -INFINITY ? 0.f : expf(m[it] - m_new);
      l[it] = l[it] * corr + wave_sum(p);
      m[it] = m_new;
      if (lane < KB) pw[lane] = p;
      // weighted sum of the latent part: a lane to the columns lane, lane + 64, ...
      const int visible = min(nk, pos[it] - k0 + 1);
#pragma unroll
      for (int r = 0; r < RPL; ++r) acc[it][r] *= corr;
      for (int j = 0; j < visible; ++j) {
        const float pj = pw[j];
        const T* kr = kblock + j * row_w;
#pragma unroll
        for (int r = 0; r < RPL; ++r) {
          const int c = lane + r * kWave;
          if (c < kv_rank) acc[it][r] = fmaf(pj, to_f32<T>(kr[c]), acc[it][r]);
        }
      }
    }
  }
#pragma unroll
  for (int it = 0; it < kLatItems; ++it) {
    if (!live[it]) continue;
    const float inv = 1.f / l[it];
    float* o = out + (static_cast<size_t>(tok[it]) * n_heads + head[it]) * kv_rank;
#pragma unroll
    for (int r = 0; r < RPL; ++r) {
      const int c = lane + r * kWave;
      if (c < kv_rank) o[c] = acc[it][r] * inv;
    }
  }
}

extern "C" int yk_latent_tile_tokens(int n_heads) {
  const int hpg = n_heads < kLatItems ? n_heads : kLatItems;
  return kLatPairs / hpg;
}

extern "C" int yk_latent_attention(const float* q_lat, const void* pages, int dtype, const int32_t* tiles, int n_tiles,
                                   const int32_t* block_table, int table_width, int page_size, int n_heads, int kv_rank,
                                   int rot_dim, float scale, const float* sink, float* out, hipStream_t stream) {
  YK_REQUIRE(n_tiles >= 0 && n_heads > 0 && kv_rank > 0 && rot_dim >= 0 && page_size > 0 && table_width > 0,
             "latent_attention: bad sizes");
  YK_REQUIRE(kv_rank <= 16 * kWave, "latent_attention: latents of more than 1,024 elements are not offered");
  if (n_tiles == 0) return 0;
  const int hpg = n_heads < kLatItems ? n_heads : kLatItems;
  const int groups = (n_heads + hpg - 1) / hpg;
  const int width = kv_rank + rot_dim;
  const size_t esz = dtype == YK_BF16 ? 2 : 4;
  // rows a whole number of 32-bit words long and an odd number of them apart: lanes that read the
  // same column of different keys then meet different banks
  int pad = 0;
  while ((static_cast<size_t>(width + pad) * esz) % 4 != 0 || ((static_cast<size_t>(width + pad) * esz) / 4) % 2 == 0) ++pad;
  int KB = 64;
  while (KB > 8 && static_cast<size_t>(KB) * (width + pad) * esz > 96 * 1024) KB /= 2;
  const size_t kbytes = static_cast<size_t>(KB) * (width + pad) * esz;
  YK_REQUIRE(kbytes <= 128 * 1024, "latent_attention: page rows too long for the key block");
  const size_t lds = kbytes + 16 - kbytes % 16 + static_cast<size_t>(kLatPairs) * KB * sizeof(float);
  const int rpl = (kv_rank + kWave - 1) / kWave;
  dim3 grid(n_tiles, groups);
#define YK_LAUNCH(T, R)                                                                                                \
  {                                                                                                                    \
    auto kern = latent_attention_kernel<T, R>;                                                                         \
    if (lds > 64 * 1024 &&                                                                                             \
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,          \
                            static_cast<int>(lds)) != hipSuccess)                                                      \
      return yk_fail("latent_attention: the key block does not fit in LDS");                                           \
    kern<<<grid, 64 * kLatWaves, lds, stream>>>(q_lat, static_cast<const T*>(pages), tiles, block_table, table_width,  \
                                                page_size, n_heads, hpg, kv_rank, rot_dim, scale, KB, pad, sink, out);       \
    return yk_check_launch("latent_attention");                                                                        \
  }
#define YK_RPL(T)                      \
  if (rpl <= 1) YK_LAUNCH(T, 1)        \
  if (rpl <= 2) YK_LAUNCH(T, 2)        \
  if (rpl <= 4) YK_LAUNCH(T, 4)        \
  if (rpl <= 8) YK_LAUNCH(T, 8)        \
  YK_LAUNCH(T, 16)
  if (dtype == YK_F32) {
    YK_RPL(float)
  }
  if (dtype == YK_BF16) {
    YK_RPL(bf16_t)
  }
#undef YK_RPL
#undef YK_LAUNCH
  return yk_fail("latent_attention: unsupported dtype");
}

// ------------------------------------------------------------------ attention on the matrix cores
// bfloat16 pages, rows of 32 KS elements of which the first 16 CT are the latent; beside the page
// rows [slot][width] the latent is kept once more transposed, [column][slot], so that both products
// take their first operand from memory as it lies there, 16 bytes a lane:
//   S^T = K . Q^T   (first operand: 16 page rows x 32 elements; second: the queries, in registers)
//   O^T = C^T . P^T (first operand: 16 latent columns x 32 slots of the transposed pages)
// A workgroup owns the 64 columns = (token, head) pairs of one tile, 16 to every pair of its eight
// waves: up to 64 heads of a token, or several tokens' heads where a model has fewer.  It walks the keys
// in groups of 32, whose page rows and transposed latents it parks in LDS once for all waves, so memory
// is asked for a key once per 64 columns.  The waves of a pair divide a group's work: each makes the
// scores of 16 keys, both read all 32 of them back (float32, through LDS) and take the same softmax
// step, and each makes the sums of one half of the latent; so a wave needs half the registers and every
// SIMD has two waves.  The walk is skewed by a group: between two barriers a wave makes the next group's
// scores and finishes this one's, while the loads of the rows after next and the latents after these
// are in flight in registers.  Lane group g takes the probabilities of keys 8g .. 8g + 7 of its column:
// the second operand of the other product as it stands.  Each lane keeps its column's running maximum
// and sum.  With n_splits > 1 the groups of keys are divided among gridDim.z workgroups, which leave
// unnormalised sums, maxima and sums of weights for a merging kernel.
// Bound by the LDS reads (a group of rows of 576 and latents of 512 is read four times over, 272 KiB).
// Before (every wave walking the pages on its own, its loads not staged) / this, 16 heads, rows of 576, shuffled pages
// (us): a prompt of 2,048 tokens 757 / 217, 512 tokens behind 1,536 525 / 93, eight decoded tokens behind 100 keys 42 /
// 14, behind 1,000 45 / 16, behind 4,000 63 / 29.  Two workgroups share a compute unit at latents of up to 128, whose registers and
// LDS leave room for them (latent 128, a prompt of 2,048 tokens 108 -> 88 us against one; eight prompts of 100, 64 heads, 33 -> 28);
// wider ones take all registers.
constexpr int kLatCols = 64;  // columns of a workgroup
typedef __bf16 lat_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float lat_f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t lat_u32x4_t __attribute__((ext_vector_type(4)));
union LatFrag {
  lat_u32x4_t u;
  lat_bf16x8_t v;
  bf16_t h[8];
};

// N products that each take a piece from LDS: the pieces are read four at a time, the next four asked
// for before these four are used (left alone the compiler keeps one read in flight, and a wave waits for
// the LDS at every product)
template <int N, typename Read, typename Use>
__device__ __forceinline__ void lat_read_ahead(Read read, Use use) {
  constexpr int B = 4;
  LatFrag f[2][B];
#pragma unroll
  for (int j = 0; j < B && j < N; ++j) f[0][j].u = read(j);
#pragma unroll
  for (int base = 0; base < N; base += B) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < B; ++j)
      if (base + B + j < N) f[(base / B + 1) % 2][j].u = read(base + B + j);
#pragma unroll
    for (int j = 0; j < B; ++j)
      if (base + j < N) use(base + j, f[base / B % 2][j]);
  }
  __builtin_amdgcn_sched_barrier(0);
}

template <int KS, int CT>
constexpr size_t lat_lds_bytes() {  // two buffers each of rows, latents and scores
  return 2 * ((32 * (32 * KS + 8) + 16 * CT * 32) * sizeof(bf16_t) + 4 * 16 * 36 * sizeof(float));
}

template <int KS, int CT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, CT <= 8 ? 4 : 2))) void latent_attention_mfma_kernel(
    const float* __restrict__ q_lat, const bf16_t* __restrict__ kpages, const bf16_t* __restrict__ vpages,
    const int32_t* __restrict__ tiles, const int32_t* __restrict__ block_table, int table_width, int page_size,
    int n_heads, float scale_log2, int n_splits, const float* __restrict__ sink, float* __restrict__ out, float* __restrict__ ws_o,
    float* __restrict__ ws_ml) {
  constexpr int WIDTH = 32 * KS, RANK = 16 * CT, HALF = CT / 2;
  // LDS: rows 16 bytes longer than their elements, latents' four pieces of 16 bytes turned by their
  // column's number, scores in rows of 36: 16 lanes that read a piece of neighbouring rows meet different banks
  constexpr int KROW = WIDTH + 8, SROW = 36;
  constexpr int KP = 32 * WIDTH / 8, VP = RANK * 4;  // 16-byte pieces of a group: page rows, transposed latents
  constexpr int KN = (KP + 511) / 512, VN = (VP + 511) / 512;
  extern __shared__ __attribute__((aligned(16))) bf16_t lat_lds[];
  auto kbuf = [&](int b) { return lat_lds + b * (32 * KROW); };
  auto vbuf = [&](int b) { return lat_lds + 2 * 32 * KROW + b * (RANK * 32); };
  float* sbase = reinterpret_cast<float*>(lat_lds + 2 * 32 * KROW + 2 * RANK * 32);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int pair = wave / 2, half = wave % 2;
  auto sbuf = [&](int b) { return sbase + (b * 4 + pair) * (16 * SROW); };
  const int tile_i = blockIdx.x;
  const int r = lane % 16, g = lane / 16;
  const int32_t* tile = tiles + 4 * tile_i;
  const int seq = tile[0], tok0 = tile[1], count = tile[2], pos0 = tile[3];
  const int chunk = blockIdx.y, split = blockIdx.z;
  const int hpt = n_heads < kLatCols ? n_heads : kLatCols;
  const int col = 16 * pair + r, tt = col / hpt, hh = col % hpt, head = chunk * kLatCols + hh;
  const bool col_ok = tt < count && head < n_heads;
  const bool wave_ok = 16 * pair < count * hpt;  // (a pair without columns only helps to park)
  const int my_pos = pos0 + (col_ok ? tt : 0);
  const int last = pos0 + count - 1;

  LatFrag qf[KS];
  {
    const float* qp = q_lat + (static_cast<size_t>(tok0 + (col_ok ? tt : 0)) * n_heads + (col_ok ? head : 0)) * WIDTH + 8 * g;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const float4 a = *reinterpret_cast<const float4*>(qp + 32 * ks), b = *reinterpret_cast<const float4*>(qp + 32 * ks + 4);
      qf[ks].u[0] = col_ok ? pack_bf16x2(a.x, a.y) : 0u;
      qf[ks].u[1] = col_ok ? pack_bf16x2(a.z, a.w) : 0u;
      qf[ks].u[2] = col_ok ? pack_bf16x2(b.x, b.y) : 0u;
      qf[ks].u[3] = col_ok ? pack_bf16x2(b.z, b.w) : 0u;
    }
  }
  const int groups = last / 32 + 1;
  const int per = (groups + n_splits - 1) / n_splits;
  const int g_lo = min(groups, split * per), g_hi = min(groups, g_lo + per);
  const int32_t* bt = block_table + static_cast<size_t>(seq) * table_width;

  float m = -INFINITY, l = 0.f;
  lat_f32x4_t acc[HALF];
#pragma unroll
  for (int ct = 0; ct < HALF; ++ct) acc[ct] = lat_f32x4_t{0.f, 0.f, 0.f, 0.f};

  lat_u32x4_t kreg[KN], vreg[VN] = {};
  auto page_of = [&](int grp) { return static_cast<size_t>(bt[grp * 32 / page_size]); };
  // (a uniform base and a 32-bit offset in bytes: one register an address)
  auto fetch_k = [&](int grp) {
    const int k0 = grp * 32;
    const char* kp = reinterpret_cast<const char*>(kpages + (page_of(grp) * page_size + k0 % page_size) * WIDTH);
#pragma unroll
    for (int i = 0; i < KN; ++i) {
      const uint32_t e = threadIdx.x + 512 * i;  // rows that do not exist yet: the last one that does
      if (KP % 512 == 0 || e < KP)
        kreg[i] = *reinterpret_cast<const lat_u32x4_t*>(kp + (min(e / (WIDTH / 8), static_cast<uint32_t>(last - k0)) * (WIDTH * 2) + e % (WIDTH / 8) * 16));
    }
  };
  auto park_k = [&](int b) {
#pragma unroll
    for (int i = 0; i < KN; ++i) {
      const int e = threadIdx.x + 512 * i;
      if (KP % 512 == 0 || e < KP) *reinterpret_cast<lat_u32x4_t*>(kbuf(b) + e / (WIDTH / 8) * KROW + e % (WIDTH / 8) * 8) = kreg[i];
    }
  };
  const uint32_t v_row = 2 * page_size;
  auto fetch_v = [&](int grp) {
    const char* vp = reinterpret_cast<const char*>(vpages + page_of(grp) * RANK * page_size + grp * 32 % page_size);
#pragma unroll
    for (int i = 0; i < VN; ++i) {
      const uint32_t e = threadIdx.x + 512 * i;
      if (VP % 512 == 0 || e < VP) vreg[i] = *reinterpret_cast<const lat_u32x4_t*>(vp + (e / 4 * v_row + e % 4 * 16));
    }
  };
  auto park_v = [&](int b, int grp) {
    const int key_max = last - grp * 32, seen_by_all = pos0 - grp * 32;
    if (seen_by_all < 31) {
      // Slots behind the last key hold whatever was there; and a later token's latents meet the weights 0 of the tile's earlier ones:
      // what is not finite in them must not make NaN of these.  (The columns that see the token have its score from the page row.)
      uint32_t full = 0;
#pragma unroll
      for (int i = 0; i < VN; ++i) {
        const int key0 = threadIdx.x % 4 * 8;
        LatFrag f;
        f.u = vreg[i];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (key0 + j > key_max) f.h[j] = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) full |= (f.u[j] & 0x7f807f80u) + 0x00800080u;  // (an exponent of ones carries)
        vreg[i] = f.u;
      }
      if (count > 1 && __any((full & 0x80008000u) != 0)) {
#pragma unroll
        for (int i = 0; i < VN; ++i) {
          LatFrag f;
          f.u = vreg[i];
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (threadIdx.x % 4 * 8 + j > seen_by_all && (f.h[j] & 0x7f80) == 0x7f80) f.h[j] = 0;
          vreg[i] = f.u;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < VN; ++i) {
      const int e = threadIdx.x + 512 * i;
      if (VP % 512 == 0 || e < VP) {
        *reinterpret_cast<lat_u32x4_t*>(vbuf(b) + e / 4 * 32 + ((e % 4) ^ (e / 16 % 4)) * 8) = vreg[i];
      }
    }
  };
  // this wave's 16 keys of a group against its columns: lane (r, g) gets column r, keys 16 half + 4 g .. + 3
  auto scores = [&](int b, int grp) {
    const bf16_t* krow = kbuf(b) + (16 * half + r) * KROW + 8 * g;
    lat_f32x4_t s0 = {0.f, 0.f, 0.f, 0.f};
    lat_read_ahead<KS>([&](int ks) { return *reinterpret_cast<const lat_u32x4_t*>(krow + 32 * ks); },
                       [&](int ks, const LatFrag& kf) { s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf.v, qf[ks].v, s0, 0, 0, 0); });
    const int key = grp * 32 + 16 * half + 4 * g;
#pragma unroll
    for (int j = 0; j < 4; ++j) s0[j] = key + j <= my_pos ? s0[j] * scale_log2 : -INFINITY;
    *reinterpret_cast<lat_f32x4_t*>(sbuf(b) + r * SROW + 16 * half + 4 * g) = s0;
  };
  // Nothing in the walk is conditional: before the last group it fetches and parks that group's rows once more, unread.  The last group is
  // a turn of its own, which fetches, parks and scores nothing (as another turn of the walk it cost 0.5 to 1.7 us a call: one token behind
  // ten keys, latent 64, 4.5 -> 3.7 us; eight, latent 512, 11.0 -> 9.5).
  const int g_end = g_hi - 1;
  if (g_lo < g_hi) {
    fetch_k(g_lo);
    fetch_v(g_lo);
    park_k(0);
    park_v(0, g_lo);
    if (g_lo < g_end) fetch_k(g_lo + 1);
    __syncthreads();
    if (wave_ok) scores(0, g_lo);
    if (g_lo < g_end) park_k(1);
  }
  auto turn = [&](int grp, auto is_last) {
    constexpr bool LAST = decltype(is_last)::value;
    const int b = (grp - g_lo) & 1;
    if (!LAST) {
      fetch_k(min(grp + 2, g_end));
      fetch_v(grp + 1);
    }
    // the rows of the next group, the latents and scores of this one are parked, and every wave is done with what is
    // written below: the rows and latents of this group's and the next one's buffers as they were two groups ago
    __syncthreads();
    if (wave_ok) {
      if (!LAST) scores(b ^ 1, grp + 1);
      // this lane: column r, keys 8 g .. 8 g + 7 of the group
      lat_f32x4_t s[2];
      s[0] = *reinterpret_cast<const lat_f32x4_t*>(sbuf(b) + r * SROW + 8 * g);
      s[1] = *reinterpret_cast<const lat_f32x4_t*>(sbuf(b) + r * SROW + 8 * g + 4);
      float tmax = -INFINITY;
#pragma unroll
      for (int sb = 0; sb < 2; ++sb)
#pragma unroll
        for (int j = 0; j < 4; ++j) tmax = fmaxf(tmax, s[sb][j]);
      tmax = column_lanes_max(tmax);
      const float m_new = fmaxf(m, tmax);
      const float m_safe = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = __builtin_amdgcn_exp2f(m - m_safe);
      float psum = 0.f;
      LatFrag pf;
#pragma unroll
      for (int sb = 0; sb < 2; ++sb) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          s[sb][j] = __builtin_amdgcn_exp2f(s[sb][j] - m_safe);
          psum += s[sb][j];
        }
        pf.u[2 * sb] = pack_bf16x2(s[sb][0], s[sb][1]);
        pf.u[2 * sb + 1] = pack_bf16x2(s[sb][2], s[sb][3]);
      }
      const bool grew = m_new > m;
      l = l * alpha + psum;
      m = m_new;
      if (__any(grew)) {
        asm volatile("" ::: "memory");  // (a branch, not a multiplication and a select per element)
#pragma unroll
        for (int ct = 0; ct < HALF; ++ct) acc[ct] *= alpha;
      }
      const bf16_t* vcol = vbuf(b) + (16 * HALF * half + r) * 32 + (g ^ (r / 4)) * 8;
      lat_read_ahead<HALF>([&](int ct) { return *reinterpret_cast<const lat_u32x4_t*>(vcol + 16 * ct * 32); },
                           [&](int ct, const LatFrag& vf) { acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf.v, pf.v, acc[ct], 0, 0, 0); });
    }
    if (!LAST) {
      park_k(b);
      park_v(b ^ 1, grp + 1);
    }
  };
  for (int grp = g_lo; grp < g_end; ++grp) turn(grp, std::false_type{});
  if (g_lo < g_hi) turn(g_end, std::true_type{});
  if (!col_ok && !__any(col_ok)) return;  // (uniform: the sum below exchanges lanes)
  l = column_lanes_sum(l);
  if (!col_ok) return;
  // acc[ct][j]: latent column 16 (HALF half + ct) + 4 g + j of this lane's column r
  if (n_splits == 1) {
    // the sink joins the sum of weights at the end (every column has seen a key: m is finite)
    if (sink != nullptr) l += __builtin_amdgcn_exp2f(sink[head] * 1.4426950408889634f - m);
    const float inv = 1.f / l;
    float* o = out + (static_cast<size_t>(tok0 + tt) * n_heads + head) * RANK + 16 * HALF * half + 4 * g;
#pragma unroll
    for (int ct = 0; ct < HALF; ++ct)
      *reinterpret_cast<float4*>(o + 16 * ct) = make_float4(acc[ct][0] * inv, acc[ct][1] * inv, acc[ct][2] * inv, acc[ct][3] * inv);
    return;
  }
  const size_t part = (static_cast<size_t>(tile_i) * gridDim.y + chunk) * n_splits + split;
  float* o = ws_o + (part * kLatCols + col) * RANK + 16 * HALF * half + 4 * g;
#pragma unroll
  for (int ct = 0; ct < HALF; ++ct) *reinterpret_cast<float4*>(o + 16 * ct) = make_float4(acc[ct][0], acc[ct][1], acc[ct][2], acc[ct][3]);
  if (g == 0 && half == 0) {
    ws_ml[(part * kLatCols + col) * 2] = m;
    ws_ml[(part * kLatCols + col) * 2 + 1] = l;
  }
}

// one workgroup per (tile, head chunk, column): the column's splits merged with weights 2^(m_s - max m), in
// the order of s; the weights are made once, by the first threads, and every thread's loads of a latent
// column's parts are asked for together
__global__ __launch_bounds__(128) void latent_attention_merge_kernel(const float* __restrict__ ws_o, const float* __restrict__ ws_ml,
                                                                     const int32_t* __restrict__ tiles, int n_heads, int rank,
                                                                     int n_splits, const float* __restrict__ sink,
                                                                     float* __restrict__ out) {
  __shared__ float w[256];
  __shared__ float inv_den;
  const int tile_i = blockIdx.x, chunk = blockIdx.y, r = blockIdx.z;
  const int32_t* tile = tiles + 4 * tile_i;
  const int tok0 = tile[1], count = tile[2];
  const int hpt = n_heads < kLatCols ? n_heads : kLatCols;
  const int tt = r / hpt, head = chunk * kLatCols + r % hpt;
  if (tt >= count || head >= n_heads) return;
  const size_t part0 = (static_cast<size_t>(tile_i) * gridDim.y + chunk) * n_splits;
  if (threadIdx.x < kWave) {
    float m_max = -INFINITY;
    for (int s = threadIdx.x; s < n_splits; s += kWave) m_max = fmaxf(m_max, ws_ml[((part0 + s) * kLatCols + r) * 2]);
    m_max = wave_max(m_max);
    float den = 0.f;
    for (int s = threadIdx.x; s < n_splits; s += kWave) {
      const float ws = exp2f(ws_ml[((part0 + s) * kLatCols + r) * 2] - m_max);
      w[s] = ws;
      den = fmaf(ws, ws_ml[((part0 + s) * kLatCols + r) * 2 + 1], den);
    }
    den = wave_sum(den);
    if (sink != nullptr) den += exp2f(sink[head] * 1.4426950408889634f - m_max);
    if (threadIdx.x == 0) inv_den = 1.f / den;
  }
  __syncthreads();
  float* o = out + (static_cast<size_t>(tok0 + tt) * n_heads + head) * rank;
  for (int c = 4 * threadIdx.x; c < rank; c += 4 * blockDim.x) {
    float4 num = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s0 = 0; s0 < n_splits; s0 += 8) {
      float4 v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (s0 + j < n_splits) v[j] = *reinterpret_cast<const float4*>(ws_o + ((part0 + s0 + j) * kLatCols + r) * rank + c);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (s0 + j < n_splits) {
          const float ws = w[s0 + j];
          num.x = fmaf(ws, v[j].x, num.x); num.y = fmaf(ws, v[j].y, num.y);
          num.z = fmaf(ws, v[j].z, num.z); num.w = fmaf(ws, v[j].w, num.w);
        }
    }
    *reinterpret_cast<float4*>(o + c) = make_float4(num.x * inv_den, num.y * inv_den, num.z * inv_den, num.w * inv_den);
  }
}

// sizes the matrix-core form is built for: (page row, latent) = (576, 512), (320, 256), (160, 128), (96, 64), and
// rows that are the latent alone (no rotated part) of 512, 256, 128 or 64 elements
extern "C" int yk_latent_mfma_ok(int kv_rank, int rot_dim, int page_size) {
  const int w = kv_rank + rot_dim;
  const bool size_ok = (w == 576 && kv_rank == 512) || (w == 320 && kv_rank == 256) || (w == 160 && kv_rank == 128) ||
                       (w == 96 && kv_rank == 64) ||
                       (rot_dim == 0 && (kv_rank == 512 || kv_rank == 256 || kv_rank == 128 || kv_rank == 64));
  return size_ok && page_size % 32 == 0 ? 1 : 0;
}

extern "C" int yk_latent_mfma_tile_tokens(int n_heads) { return n_heads >= kLatCols ? 1 : kLatCols / n_heads; }

// floats of workspace a launch with these tiles and splits needs
extern "C" size_t yk_latent_mfma_workspace(int n_tiles, int n_heads, int kv_rank, int n_splits) {
  if (n_splits <= 1) return 0;
  const size_t parts = static_cast<size_t>(n_tiles) * ((n_heads + kLatCols - 1) / kLatCols) * n_splits;
  return parts * kLatCols * (kv_rank + 2);
}

extern "C" int yk_latent_attention_mfma(const float* q_lat, const void* kpages, const void* vpages, const int32_t* tiles,
                                        int n_tiles, const int32_t* block_table, int table_width, int page_size, int n_heads,
                                        int kv_rank, int rot_dim, float scale, int n_splits, const float* sink, float* workspace,
                                        size_t workspace_floats, float* out, hipStream_t stream) {
  YK_REQUIRE(yk_latent_mfma_ok(kv_rank, rot_dim, page_size), "latent_attention_mfma: sizes the matrix-core form is not built for");
  YK_REQUIRE(n_tiles >= 0 && n_heads > 0 && table_width > 0 && n_splits >= 1 && n_splits <= 256, "latent_attention_mfma: bad sizes");
  YK_REQUIRE(workspace_floats >= yk_latent_mfma_workspace(n_tiles, n_heads, kv_rank, n_splits) && (n_splits == 1 || workspace != nullptr),
             "latent_attention_mfma: the workspace is too small");
  if (n_tiles == 0) return 0;
  const int chunks = (n_heads + kLatCols - 1) / kLatCols;
  dim3 grid(n_tiles, chunks, n_splits);
  const float scale_log2 = scale * 1.4426950408889634f;
  float* ws_o = workspace;
  float* ws_ml = workspace == nullptr ? nullptr : workspace + static_cast<size_t>(n_tiles) * chunks * n_splits * kLatCols * kv_rank;
#define YK_CASE(KS, CT)                                                                                                      \
  if (kv_rank + rot_dim == 32 * KS && kv_rank == 16 * CT) {                                                                  \
    auto kern = latent_attention_mfma_kernel<KS, CT>;                                                                        \
    constexpr size_t lds = lat_lds_bytes<KS, CT>();                                                                          \
    if (lds > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, \
                                               static_cast<int>(lds)) != hipSuccess)                                         \
      return yk_fail("latent_attention_mfma: the group's buffers do not fit in LDS");                                        \
    kern<<<grid, 512, lds, stream>>>(                                                                                        \
        q_lat, static_cast<const bf16_t*>(kpages), static_cast<const bf16_t*>(vpages), tiles, block_table,                   \
        table_width, page_size, n_heads, scale_log2, n_splits, sink, out, ws_o, ws_ml);                                            \
    if (yk_check_launch("latent_attention_mfma") != 0) return -1;                                                            \
  }
  YK_CASE(18, 32)
  YK_CASE(10, 16)
  YK_CASE(5, 8)
  YK_CASE(3, 4)
  YK_CASE(16, 32)
  YK_CASE(8, 16)
  YK_CASE(4, 8)
  YK_CASE(2, 4)
#undef YK_CASE
  if (n_splits > 1) {
    latent_attention_merge_kernel<<<dim3(n_tiles, chunks, kLatCols), 128, 0, stream>>>(ws_o, ws_ml, tiles, n_heads, kv_rank, n_splits, sink, out);
    return yk_check_launch("latent_attention_merge");
  }
  return 0;
}
