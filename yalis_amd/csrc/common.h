// Shared helpers of the HIP kernels: bfloat16 storage, wave and block reductions,
// error reporting of the C interface.
//
// Conventions of the library: every entry point is extern "C", takes raw device
// pointers and sizes plus the stream to launch on, checks its arguments on the host
// (a size a kernel cannot take is refused with a message, never computed wrongly),
// returns 0 on success and a negative number on failure; yk_last_error() returns the
// message.  dtype codes: 0 = float32, 1 = bfloat16.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#define YK_F32 0
#define YK_BF16 1

typedef uint16_t bf16_t;  // bfloat16 storage

std::string& yk_error_slot();
int yk_fail(const std::string& msg);
int yk_check_launch(const char* what);

#define YK_REQUIRE(cond, msg)        \
  do {                               \
    if (!(cond)) return yk_fail(msg); \
  } while (0)

__device__ __forceinline__ float bf16_to_f32(bf16_t x) {
  return __uint_as_float(static_cast<uint32_t>(x) << 16);
}

// Over the four lanes r, r + 16, r + 32 and r + 48 (the lanes that share a column of a 16 x 16
// matrix-core tile): the maximum, or the sum, in all four of them.  The swaps of half-waves and
// of rows of 16 lanes move registers directly; a shuffle would go through the LDS pipe and
// wait on its counter together with the operand reads.
__device__ __forceinline__ float column_lanes_max(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float column_lanes_sum(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// max(x, 0) + log1p(u), u = e^-|x|.  log1p(u) is 2 atanh(u / (2 + u)): the quotient with its remainder, the series' tail fitted over
// its range (to 1e-10 of the sum).  Against 64 bits, four million normal x of deviation 4: largest error 1.17e-7 of the result as with
// log1pf, mean 2.54e-8 (2.55e-8), in some 35 instructions where that took 120, one after the other.
__device__ __forceinline__ float softplus_f32(float x) {
  const float u = expf(-fabsf(x)), w = 2.f + u, left = u - (w - 2.f), inverse = __builtin_amdgcn_rcpf(w);
  const float q = u * inverse, z = q * q, rest = fmaf(-q, left, fmaf(-q, w, u)) * inverse;
  const float tail = fmaf(z, fmaf(z, fmaf(z, fmaf(z, 0.121287405f, 0.107200928f), 0.143078059f), 0.199994653f), 0.333333373f);
  return fmaf(2.f, q + fmaf(q * z, tail, rest), fmaxf(x, 0.f));
}

// two floats to two bfloat16 (round to nearest even; NaN stays NaN) in one word: gfx950
// converts in hardware (v_cvt_pk_bf16_f32), one instruction where the shifts and adds of a
// conversion by hand take six (measured: 2 us of a 41 us product that converted its staged rows)
typedef __bf16 yk_bf16x2_t __attribute__((ext_vector_type(2)));
typedef float yk_f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  union {
    yk_bf16x2_t v;
    uint32_t u;
  } c;
  c.v = __builtin_convertvector(yk_f32x2_t{lo, hi}, yk_bf16x2_t);
  return c.u;
}

__device__ __forceinline__ bf16_t f32_to_bf16(float f) { return static_cast<bf16_t>(pack_bf16x2(f, 0.f) & 0xffffu); }

template <typename T>
__device__ __forceinline__ float to_f32(T x);
template <>
__device__ __forceinline__ float to_f32<float>(float x) {
  return x;
}
template <>
__device__ __forceinline__ float to_f32<bf16_t>(bf16_t x) {
  return bf16_to_f32(x);
}

template <typename T>
__device__ __forceinline__ T from_f32(float x);
template <>
__device__ __forceinline__ float from_f32<float>(float x) {
  return x;
}
template <>
__device__ __forceinline__ bf16_t from_f32<bf16_t>(float x) {
  return f32_to_bf16(x);
}

constexpr int kWave = 64;

// ------------------------------------------------------------------ layout of a cache page
// A page holds, for every kv head, a slab of page_size x head_dim keys and one of values.
// Plain slabs: keys [slot][dim], values transposed [dim][slot].
// Tiled slabs (bfloat16, a head size the matrix-core attention takes, pages of a multiple of
// 64 tokens): the slab is cut into blocks of 64 slots, and a block is stored as the 16-byte
// pieces that the matrix-core attention loads, in the order of the lanes that load them, so
// that one wave-wide load reads 1 KiB of consecutive memory:
//   keys:   piece (((u*2 + sb) * head_dim/32 + ks) * 4 + g) * 16 + r holds dims 32ks + 8g .. 8g+7
//           of slot 32u + 8(r/4) + 4sb + r%4 (the row order of the two score products of a
//           group of 32 keys),
//   values: piece ((u * head_dim/16 + dt) * 4 + g) * 16 + r holds slots 32u + 8g .. 8g+7 of dim
//           16dt + r.
// Writers (rotary + append) and readers (the attention kernels) go through these functions.
__host__ __device__ inline bool cache_is_tiled(int dtype, int head_dim, int page_size) {
  return dtype == YK_BF16 && (head_dim == 64 || head_dim == 128) && page_size % 64 == 0;
}
// element offsets within a slab
__host__ __device__ inline size_t cache_k_offset(bool tiled, int page_size, int head_dim, int slot, int d) {
  if (!tiled) return static_cast<size_t>(slot) * head_dim + d;
  const int j = slot % 64, u = j / 32, r = 4 * ((j % 32) / 8) + j % 4, sb = (j % 8) / 4;
  const int piece = (((u * 2 + sb) * (head_dim / 32) + d / 32) * 4 + (d % 32) / 8) * 16 + r;
  return static_cast<size_t>(slot / 64) * 64 * head_dim + piece * 8 + d % 8;
}
__host__ __device__ inline size_t cache_v_offset(bool tiled, int page_size, int head_dim, int slot, int d) {
  if (!tiled) return static_cast<size_t>(d) * page_size + slot;
  const int j = slot % 64, u = j / 32, g = (j % 32) / 8;
  const int piece = ((u * (head_dim / 16) + d / 16) * 4 + g) * 16 + d % 16;
  return static_cast<size_t>(slot / 64) * 64 * head_dim + piece * 8 + j % 8;
}

// Four neighbouring values: as they lie in memory, as float32, and back.  A load under a condition (a weight that may be absent) is kept
// as it lies until the condition's end: widened under it, it would be waited for there.
template <typename T>
struct Four;
template <>
struct Four<float> {
  typedef float4 raw;
  static __device__ __forceinline__ raw at(const float* p) { return *reinterpret_cast<const float4*>(p); }
  static __device__ __forceinline__ raw all(float v) { return make_float4(v, v, v, v); }
  static __device__ __forceinline__ float4 wide(raw r) { return r; }
  static __device__ __forceinline__ void put(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
};
template <>
struct Four<bf16_t> {
  typedef uint2 raw;
  static __device__ __forceinline__ raw at(const bf16_t* p) { return *reinterpret_cast<const uint2*>(p); }
  static __device__ __forceinline__ raw all(float v) { return make_uint2(pack_bf16x2(v, v), pack_bf16x2(v, v)); }
  static __device__ __forceinline__ float4 wide(raw r) {
    return make_float4(__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xffff0000u), __uint_as_float(r.y << 16),
                       __uint_as_float(r.y & 0xffff0000u));
  }
  static __device__ __forceinline__ void put(bf16_t* p, float4 v) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
  }
};
template <typename T>
__device__ __forceinline__ float4 four_at(const T* p) {
  return Four<T>::wide(Four<T>::at(p));
}
template <typename T>
__device__ __forceinline__ void put_four(T* p, float4 v) {
  Four<T>::put(p, v);
}

// `left` slices of IT pieces of four values (`at` elements from p, which is the same in every lane), `stride` elements from one slice to the next, added to s in the slices' order.  SL of
// them (at most) are asked for before the first is used: a kernel of a few microseconds lasts as long as the waits for memory it makes
// one after another, and the compiler moves a load to the condition that its value alone is used under, and waits there.  So they are
// asked for in groups (one, two, four, eight: few slices ask for few), inside a group unconditionally; what lies beyond the last
// slice is read from the last and masked to +0 with a number that the compiler cannot take for a condition (a sum that began
// with +0 is never -0, and +0 leaves it as it is).  ask_slices and join_slices are the two halves, for kernels that have more to ask for in
// between.
template <int SL, int IT, typename T, int FROM = 0, int TO = 1>
__device__ __forceinline__ void ask_slices(const T* p, const uint32_t (&at)[IT], int left, size_t stride, typename Four<T>::raw (&d)[SL][IT]) {
#pragma unroll
  for (int j = FROM; j < TO; ++j) {
#pragma unroll
    for (int k = 0; k < IT; ++k) d[j][k] = Four<T>::at(p + at[k]);
    p += j + 1 < left ? stride : 0;
  }
  if constexpr (TO < SL) {
    if (left > TO) ask_slices<SL, IT, T, TO, 2 * TO>(p, at, left, stride, d);
  }
}
template <int SL, int IT, typename T, int FROM = 0, int TO = 1>
__device__ __forceinline__ void join_slices(const typename Four<T>::raw (&d)[SL][IT], int left, float4 (&s)[IT]) {
#pragma unroll
  for (int j = FROM; j < TO; ++j) {
    const uint32_t keep = __builtin_amdgcn_readfirstlane((j - left) >> 31);
    auto kept = [&](float v) { return __uint_as_float(__float_as_uint(v) & keep); };
#pragma unroll
    for (int k = 0; k < IT; ++k) {
      const float4 v = Four<T>::wide(d[j][k]);
      s[k].x += kept(v.x);
      s[k].y += kept(v.y);
      s[k].z += kept(v.z);
      s[k].w += kept(v.w);
    }
  }
  if constexpr (TO < SL) {
    if (left > TO) join_slices<SL, IT, T, TO, 2 * TO>(d, left, s);
  }
}
// The rest of the slices after the first SL have joined, SL at a time.
template <int SL, int IT, typename T>
__device__ __forceinline__ void join_rest(const T* p, const uint32_t (&at)[IT], int left, size_t stride, float4 (&s)[IT]) {
  if constexpr (sizeof(T) == 4) {  // (slices are float32)
    for (left -= SL; left > 0; left -= SL) {
      typename Four<T>::raw d[SL][IT];
      p += SL * stride;
      ask_slices<SL, IT, T>(p, at, left, stride, d);
      join_slices<SL, IT, T>(d, left, s);
    }
  }
}
// Slices asked for at a time by a kernel with IT pieces a thread, where rows are few and where they fill the chip.  Few rows are bound by their waits,
// many by how many waves a unit holds: registers of slices that are not there, or more than a workgroup of 1,024 threads has (128), cost more
// than waits.  With the registers of many slices everywhere / now, float32 rows, us: one row of 10,240 and its residual's norm (spilled) 8.2 / 3.9, 2,048 of
// them 86 / 43, 500 of 8,192 9.7 / 7.7, 2,048 normed alone 21.4 / 17.0; 1,023 rows of 4,096 as two terms 15.8 / 11.7.
enum SlicesAtOnce { kOneSlice, kManyRows, kFewRows };
template <SlicesAtOnce HOW, int IT>
constexpr int slices_at_once = HOW == kOneSlice ? 1 : HOW == kManyRows ? (IT == 1 ? 4 : 2) : (IT == 1 ? 16 : 8);
inline SlicesAtOnce slices_how(int n_splits, size_t n_rows) { return n_splits <= 1 ? kOneSlice : n_rows > 256 ? kManyRows : kFewRows; }
// The sum over n >= 1 slices (kOneSlice: one) of IT pieces of four values, `at` elements from p.
template <SlicesAtOnce HOW, int IT, typename T>
__device__ __forceinline__ void sum_slices(const T* p, const uint32_t (&at)[IT], int n, size_t stride, float4 (&s)[IT]) {
  constexpr int SL = slices_at_once<HOW, IT>;
#pragma unroll
  for (int k = 0; k < IT; ++k) s[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  do {
    typename Four<T>::raw d[SL][IT];
    ask_slices<SL, IT, T>(p, at, n, stride, d);
    join_slices<SL, IT, T>(d, n, s);
    p += SL * stride;
    n -= SL;
  } while (SL > 1 && n > 0);
}
// Arguments that did not come with the launch, asked for here and not where they are first used, one wait after the other.
__device__ __forceinline__ void arguments_now(const void* a, const void* b = nullptr, const void* c = nullptr, const void* d = nullptr) {
  asm volatile("" ::"s"(a), "s"(b), "s"(c), "s"(d));
}

// Sums and maxima over a wave's 64 lanes, all of them active, in every lane: partners 32, 16, 8, 4, 2 and 1 lanes away, as moves between
// registers (half-waves and rows of 16 swapped, rows rotated, quads permuted).  The same additions as with six shuffles, which go
// through the LDS pipe and wait for it one after the other (a row's norm of one decode step: eight slices to add, 4.7 -> 4.0 us).
template <int CTRL>
__device__ __forceinline__ float row_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// over the rows of 16 lanes alone
__device__ __forceinline__ float row_sum(float v) {
  v += row_move<0x128>(v);  // row_ror:8
  v += row_move<0x124>(v);  // row_ror:4
  v += row_move<0x4E>(v);   // quad_perm [2,3,0,1]
  return v + row_move<0xB1>(v);  // quad_perm [1,0,3,2]
}
__device__ __forceinline__ float row_max(float v) {
  v = fmaxf(v, row_move<0x128>(v));
  v = fmaxf(v, row_move<0x124>(v));
  v = fmaxf(v, row_move<0x4E>(v));
  return fmaxf(v, row_move<0xB1>(v));
}
__device__ __forceinline__ float wave_sum(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return row_sum(__uint_as_float(b[0]) + __uint_as_float(b[1]));
}
__device__ __forceinline__ float wave_max(float v) { return row_max(column_lanes_max(v)); }

// Lane i's 16 bytes at `at` + `lane_off` + `off` (zeros beyond `bytes`, against which both offsets count) to place i of the KiB of LDS at `to`.
__device__ __forceinline__ void load_to_lds(const void* at, int bytes, void* to, int lane_off, int off) {
#ifdef __HIP_DEVICE_COMPILE__  // the builtin takes 16 bytes for the device alone
  typedef __attribute__((address_space(3))) void lds_void_t;
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(at), 0, bytes, 0x00027000), (lds_void_t*)to, 16,
                                           lane_off, off, 0, 0);
#endif
}

// x / n for x from 0 and n from 2 up: by ceil(2^32 / n) the quotient is less than x / 2^32 too large before it is cut, so at most one
inline uint32_t inverse_of(int n) { return static_cast<uint32_t>(((1ull << 32) + n - 1) / n); }
__device__ __forceinline__ int divide_by(int x, int n, uint32_t inverse) {
  const uint32_t q = __umulhi(static_cast<uint32_t>(x), inverse);
  return static_cast<int>(q - (q * static_cast<uint32_t>(n) > static_cast<uint32_t>(x) ? 1u : 0u));
}

// Gated activations: 0 = silu, 1 = gelu (tanh form); float32.
__device__ __forceinline__ float act_silu(float z) { return z / (1.f + expf(-z)); }
__device__ __forceinline__ float act_gelu_tanh(float z) {
  const float k = 0.7978845608028654f;  // sqrt(2/pi)
  return 0.5f * z * (1.f + tanhf(k * (z + 0.044715f * z * z * z)));
}
__device__ __forceinline__ float act_apply(float z, int act) { return act == 0 ? act_silu(z) : act_gelu_tanh(z); }
// Plain activations: 0 = silu, 1 = gelu (tanh form), 2 = the square of relu.
#define YK_PLAIN_KINDS 3
__device__ __forceinline__ float act_plain(float z, int kind) {
  if (kind == 2) {
    const float r = fmaxf(z, 0.f);
    return r * r;
  }
  return act_apply(z, kind);
}
// A gated pair: what a feed-forward makes of a gate value g and an up value u.  Kinds 0 and 1:
// act(g) * u.  Kind 2, the clamped swish gate: g' = min(g, p0), u' = clamp(u, -p0, p0),
// g' * sigmoid(p1 * g') * (u' + 1) (p0 the limit, p1 the slope of the sigmoid).
#define YK_GATED_KINDS 3
__device__ __forceinline__ float gated_pair(float g, float u, int kind, float p0, float p1) {
  if (kind < 2) return act_apply(g, kind) * u;
  g = fminf(g, p0);
  u = fminf(fmaxf(u, -p0), p0);
  return g / (1.f + expf(-p1 * g)) * (u + 1.f);
}

// The sum of a product's K slices (or an accumulator) stands for the product's output: with
// `round_sum` it is rounded to bfloat16 as that output would have been, so that what follows
// rounds at the same places whether the product came reduced (bfloat16), as slices, or fused
// (and has the same bits where the same kernel made the sums).
__device__ __forceinline__ float as_output(float v, int round_sum) {
  return round_sum ? to_f32<bf16_t>(from_f32<bf16_t>(v)) : v;
}

// Rotation of a pair (a, b) by the angle with cosine c and sine s: a' = a c - b s, b' = b c + a s.
// One rounding of b*s (or a*s), then a fused multiply-add: written out so that every kernel
// that rotates (rotary + append on its own, or inside the attention launch) gives the same bits.
__device__ __forceinline__ float rot_first(float a, float b, float c, float s) { return fmaf(a, c, -__fmul_rn(b, s)); }
__device__ __forceinline__ float rot_second(float a, float b, float c, float s) { return fmaf(b, c, __fmul_rn(a, s)); }

// The first key that the query at position p sees: with a window, the window's first position; with `chunked`, the first
// position of the query's own chunk of `window` positions, counted from the sequence's start; without one, 0.
__host__ __device__ inline int first_visible(int p, int window, int chunked) {
  if (window <= 0) return 0;
  if (chunked) return p - p % window;
  return p - window + 1 > 0 ? p - window + 1 : 0;
}

// ------------------------------------------------ attention whose keys were split across workgroups
// Heads of one kv head that share a wave of the matrix-core attention (its 16 columns hold
// 16 / heads_per_tile tokens of those heads); a kv group with more heads takes several
// chunks of them.
__host__ __device__ inline int attn_heads_per_tile(int n_heads, int n_kv) {
  const int qpk = n_heads / n_kv;
  return qpk < 16 ? qpk : 16;
}

// What the splits of a launch leave behind: for every group of 16 columns and split, the
// unnormalised outputs [16][head_dim] in `o` and (running maximum, sum) pairs [16][2] in `ml`,
// groups numbered (tile * groups_y + kv head * chunks + chunk) * n_splits + split.
// Four consecutive output elements of one column, merged over its splits: weights
// exp2(m_s - max m), in the order of s.  `col0` is the column's index in split 0
// (group * 16 + column); split s lies 16 columns further each.  `sink_log2` (-inf: none): a term 2^sink_log2 that joins
// the sum of weights once, with no output of its own.
// Up to MERGE_AT_ONCE splits are all asked for before any is used (in groups, as ask_slices does it: what lies beyond the last is read
// from the last and masked to zero).
constexpr int MERGE_AT_ONCE = 8;
template <int FROM = 0, int TO = 1>
__device__ __forceinline__ void merge_ask(const float* o, const float* ml, int n_splits, size_t o_stride, float2 (&w)[MERGE_AT_ONCE],
                                          float4 (&v)[MERGE_AT_ONCE]) {
#pragma unroll
  for (int j = FROM; j < TO; ++j) {
    w[j] = *reinterpret_cast<const float2*>(ml);
    v[j] = *reinterpret_cast<const float4*>(o);
    ml += j + 1 < n_splits ? 32 : 0;
    o += j + 1 < n_splits ? o_stride : 0;
  }
  if constexpr (TO < MERGE_AT_ONCE) {
    if (n_splits > TO) merge_ask<TO, 2 * TO>(o, ml, n_splits, o_stride, w, v);
  }
}
template <int FROM = 0, int TO = 1>
__device__ __forceinline__ float merge_max(int n_splits, const float2 (&w)[MERGE_AT_ONCE], float m_max) {
#pragma unroll
  for (int j = FROM; j < TO; ++j) m_max = fmaxf(m_max, w[j].x);
  if constexpr (TO < MERGE_AT_ONCE) {
    if (n_splits > TO) return merge_max<TO, 2 * TO>(n_splits, w, m_max);
  }
  return m_max;
}
template <int FROM = 0, int TO = 1>
__device__ __forceinline__ void merge_join(int n_splits, const float2 (&w)[MERGE_AT_ONCE], const float4 (&v)[MERGE_AT_ONCE], float m_max,
                                           float (&num)[4], float& den) {
#pragma unroll
  for (int j = FROM; j < TO; ++j) {
    const uint32_t keep = __builtin_amdgcn_readfirstlane((j - n_splits) >> 31);
    auto kept = [&](float x) { return __uint_as_float(__float_as_uint(x) & keep); };
    const float e = exp2f(w[j].x - m_max);
    num[0] += e * kept(v[j].x);
    num[1] += e * kept(v[j].y);
    num[2] += e * kept(v[j].z);
    num[3] += e * kept(v[j].w);
    den += e * kept(w[j].y);
  }
  if constexpr (TO < MERGE_AT_ONCE) {
    if (n_splits > TO) merge_join<TO, 2 * TO>(n_splits, w, v, m_max, num, den);
  }
}
__device__ __forceinline__ void attn_merge_splits(const float* __restrict__ o, const float* __restrict__ ml,
                                                  size_t col0, int n_splits, int head_dim, int d,
                                                  float out[4], float sink_log2 = -INFINITY) {
  const float* mlc = ml + col0 * 2;
  const float* oc = o + col0 * head_dim + d;
  float m_max = sink_log2;
  float num[4] = {0.f, 0.f, 0.f, 0.f};
  float den = 0.f;
  if (n_splits <= MERGE_AT_ONCE) {
    float2 w[MERGE_AT_ONCE];
    float4 v[MERGE_AT_ONCE];
    merge_ask(oc, mlc, n_splits, static_cast<size_t>(16) * head_dim, w, v);
    m_max = merge_max(n_splits, w, m_max);
    merge_join(n_splits, w, v, m_max, num, den);
  } else {
#pragma unroll 4
    for (int s = 0; s < n_splits; ++s) m_max = fmaxf(m_max, mlc[static_cast<size_t>(s) * 32]);
#pragma unroll 4
    for (int s = 0; s < n_splits; ++s) {
      const float w = exp2f(mlc[static_cast<size_t>(s) * 32] - m_max);
      const float4 v = *reinterpret_cast<const float4*>(oc + static_cast<size_t>(s) * 16 * head_dim);
      num[0] += w * v.x;
      num[1] += w * v.y;
      num[2] += w * v.z;
      num[3] += w * v.w;
      den += w * mlc[static_cast<size_t>(s) * 32 + 1];
    }
  }
  if (sink_log2 != -INFINITY) den += exp2f(sink_log2 - m_max);
  const float inv = 1.f / den;
#pragma unroll
  for (int e = 0; e < 4; ++e) out[e] = num[e] * inv;
}

// Sum, or maximum, over a block of whole waves, up to 1,024 threads; every thread gets the result.  `scratch` is shared memory for 16
// floats.  Every wave adds up the waves' sums by itself.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, nwaves = blockDim.x / kWave;
  __syncthreads();  // scratch may still be read from an earlier call
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  return row_sum(lane % 16 < nwaves ? scratch[lane % 16] : 0.f);
}

// The same with the number of waves given, for a scratch that nothing has used yet: one barrier less, and no load of the block's size.
__device__ __forceinline__ float block_sum_first(float v, float* scratch, int nwaves) {
  v = wave_sum(v);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  return row_sum(lane % 16 < nwaves ? scratch[lane % 16] : 0.f);
}

__device__ __forceinline__ float block_max(float v, float* scratch) {
  v = wave_max(v);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, nwaves = blockDim.x / kWave;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  return row_max(lane % 16 < nwaves ? scratch[lane % 16] : -INFINITY);
}
