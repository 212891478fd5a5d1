// Products of many rows: y = x . w^T, bfloat16 operands, float32 accumulation, in large tiles; K cut into slices where tiles are few, and
// gate/up products with their activation in the end.  The reference leaves these to its vendor library (yalis/external/model.py:449, 462-466,
// 717-722); so does this engine where the library is faster (plan()).
//
// What bounds it.  With every compute unit at work the card's power: the clock falls to 1.4 to 1.9 GHz, so what counts is what a product
// costs beside the matrix instructions.  v_mfma_f32_16x16x32_bf16 reads and writes fewer registers for the same products than 32x32x16 (8,192 x
// 28,672 x 4,096: 1,325 us where 32x32x16 takes 1,450), tiles of 256 x 256 fetch least, and workgroups of one die take tiles that share rows
// (L2 answers 4 of 5 reads).  Dies that start at different places of K spread their reads over the memory channels (1,325 -> 1,286).
// Loads go to LDS without registers between (a form with them, 128 x 128, ended at 0.4 to 0.77 PFLOP/s: 1,024 clocks of writes a
// step), and stand one by one between the matrix instructions: all at once behind the barrier the same product takes 5 to 7 % longer.
// One operand has a step more under way than the other, which is what LDS holds (2,048 x 6,144 x 4,096 as 192 x 256: 87 -> 77 us).
// With few tiles the memory's latency: slices along K put more under way.
// Measured in replayed graphs, weights from memory, with the norm that follows where slices are handed on (us, the library and the
// kernels for fewer rows before / this): 999 x 3,072 x 2,048 21.4 / 17.8, 797 x 4,096 x 4,096 39 / 33, 2,048 x 2,048 x 2,048 22 / 19, 2,048 x 1,360 x 2,048
// 20 / 16; slices: 150 x 3,072 x 8,192 29 / 23, 512 x 2,048 x 8,192 39 / 32, 999 x 4,096 x 14,336 151 / 114; gate/up with its activation: 256 x 16,384 x 3,072 45 /
// 35, 999 x 16,384 x 2,048 67 / 58, 3,985 x 16,384 x 3,072 321 / 299, 8,192 x 28,672 x 4,096 1,374 / 1,313.  Of 21,680 products (65 to
// 4,096 rows, 512 to 32,768 columns, K 512 to 28,672, spread over their logarithms) that earlier lines took the 16,470 still taken take 0.84 of the time that
// the other kernels and the library do (geometric mean), 228 of them more than 1.06 of it.
#include <algorithm>

#include "common.h"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// Until no more than VM loads and stores and LGKM LDS reads of this wave are under way (the builtin: the compiler then adds no waits of its
// own for those reads).
template <int VM, int LGKM>
__device__ __forceinline__ void wait_for() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4) << 14 | 7 << 4 | LGKM << 8);
}

enum { OUT_BF16 = 0, OUT_F32 = 1, OUT_GATED = 2, OUT_ACT = 3 };

// x * sigmoid(slope * x), within about three units of float32's last place: exp(y) as 2^(y log2 e) with the product's rounding carried
// along, unless the power is infinite (or y no number), which has no rest: the result is then zero (or no number), as a division's would be.
// A quarter of the divisor, so that its reciprocal is no subnormal number, which the instruction gives as zero.
__device__ __forceinline__ float swish(float x, float slope) {
  float y = -slope * x;
  y = y < -90.f ? -90.f : y;
  const float t = y * 1.44269504f;
  const float low = fmaf(y, 1.92596303e-8f, fmaf(y, 1.44269504f, -t));
  const float e = __builtin_amdgcn_exp2f(t);
  const float power = t < 128.f ? fmaf(e, low * 0.693147181f, e) : e;
  return 0.25f * x * __builtin_amdgcn_rcpf(fmaf(0.25f, power, 0.25f));
}
__device__ __forceinline__ float gated(float g, float u, int kind, float p0, float p1) {
  if (kind == 0) return swish(g, 1.f) * u;
  if (kind == 1) return gated_pair(g, u, 1, p0, p1);
  return swish(fminf(g, p0), p1) * (fminf(fmaxf(u, -p0), p0) + 1.f);
}

// A workgroup of WN x WM waves makes BN columns (rows of w) x BM rows of y over `per` steps of 64 along K.
//
// LDS: a step's rows of w, then of x, 128 bytes each, STAGES steps in flight.  buffer_load ... lds writes lane i's 16 bytes to
// place i of a KiB, so what is swapped is the address each lane reads from: piece c of row p lies at place c ^ (p / 2 % 8), with which
// the operand reads (16 rows x 64 bytes a wave) meet every bank once.  Row p of w's part holds row 32 (p / 32) + 8 (p / 4 % 4) +
// 4 (p / 16 % 2) + p % 4 of the tile: two products of 16 x 16 then leave eight consecutive columns of a row in a lane.
template <int BN, int BM, int WN, int WM, int SUB, int AHEAD, bool X_FIRST, int OUT>
__global__ __launch_bounds__(64 * WN * WM, 1) void gemm_block_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                     void* __restrict__ yv, int M, int N, int K, int ldx, int ldw, int ldy,
                                                                     int slices, int kind, float p0, float p1) {
  constexpr int NW = WN * WM, BK = 64 * SUB, FN = BN / WN / 16, FM = BM / WM / 16, WS = BN * 128, XS = BM * 128, WB = WS * SUB, XB = XS * SUB;
  constexpr int LW = BN / 8 / NW, LX = BM / 8 / NW, L = LW + LX, Q = FN * FM, R = FN + FM;
  // of one operand AHEAD steps lie in LDS, of the other, which is loaded half a step later, one more
  constexpr int SW = AHEAD + X_FIRST, SX = AHEAD + !X_FIRST, LF = X_FIRST ? LX : LW, LT = X_FIRST ? LW : LX;
  static_assert(BN % (8 * NW) == 0 && BM % (8 * NW) == 0 && (NW == 4 || NW == 8) && FN % 2 == 0 && (OUT != OUT_GATED || FN % 4 == 0), "tiles");
  __shared__ __attribute__((aligned(1024))) unsigned char lds[SW * WB + SX * XB];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  // The dies take turns with workgroups; each die gets a run of tiles, which its workgroups walk side by side; eight tiles of rows to a
  // band of tiles.
  const int tn = (N + BN - 1) / BN, tm = (M + BM - 1) / BM, flat = tn * tm, total = flat * slices, die = blockIdx.x % 8;
  const int mine = total / 8 + (die < total % 8), run0 = die * (total / 8) + min(die, total % 8);
  const int all = K / BK, per = (all + slices - 1) / slices;
  struct Tile {
    int m0, n0, slice, steps;
  };
  auto tile_of = [&](int at) {
    int t = run0 + at;
    const int slice = t / flat;
    t -= slice * flat;
    constexpr int BAND = 8;
    const int first = t / (BAND * tn) * BAND, high = min(BAND, tm - first), r = t - first * tn;
    return Tile{(first + r % high) * BM, r / high * BN, slice, min(per, all - slice * per)};
  };
  // a tile's rows of an operand: where they begin and how many bytes they reach over, behind which nothing is read (rows beyond N or M)
  struct Rows {
    const bf16_t* at;
    int bytes;
  };
  auto w_of = [&](const Tile& t) {
    return Rows{w + static_cast<size_t>(t.n0) * ldw + t.slice * per * BK, ((min(BN, N - t.n0) - 1) * ldw + t.steps * BK) * 2};
  };
  auto x_of = [&](const Tile& t) {
    return Rows{x + static_cast<size_t>(t.m0) * ldx + t.slice * per * BK, ((min(BM, M - t.m0) - 1) * ldx + t.steps * BK) * 2};
  };
  const int piece = 8 * ((lane & 7) ^ (4 * (wave & 1) + (lane >> 4)));
  const int wrow = 32 * (wave / 4) + 8 * (2 * (wave & 1) + (lane >> 5)) + 4 * (wave / 2 % 2) + ((lane >> 3) & 3);
  const int wvo = (wrow * ldw + piece) * 2, xvo = ((8 * wave + (lane >> 3)) * ldx + piece) * 2;
  const int wstep = 8 * NW * ldw * 2, xstep = 8 * NW * ldx * 2;
  // What is loaded runs AHEAD steps before what is multiplied, into the workgroup's next tile, and past its last one into nothing (a
  // buffer of no bytes): every tile has more steps than that.  Every die starts at a place of its own along K.
  const int stride = gridDim.x / 8 + (die < static_cast<int>(gridDim.x % 8));
  int at_tile = blockIdx.x / 8;
  if (at_tile >= mine) return;
  Tile t = tile_of(at_tile);
  Rows wr = w_of(t), xr = x_of(t);
  constexpr int STEP = BK * 2;
  int wk = die * t.steps / 8 * STEP, xk = wk, around = t.steps * STEP;
  auto load_w = [&](int buf, int sub, int l) {
    load_to_lds(wr.at, wr.bytes, lds + buf + sub * WS + (l * NW + wave) * 1024, wvo, l * wstep + sub * 128 + wk);
  };
  auto load_x = [&](int buf, int sub, int l) {
    load_to_lds(xr.at, xr.bytes, lds + SW * WB + buf + sub * XS + (l * NW + wave) * 1024, xvo, l * xstep + sub * 128 + xk);
  };
  auto onward = [&](int& k) { k = k + STEP == around ? 0 : k + STEP; };
  const int wn = wave % WN, wm = wave / WN, row = lane % 16, quarter = lane / 16;
  const int at = row * 128 + ((quarter ^ (row >> 1)) * 16);
  const unsigned char* const wl = lds + wn * FN * 2048;
  const unsigned char* const xl = lds + SW * WB + wm * FM * 2048;
  f32x4_t acc[FN][FM] = {};
  bf16x8_t a[2][FN], b[2][FM];
  auto read_one = [&](int wat, int xat, int sub, int to, int f) {
    if (f < FN)
      a[to][f] = *reinterpret_cast<const bf16x8_t*>(wl + sub * WS + f * 2048 + wat);
    else
      b[to][f - FN] = *reinterpret_cast<const bf16x8_t*>(xl + sub * XS + (f - FN) * 2048 + xat);
  };
  // 32 along K: the products from operands p % 2, and spread evenly between them the reads of the next 32's operands, loads, and what
  // `beside` says (one wave a SIMD issues an instruction every four clocks, a product takes sixteen: what stands together leaves the
  // matrix cores idle)
  auto part = [&](int p, int wat, int xat, int to, auto beside) {
    const int use = p % 2, sub = (p + 1) / 2 % SUB, n = p == 2 * SUB - 1 ? LF * SUB : LT * SUB, parts = p == 2 * SUB - 1 ? 1 : 2 * SUB - 1, c = p == 2 * SUB - 1 ? 0 : p;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = q / FM, j = i % 2 ? FM - 1 - q % FM : q % FM;  // neighbours share an operand
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[use][i], b[use][j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int f = (q * R + Q - 1) / Q; f < ((q + 1) * R + Q - 1) / Q; ++f) read_one(wat, xat, sub, use ^ 1, f);
#pragma unroll
      for (int l = (c * Q + q) * n / (parts * Q); l < (c * Q + q + 1) * n / (parts * Q); ++l) {
        if ((p == 2 * SUB - 1) == X_FIRST)
          load_x(to, l / LX, l % LX);
        else
          load_w(to, l / LW, l % LW);
      }
      beside(q);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto meet = [] {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
#pragma unroll
  for (int s = 0; s < AHEAD; ++s) {
#pragma unroll
    for (int sub = 0; sub < SUB; ++sub) {
#pragma unroll
      for (int l = 0; l < LX; ++l) load_x(s * XB, sub, l);
#pragma unroll
      for (int l = 0; l < LW; ++l) load_w(s * WB, sub, l);
    }
    onward(wk);
    onward(xk);
  }
  wait_for<(AHEAD - 1) * L * SUB, 15>();
  meet();
#pragma unroll
  for (int f = 0; f < R; ++f) read_one(at, at, 0, 0, f);
  int wcur = 0, xcur = 0;
  int late = AHEAD * (X_FIRST ? WB : XB);  // the buffer that the last step left of the operand loaded later
  int wat = at, xat = at;
  for (;;) {
    at_tile += stride;
    const bool more = at_tile < mine;
    const Tile next = tile_of(more ? at_tile : 0);
    Rows wnext = w_of(next), xnext = x_of(next);
    if (!more) wnext.bytes = xnext.bytes = 0;
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    int s = t.steps - AHEAD;
    for (bool last = false;; last = true) {
      do {
        int wnxt = 0, xnxt = 0;
#pragma unroll
        for (int p = 0; p < 2 * SUB - 1; ++p)
          part(p, wat ^ (p % 2 ? 0 : 64), xat ^ (p % 2 ? 0 : 64), late, [&](int q) {
            if (p == 0 && q == 1) wnxt = wcur + WB == SW * WB ? 0 : wcur + WB;
            if (p == 0 && q == 2) xnxt = xcur + XB == SX * XB ? 0 : xcur + XB;
            if (p == 0 && q == 1) asm volatile("" : "+s"(wnxt));
            if (p == 0 && q == 2) asm volatile("" : "+s"(xnxt));
          });
        onward(X_FIRST ? wk : xk);
        // the next step has landed, and every wave holds the last operands of this one, whose buffers are loaded into from here on
        wait_for<((AHEAD - 2) * L + LT) * SUB, 0>();
        meet();
        wat = wnxt + at;
        xat = xnxt + at;
        part(2 * SUB - 1, wat, xat, X_FIRST ? xcur : wcur, [](int) {});
        onward(X_FIRST ? xk : wk);
        late = X_FIRST ? wcur : xcur;
        wcur = wnxt;
        xcur = xnxt;
      } while (--s > 0);
      if (last) break;
      wr = wnext;
      xr = xnext;
      around = next.steps * STEP;
      wk = xk = die * next.steps / 8 * STEP;
      s = AHEAD;
    }
  // lane l holds columns 8 (l / 16) .. + 3 of 32 in one product's registers and the four after them in the next one's
  const int m = t.m0 + wm * FM * 16 + row, nw = t.n0 + wn * FN * 16;
#pragma unroll
  for (int j = 0; j < FM; ++j) {
    const int mj = m + 16 * j;
    if constexpr (OUT == OUT_GATED) {
      bf16_t* const y = static_cast<bf16_t*>(yv) + static_cast<size_t>(mj) * ldy;
#pragma unroll
      for (int i = 0; i < FN; i += 4) {
        float o[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          // eight columns of gate lie in even rows of 16 lanes, their eight of up in the odd row after
          const auto s2 = __builtin_amdgcn_permlane16_swap(__float_as_uint(as_output(acc[i + e / 4][j][e % 4], 1)),
                                                           __float_as_uint(as_output(acc[i + 2 + e / 4][j][e % 4], 1)), false, false);
          o[e] = gated(__uint_as_float(s2[0]), __uint_as_float(s2[1]), kind, p0, p1);
        }
        const int n = nw + 16 * i + 32 * (quarter & 1) + 16 * (quarter >> 1);  // of the packed matrix
        if (mj < M && n < N)
          *reinterpret_cast<u32x4_t*>(y + n / 2) = u32x4_t{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]), pack_bf16x2(o[4], o[5]), pack_bf16x2(o[6], o[7])};
      }
    } else if constexpr (OUT == OUT_BF16 || OUT == OUT_ACT) {
      bf16_t* const y = static_cast<bf16_t*>(yv) + static_cast<size_t>(mj) * ldy;
#pragma unroll
      for (int i = 0; i < FN; i += 2) {
        const int n = nw + 16 * i + 8 * quarter;
        f32x4_t u = acc[i][j], v = acc[i + 1][j];
        if constexpr (OUT == OUT_ACT) {
#pragma unroll
          for (int e = 0; e < 4; ++e) u[e] = act_plain(as_output(u[e], 1), kind), v[e] = act_plain(as_output(v[e], 1), kind);
        }
        if (mj < M && n < N)
          *reinterpret_cast<u32x4_t*>(y + n) = u32x4_t{pack_bf16x2(u[0], u[1]), pack_bf16x2(u[2], u[3]), pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
    } else {
      float* const y = static_cast<float*>(yv) + (static_cast<size_t>(t.slice) * M + mj) * ldy;
#pragma unroll
      for (int i = 0; i < FN; i += 2) {
        f32x4_t u, v;  // columns 4 (l / 16) .. + 3 of the 32, and those 16 further: a row's 64 bytes in one store
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const auto s2 = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i][j][e]), __float_as_uint(acc[i + 1][j][e]), false, false);
          const auto s4 = __builtin_amdgcn_permlane32_swap(s2[0], s2[1], false, false);
          u[e] = __uint_as_float(s4[0]);
          v[e] = __uint_as_float(s4[1]);
        }
        const int n = nw + 16 * i + 4 * quarter;
        if (mj < M && n < N) *reinterpret_cast<f32x4_t*>(y + n) = u;
        if (mj < M && n + 16 < N) *reinterpret_cast<f32x4_t*>(y + n + 16) = v;
      }
    }
  }
    if (!more) break;
    t = next;
  }
  wait_for<0, 15>();  // no load may still be on its way into LDS
}

// Columns and rows of a tile, workgroups a compute unit holds, 64s of K a step, steps under way; and what a product takes, in us: `once`, and
// for every time the compute units are filled `each` and, per 64 of K, `step` (`full` more where every compute unit is at work), and
// `out` a million bytes written.  Least squares over some 7,000 products timed back to back (72 to 8,192 rows, 512 to 28,672 columns, K 768 to
// 16,384, one to four slices; 7 to 15 % off on average), only to choose among the forms.
struct Form {
  int bn, bm, fit, sub, ahead;
  float once, each, step, full, out;
};
constexpr Form FORMS[] = {{256, 256, 1, 1, 2, 6.9f, 2.4f, 0.97f, 0.21f, 0.15f},
                          {192, 256, 1, 1, 2, 6.1f, -0.4f, 1.03f, 0.05f, 0.21f},
                          {256, 128, 1, 1, 3, 7.0f, -1.7f, 0.72f, 0.02f, 0.25f},
                          {128, 128, 1, 2, 2, 5.7f, -2.4f, 0.45f, 0.01f, 0.38f},
                          {128, 64, 2, 1, 3, 3.9f, -2.2f, 0.34f, 0.31f, 0.44f}};
constexpr int N_FORMS = sizeof(FORMS) / sizeof(FORMS[0]);
constexpr int UNITS = 256;  // compute units

bool fits(const Form& f, int K, int slices) {
  const int steps = K / (64 * f.sub);
  return K % (64 * f.sub) == 0 && steps - (slices - 1) * ((steps + slices - 1) / slices) > f.ahead;
}

struct Choice {
  int form = -1, slices = 1, rounds = 1;
  float us = 1e30f;
};
// The cheapest form with `from` to `to` slices of K.
Choice cheapest(int M, int N, int K, bool gated, int from, int to) {
  Choice best;
  for (int i = 0; i < N_FORMS; ++i) {
    const Form& f = FORMS[i];
    if (gated && i == 1) continue;
    for (int slices = from; slices <= to; slices *= 2) {
      if (!fits(f, K, slices)) continue;
      const long long tiles = static_cast<long long>((N + f.bn - 1) / f.bn) * ((M + f.bm - 1) / f.bm) * slices;
      const int room = UNITS * f.fit, rounds = static_cast<int>((tiles + room - 1) / room);
      const float steps = static_cast<float>((K / 64 + slices - 1) / slices), fill = static_cast<float>(tiles) / room / rounds;
      const float megabytes = static_cast<float>(M) * N * (slices > 1 ? 4 * slices : 2) * 1e-6f;
      // (the consumer of slices reads them all, where it would read bfloat16)
      const float us = f.once + rounds * (f.each + steps * (f.step + f.full * fill)) + megabytes * f.out +
                       (slices > 1 ? static_cast<float>(M) * N * (4 * slices - 2) / 4.5e6f : 0.f);
      if (us < best.us) best = {i, slices, rounds, us};
    }
  }
  return best;
}

int rounds_of(int M, int N, int bn, int bm) {
  return static_cast<int>((static_cast<long long>((N + bn - 1) / bn) * ((M + bm - 1) / bm) + UNITS - 1) / UNITS);
}
// The part of the compute units' rounds that has a tile.
float filled(const Choice& c, int M, int N) {
  const Form& f = FORMS[c.form];
  return static_cast<float>((N + f.bn - 1) / f.bn) * ((M + f.bm - 1) / f.bm) * c.slices / (c.rounds * UNITS * f.fit);
}

// Whether a product with a pass over it saved is faster here than the product in slices or in the library and the pass.  What is saved grows with
// y, what is lost with K: the fused product cannot be cut, so that few tiles leave compute units idle for all of K, and the library's
// product alone is up to 6 % ahead.  Short K always pays (few rows' slices lie closer: 768, else 1,024).  Beyond, small tiles only where they fill
// half of the units (128 x 128) or a fifth and K is up to 2,048 (128 x 64); large ones where their rounds are full enough for their K.  us, without
// / with the pairs here: 105 rows, 2,048 x 4,096 19 / 21, 107 rows, 2,048 x 8,192 24 / 42, 103 rows, 16,384 x 2,048 24 / 21; in tiles of 128 x 128 106
// rows, 14,336 x 8,192 64 / 72; of 256 x 128 in three rounds 2,366 rows, 8,192 x 4,096 146 / 160, in one 1,005 rows 72 / 63.  Of 9,288 products with
// pairs (65 to 4,096 rows, 1,024 to 32,768 columns, K 512 to 28,672) that a rule of the used part alone took 2,338 were more than 6 % slower than without;
// this one takes 5,883, of which 162 are, in 0.82 of the time.  Of 4,870 with an activation it was 635, and is 45 of 3,488, in 0.83.
bool pass_pays(const Choice& c, int M, int N, int K, bool act) {
  if (K <= (act ? 1024 : 768)) return true;
  const Form& f = FORMS[c.form];
  const float fill = filled(c, M, N);
  if (c.form == 4) return K <= 2048 && c.rounds == 1 && fill >= 0.2f;
  if (c.form == 3) return c.rounds == 1 ? fill > (act && K > 4096 ? 0.6f : 0.5f) : c.rounds > 3 && K <= 2048;
  // (the library's tiles of 256 x 192 in no more rounds than ours of 256 x 256: a quarter less of everything)
  if (c.form == 0 && std::min(rounds_of(M, N, 256, 192), rounds_of(M, N, 192, 256)) <= c.rounds) return false;
  if (K <= 2048) return true;
  if (c.form == 2) return c.rounds <= 2 ? fill >= (act ? 0.8f : K <= 4096 ? 0.f : 0.75f) : c.rounds > 3 && fill >= 0.9f;
  if (c.form == 1) return c.rounds > 2 || (K < 4096 && static_cast<float>(M) * N / (c.rounds * UNITS * f.bn * f.bm) >= 0.8f);
  return c.rounds > 1 || (K <= 4096 && fill >= 0.8f);
}

// The form and the slices of K for a product (form * 256 + slices), or -1 where the vendor library, or the kernels for fewer rows, do better.
int plan(int M, int N, int K, bool partial, bool gated, bool act) {
  if (M <= (act ? 128 : 64) || K % 64 || N % (gated ? 16 : 8)) return -1;
  const Choice whole = cheapest(M, N, K, gated, 1, 1);
  if (partial) {
    // Up to 1,100 rows: beyond, whole tiles fill the compute units (us, library / whole / two slices: 1,110 x 3,072 x 8,192 82 / 76 / 72, but 1,300 89 /
    // - / 112; 1,110 x 4,096 x 8,192 102 / - / 122, 4,096 x 4,096 62 / - / 75).  Up to 5,120 columns, and up to 8,192 where K is twice as long, which
    // the library has no tiles for (library / gemm_tile / here: 8,192 x 28,672, 129 rows 308 / 197 / 137, 256 323 / 204 / 162; 7,168 x 20,480, 256 rows
    // 240 / 139 / 112; 6,144 x 16,384, 129 rows 151 / 102 / 67).
    // Up to 128 rows the few-row kernel's slices are as fast unless K is short or long (its / here: 103 rows, 512 x 768 9.7 / 6.9, 1,024 x 3,072 11.0 / 13.3, 2,560 x
    // 1,024 11.0 / 11.9); tiles of 128 x 64 that fill more than half of the units only where K is long (536 rows, 3,584 x 5,120 44 / 52, 660 rows, 1,536 x
    // 3,072 23 / 25).
    const Choice cut = cheapest(M, N, K, gated, 2, 4);
    if (cut.form != 1 && cut.us < whole.us && M <= 1100 && (N >= 1024 || M <= 512) && !(cut.form == 4 && filled(cut, M, N) > 0.5f && K < 8192) &&
        (N <= 5120 ? K >= (M <= 128 && N < 1280 ? 4096 : 3072) || (M <= 128 ? K <= (N <= 1536 ? 1024 : 768) : M <= 256 && N <= 2560 && (N > 640 || K >= 1024))
                   : N <= 8192 && K >= 2 * N && M > 128 && M <= 256))
      return cut.form * 256 + cut.slices;
  }
  if (whole.form < 0) return -1;
  const Form& f = FORMS[whole.form];
  const int best = whole.form, best_rounds = whole.rounds;
  // the part of the compute units' time that goes into y and not into tiles that hang over or units without one
  const float used = static_cast<float>(M) * N / (static_cast<float>(best_rounds) * UNITS * f.fit * f.bn * f.bm);
  bool ours;
  // With an activation of every element in the product's end, library (or slices) and pass / here, us: 8,192 x 2,048, 129 rows 22.5 / 13.4, 512
  // 24.6 / 21.2, 2,048 67.8 / 58.0, 4,096 126 / 111; 2,048 x 1,024 16.3 / 8.8, 22.2 / 9.2, 19.2 / 12.7, 27.7 / 22.8; 16,384 x 4,096 35.2 / 31.1,
  // 63.0 / 58.3, 209 / 195, 415 / 399.
  if (act)
    ours = N >= 2048 && K <= N && (used >= 0.66f || best != 0 || K <= 2048) && pass_pays(whole, M, N, K, true);
  // Pairs: not where the library's product of the same tiles of 256 x 256 gains more than its pass for the pairs costs: long and wide matrices (us, library
  // and pass / here: 28,672 x 4,096, 1,300 rows 275 / 289, 2,048 378 / 396, 57,344 x 8,192 1,032 / 1,091, 1,316 / 1,382; from 2,560 rows on
  // 581 / 574, 982 / 871; 24,576 x 4,096 304.5 / 303.9 at 2,048; of fewer rows 512 102 / 103, 900 184 / 189, 57,344 x 8,192 397 / 391, 784 / 719).
  else if (gated)
    ours = N >= 2048 && !(best == 0 && N > 24576 && K >= 4096 && M <= 2560) && pass_pays(whole, M, N, K, false) &&
           (M <= 128 || used >= (M <= 256 ? 0.6f : M <= 720 ? 0.76f : 0.65f));
  // Whole tiles where one time round is nearly full, and widths of no whole number of the library's tiles, of a long K only in the smaller tiles and where half
  // of the time is y's (us, library / here: 1,360 x 2,048, 1,055 rows 21 / 20; 1,360 x 8,192, 1,154 rows, .37 of the time 50 / 62, 1,877, .61, 69 / 62; 1,360 x
  // 5,120, 1,418 rows, .46, 41 / 48; in tiles of 256 x 128 3,195 rows, 1,360 x 8,192 77 / 85).  Tiles of 128 x 128 wait for memory the longer K is (1,148 x 2,560 x
  // 14,336, .70 109 / 126, 1,343 rows, .82, 132 / 120; 439 x 8,192 x 14,336, .86, 150 / 130; 373 x 8,192 x 6,144, .73 52 / 58), and those of 256 x 128 beyond
  // 16,384 (893 x 8,192 x 28,672 358 / 406).  The same whether slices would do or not: 1,649 x 4,096 x 8,192 125 / 120, 1,187 x 3,072 x 11,008 106 / 98.
  else
    ours = (best_rounds == 1 && ((best == 2 && used >= 0.8f && K <= 16384) || (best == 3 && used >= (K > 4096 ? 0.75f : 0.7f)))) ||
           (N % 128 && N <= 8192 && M > 720 && (K <= 2048 || (used >= 0.5f && best != 2)));
  return ours ? best * 256 + 1 : -1;
}

template <int OUT>
int launch(int form, const bf16_t* x, const bf16_t* w, void* y, int M, int N, int K, int ldx, int ldw, int ldy, int slices, int kind, float p0,
           float p1, hipStream_t stream) {
  const Form f = FORMS[form];
  const int total = ((N + f.bn - 1) / f.bn) * ((M + f.bm - 1) / f.bm) * slices;
  const int room = UNITS * f.fit, rounds = (total + room - 1) / room, grid = std::min(room, ((total + rounds - 1) / rounds + 7) / 8 * 8);
  switch (form) {
    case 0:
      if constexpr (OUT != OUT_GATED && OUT != OUT_ACT)  // (whose ends need the registers of four waves more)
        gemm_block_kernel<256, 256, 2, 2, 1, 2, true, OUT><<<grid, 256, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy, slices, kind, p0, p1);
      else
        gemm_block_kernel<256, 256, 2, 4, 1, 2, true, OUT><<<grid, 512, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy, slices, kind, p0, p1);
      break;
    case 1:
      if constexpr (OUT != OUT_GATED) gemm_block_kernel<192, 256, 2, 4, 1, 2, true, OUT><<<grid, 512, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy, slices, kind, p0, p1);
      break;
    case 2: gemm_block_kernel<256, 128, 2, 4, 1, 3, false, OUT><<<grid, 512, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy, slices, kind, p0, p1); break;
    case 3: gemm_block_kernel<128, 128, 2, 4, 2, 2, true, OUT><<<grid, 512, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy, slices, kind, p0, p1); break;
    default: gemm_block_kernel<128, 64, 2, 2, 1, 3, false, OUT><<<grid, 256, 0, stream>>>(x, w, y, M, N, K, ldx, ldw, ldy, slices, kind, p0, p1); break;
  }
  return yk_check_launch("gemm_block");
}

int g_force_block = -1;

}  // namespace

// The form and slices for a product as form * 256 + slices, -1: not this kernel's.  `partial`: slices may be handed on.
// gated: 1 pairs, 2 an activation of every element.
extern "C" int yk_gemm_block_plan(int M, int N, int K, int partial, int gated) {
  if (g_force_block != -1) return std::max(g_force_block, -1);
  return plan(M, N, K, partial != 0, gated == 1, gated == 2);
}

// For tests and measurements: the plan of every product (form * 256 + slices; -1: the rule; -2: nothing is this kernel's).
extern "C" int yk_gemm_block_force(int plan) {
  YK_REQUIRE(plan >= -2 && (plan < 0 || (plan / 256 < N_FORMS && plan % 256 >= 1)), "gemm_block_force: form * 256 + slices, or -1");
  g_force_block = plan;
  return 0;
}

// y [M, N] = x [M, K] . w [N, K]^T, bfloat16 operands, in the form and slices of `plan`.  out: 0 bfloat16, 1 float32 (`slices` > 1: the unreduced
// slices [slices, M, N] one behind the other, ldy = N), 2 gated pairs of groups of eight columns, bfloat16 [M, N / 2] (kind, p0, p1: common.h), 3
// bfloat16 with the activation `kind` (act_plain) of the rounded product.
extern "C" int yk_gemm_block(const void* x, const void* w, void* y, int out, int M, int N, int K, int ldx, int ldw, int ldy, int plan, int kind,
                             float p0, float p1, hipStream_t stream) {
  const int form = plan / 256, slices = plan % 256;
  YK_REQUIRE(M > 0 && N > 0 && K > 0 && K % 64 == 0 && N % 8 == 0, "gemm_block: K is a multiple of 64, N of 8");
  YK_REQUIRE(out >= 0 && out <= 3 && plan >= 0 && form < N_FORMS, "gemm_block: unknown output or form");
  YK_REQUIRE(!(out == OUT_GATED && (N % 16 || form == 1)), "gemm_block: gated pairs are groups of eight columns, and form 1 has none");
  YK_REQUIRE(out != OUT_GATED || (kind >= 0 && kind < YK_GATED_KINDS), "gemm_block: unknown activation");
  YK_REQUIRE(out != OUT_ACT || (kind >= 0 && kind <= 2), "gemm_block: unknown activation");
  YK_REQUIRE(slices >= 1 && (slices == 1 || (out == OUT_F32 && ldy == N)), "gemm_block: slices are float32, one behind the other");
  YK_REQUIRE(fits(FORMS[form], K, slices), "gemm_block: a slice of K is too short");
  YK_REQUIRE(ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0 && ldx < 1 << 21 && ldw < 1 << 21, "gemm_block: rows of x and w");
  YK_REQUIRE(ldy >= (out == OUT_GATED ? N / 2 : N) && ldy % 8 == 0, "gemm_block: rows of y");
  YK_REQUIRE(static_cast<long long>((N + 63) / 64) * ((M + 63) / 64) * slices < 1 << 30, "gemm_block: too many tiles");
  YK_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0,
             "gemm_block: operands must be 16-byte aligned");
  const auto* xb = static_cast<const bf16_t*>(x);
  const auto* wb = static_cast<const bf16_t*>(w);
  if (out == OUT_BF16) return launch<OUT_BF16>(form, xb, wb, y, M, N, K, ldx, ldw, ldy, slices, kind, p0, p1, stream);
  if (out == OUT_ACT) return launch<OUT_ACT>(form, xb, wb, y, M, N, K, ldx, ldw, ldy, slices, kind, p0, p1, stream);
  if (out == OUT_F32) return launch<OUT_F32>(form, xb, wb, y, M, N, K, ldx, ldw, ldy, slices, kind, p0, p1, stream);
  return launch<OUT_GATED>(form, xb, wb, y, M, N, K, ldx, ldw, ldy, slices, kind, p0, p1, stream);
}
