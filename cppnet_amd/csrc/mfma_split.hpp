// fp32 products on the bf16 matrix cores (v_mfma_f32_32x32x16_bf16, wave64).
//
// The fp32 MFMA runs at 157 TFLOP/s, the bf16 one at 2.5 PFLOP/s (1.82 PFLOP/s
// sustained on random operands, where the card's power limit lowers the
// clock).  Every operand element is split while it is staged into LDS into
// three bf16 terms, x = x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x - x0),
// x2 = bf16(x - x0 - x1) (round to nearest even): 8 + 8 + 8 significand bits
// and the signs of the remainders hold all 24 bits of x.  A product takes the
// six MFMAs
//   a2 b0 + a0 b2 + a1 b1 + a1 b0 + a0 b1 + a0 b0,
// all into one fp32 accumulator; the three terms left out are below 2^-26 of
// a b.  Two properties of the matrix core shape the accumulation (measured
// against float64, 64 Ki outputs, contractions of 128 .. 4096): it cuts the
// low bits of a sum towards minus infinity, so a running sum drifts by
// -2e-7 of the result's size per 4096 k where the fp32 MFMA has no drift;
// and it cuts them for zero products too, where an fp32 product of zero adds
// no rounding, which makes it the worse of the two on ReLU outputs (9.4e-7
// against 8.1e-7 at 4096).  So every contraction runs as two half sums, the
// second over the negated A, and the result is their difference: the drifts
// cancel (2e-9) and the error is 0.81 (ReLU outputs), 0.60 (normal) and 0.32
// (positive) of the fp32 MFMA's.
//
// What bf16 terms cannot hold is caught per wave after the contraction
// (needs_fp32 below) and that wave's outputs are formed again with fp32 MFMAs
// straight from memory: infinities and NaN (inf = inf + NaN + NaN would turn
// an infinite product into NaN), values whose bf16 rounding overflows, and
// values at the low end of the range.  The matrix cores keep subnormal bf16
// inputs, products and sums (measured: 2^-70 * 2^-70 and 2^-130 * 2^10 come
// back exact), but the terms themselves lie on a grid of 2^-133, so a value
// below 2^-110 can lose up to 2^-134.  Where a block's operands hold such a
// value, an output of the block is off by at most K 2^-133 times the largest
// element, and a wave is formed again where that is more than 2^-24 of one of
// its outputs (range, Tile::run).  Both bounds are kept while the operands are
// staged, so nothing is read twice to find them.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "mfma_kpack.hpp"

namespace cnhip {
namespace sp {

using kp::f32x16;
using kp::f32x4;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
using kp::f32x4u;

constexpr int KT = 16;  // k-tile depth: one MFMA step

// Of the elements a thread stages: the smallest nonzero one, as 2 |x| - 1 of
// its bits (so zeros, 2^32 - 1, do not count), and the largest |x|.  Taken
// from x itself: its first term is zero for |x| <= 2^-134.
struct Range {
  uint32_t lo = 0xffffffffu;
  float hi = 0.f;
  __device__ __forceinline__ void add(float x, float y) {
    // one instruction each for both elements (the compiler regroups the minima
    // of several pairs, and quiets the operands of fmaxf first)
    asm("v_min3_u32 %0, %1, %2, %0" : "+v"(lo) : "v"(2u * __float_as_uint(x) - 1u), "v"(2u * __float_as_uint(y) - 1u));
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(hi) : "v"(x), "v"(y));
  }
};
constexpr uint32_t kLossyCode = 2u * (17u << 23);  // 2 * the bits of 2^-110

// Two elements adjacent in k, split: w[p] holds term p of both, the lower k
// in the low half.
__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2));
}
__device__ __forceinline__ void split_pair(float x, float y, uint32_t (&w)[3], Range& range) {
  range.add(x, y);
  w[0] = pack_bf16(x, y);
  x -= __builtin_bit_cast(float, w[0] << 16);
  y -= __builtin_bit_cast(float, w[0] & 0xffff0000u);
  w[1] = pack_bf16(x, y);
  x -= __builtin_bit_cast(float, w[1] << 16);
  y -= __builtin_bit_cast(float, w[1] & 0xffff0000u);
  w[2] = pack_bf16(x, y);
}

// An R x KT operand tile in LDS: three bf16 planes, each two chunks of 8 k,
// a chunk being [R][8] (16 bytes per row), so an MFMA fragment (32 rows, 8 k
// per half-wave) is one ds_read_b128 of 512 contiguous bytes per half-wave.
// Staging moves units of 4 x 4 elements:
//   KC:  X(r, k) = X[k + ld*r], k-contiguous: rows r + j R/4 (j = 0..3), one
//        float4 along k each;
//   !KC: X(r, k) = X[r + ld*k]: rows r .. r+3, float4s along r at 4 k, turned
//        in registers while the terms are packed.
// Either way a row's 4 k leave as one ds_write_b64 per plane; the chunks are
// padded apart so that 16 consecutive lanes (4 k-groups x 4 row groups) hit
// different banks.
template <bool KC, int R>
struct Operand {
  static constexpr int HS = R * 16 + (KC ? 64 : 32);  // bytes from one 8-k chunk to the next
  static constexpr int PLANE = 2 * HS;
  static constexpr int BYTES = 3 * PLANE;
  static constexpr int UNITS = R;  // R * KT / 16

  __device__ __forceinline__ static int row(int u, int j) { return KC ? u / 4 + j * (R / 4) : 4 * (u / 4) + j; }
  __device__ __forceinline__ static int kof(int u) { return 4 * (u % 4); }

  // v: the unit's float4s, KC: v[j] = row j; !KC: v[e] = k e
  __device__ __forceinline__ static void store(char* lds, int u, const f32x4 (&v)[4], Range& range) {
    char* p = lds + (u % 4 >> 1) * HS + (u & 1) * 8;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t lo[3], hi[3];
      if (KC) {
        split_pair(v[j][0], v[j][1], lo, range);
        split_pair(v[j][2], v[j][3], hi, range);
      } else {
        split_pair(v[0][j], v[1][j], lo, range);
        split_pair(v[2][j], v[3][j], hi, range);
      }
#pragma unroll
      for (int t = 0; t < 3; ++t) *reinterpret_cast<u32x2*>(p + t * PLANE + row(u, j) * 16) = u32x2{lo[t], hi[t]};
    }
  }
  __device__ __forceinline__ static bf16x8 frag(const char* lds, int plane, int r, int h) {
    return *reinterpret_cast<const bf16x8*>(lds + plane * PLANE + h * HS + r * 16);
  }
};

// One operand of a block's staging: the unit of this thread, read through a
// wave-uniform base pointer (the tile's first row at the next k-tile) and
// 32-bit element offsets of its four float4s, fixed for the whole
// contraction.  No load leaves the operand (which has >= 4 rows and a
// contraction of >= 4): rows past the last are read from a valid row, their
// products never stored; where a float4 would cross the end of the rows (!KC)
// or of K (KC, last k-tile) it starts earlier and its values move to their
// places before the split (place_rows, place_tail), zeros past the end of K.
struct UnitLoader {
  const float* base;  // X + tile row origin at k_begin; advanced by one k-tile per load
  int64_t ld, ks;     // leading dimension; elements per k-tile step along k
  uint32_t off[4];
  int shift;          // !KC: rows by which the float4s start early (0 .. 3)
  bool edge;          // wave-uniform: some shift of the block is not 0

  template <bool KC, int R>
  __device__ __forceinline__ void init(const float* X, int64_t ld_, int64_t r0, int64_t rows, int64_t k0, int kstep,
                                       int u) {
    using O = Operand<KC, R>;
    ld = ld_;
    ks = KC ? kstep : kstep * ld;
    const int last = (int)(rows - r0 < R ? rows - r0 : R) - 1;  // the operand's last row in this tile
    const int k = O::kof(u);
    shift = 0;
    edge = false;
    if (KC) {
      base = X + ld * r0 + k0;
#pragma unroll
      for (int j = 0; j < 4; ++j) off[j] = (uint32_t)k + (uint32_t)ld * (uint32_t)min(O::row(u, j), last);
    } else {
      edge = (last & 3) != 3;
      const int back = last < 3 ? 3 - last : 0;  // rows before the tile that the last float4 reaches
      base = X + (r0 - back) + ld * k0;
      const int r = O::row(u, 0);
      const int at = r + 3 <= last ? r : last - 3;
      shift = r - at <= 3 ? r - at : 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) off[j] = (uint32_t)(at + back) + (uint32_t)ld * (uint32_t)(k + j);
    }
  }
  __device__ __forceinline__ void load(f32x4 (&v)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = *reinterpret_cast<const f32x4u*>(base + off[j]);
    base += ks;
  }
  // the last k-tile, cut to `left` (1 .. KT-1) values of k; kof: the unit's first
  template <bool KC>
  __device__ __forceinline__ void load_tail(int kof, int left, f32x4 (&v)[4]) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int over = KC ? max(kof + 4 - left, 0) : max(kof + j + 1 - left, 0);
      v[j] = *reinterpret_cast<const f32x4u*>(base + ((int64_t)off[j] - (KC ? over : over * ld)));
    }
  }
  template <bool KC>
  __device__ __forceinline__ static void place_tail(int kof, int left, f32x4 (&v)[4]) {
    if (KC) {
      const int over = max(kof + 4 - left, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4 x = v[j];
        if (over & 1) x = f32x4{x[1], x[2], x[3], 0.f};
        if (over & 2) x = f32x4{x[2], x[3], 0.f, 0.f};
        if (over & ~3) x = f32x4{0.f, 0.f, 0.f, 0.f};
        v[j] = x;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (kof + j >= left) v[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  // !KC: the values of rows r .. r+3 to their places (the last one repeated)
  __device__ __forceinline__ void place_rows(f32x4 (&v)[4]) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 x = v[j];
      if (shift & 1) x = f32x4{x[1], x[2], x[3], x[3]};
      if (shift & 2) x = f32x4{x[2], x[3], x[3], x[3]};
      v[j] = x;
    }
  }
};

// Whether 32-bit offsets reach every element of a tile of `rows` rows.
inline bool offsets_fit(int64_t ld, bool kc, int rows) {
  return ld < (int64_t)((1u << 30) - 64) / (kc ? rows : 16);
}

template <class C, class OA, class OB>
__device__ __forceinline__ void frags(const char* la, bf16x8 (&a)[C::WM][3], bf16x8 (&b)[C::WN][3], int ra, int rb,
                                      int h) {
  const char* lb = la + OA::BYTES;
#pragma unroll
  for (int q = 0; q < 3; ++q) {
#pragma unroll
    for (int i = 0; i < C::WM; ++i) a[i][q] = OA::frag(la, q, ra + 32 * i, h);
#pragma unroll
    for (int j = 0; j < C::WN; ++j) b[j][q] = OB::frag(lb, q, rb + 32 * j, h);
  }
}

template <class C>
__device__ __forceinline__ void mfmas(const bf16x8 (&a)[C::WM][3], const bf16x8 (&b)[C::WN][3],
                                      f32x16 (&acc)[C::WM][C::WN]) {
  auto term = [&](int x, int y) {
#pragma unroll
    for (int i = 0; i < C::WM; ++i)
#pragma unroll
      for (int j = 0; j < C::WN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i][x], b[j][y], acc[i][j], 0, 0, 0);
  };
  term(2, 0);
  term(0, 2);
  term(1, 1);
  term(1, 0);
  term(0, 1);
  term(0, 0);
}

template <class C>
__device__ __forceinline__ void negate(f32x16 (&acc)[C::WM][C::WN]) {
#pragma unroll
  for (int i = 0; i < C::WM; ++i)
#pragma unroll
    for (int j = 0; j < C::WN; ++j) acc[i][j] = -acc[i][j];
}

// Where a 256 x 256 block parks its first half sum: its own part of C.
struct Park {
  float* C;
  int64_t ldc, M, N, m0, n0;
};

// f(reference to 4 accumulators, their row and column in C) for every run of
// 4 rows that this lane holds.
template <class C, class F>
__device__ __forceinline__ void each_run(f32x16 (&acc)[C::WM][C::WN], const Park& p, F&& f) {
  const int lane = threadIdx.x & 63;
  int wm, wn, wk;
  kp::wave_pos<C>(wm, wn, wk);
#pragma unroll
  for (int i = 0; i < C::WM; ++i)
#pragma unroll
    for (int j = 0; j < C::WN; ++j) {
      const int64_t n = p.n0 + wn * (C::WN * 32) + j * 32 + (lane & 31);
#pragma unroll
      for (int q = 0; q < 4; ++q) f(acc[i][j], 4 * q, p.m0 + wm * (C::WM * 32) + i * 32 + 8 * q + 4 * (lane >> 5), n);
    }
}

// The block's k loop over [k_begin, k_end) of a GEMM tile.  The 8 waves form
// two groups of 4, one wave of each group on every SIMD, which alternate: in
// one phase a group stages (splits its next k-tile's float4s into LDS, sends
// the loads of the one after, reads its fragments), in the next it issues
// nothing but its MFMAs, while the other group does the opposite; a barrier
// ends each phase.  So a SIMD's matrix pipe always has one wave feeding it
// (4096^3: 640 us against 700 us for the same tile with both groups in step).
//   WGK == 1: the groups own different columns of the tile, stage the k-tile
//     together and share one double buffer.  The half sums are the first and
//     the second half of k, one loop each; the first waits in the block's own
//     part of C (Park) while the second is formed.  Split-K partials are half
//     sums already: those of odd splits are formed negated (and stored with
//     their own sign).
//   WGK == 2: each group owns the whole tile over every second k-tile, with a
//     double buffer of its own; group 1's is the negated half sum.
template <bool TA, bool TB, class C>
struct Tile {
  using OA = Operand<TA, C::BM>;
  using OB = Operand<!TB, C::BN>;
  static_assert(C::NT == 512 && (C::WGK == 1 || C::WGK == 2), "two groups of 4 waves");
  static constexpr int SB = OA::BYTES + OB::BYTES;          // one k-tile
  static constexpr int NS = C::NT / C::WGK;                 // staging threads per k-tile
  static_assert(OA::UNITS + OB::UNITS <= NS && OA::UNITS % 64 == 0, "one unit per thread, waves of one operand");
  static constexpr int RED = C::WGK == 2 ? 4 * C::WM * C::WN * 16 * 64 * 4 : 0;  // reduce_wgk's bytes
  static constexpr int LDS = 2 * C::WGK * SB > RED ? 2 * C::WGK * SB : RED;

  // Adds to `range` what this thread stages; returns whether some element that
  // the block has staged so far was nonzero and below 2^-110.  Ends with a
  // barrier.
  template <bool EDGE>
  __device__ __forceinline__ static bool loop(const float* A, int64_t lda, const float* B, int64_t ldb, int64_t M,
                                             int64_t N, int64_t m0, int64_t n0, int64_t k_begin, int64_t k_end,
                                             char* lds, bool neg, Range& range, f32x16 (&acc)[C::WM][C::WN]) {
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int grp = wave >> 2;                              // ping-pong group
    const int kg = C::WGK == 2 ? grp : 0;                   // k group
    const int w0 = 64 * wave - kg * NS;                     // first staging thread of this wave
    const int u = (int)threadIdx.x - kg * NS;
    const bool doA = w0 < OA::UNITS, doB = !doA && w0 < OA::UNITS + OB::UNITS;
    constexpr int KSTEP = KT * C::WGK;
    const int64_t kfirst = k_begin + kg * KT;
    UnitLoader ld;
    const int ub = doA ? u : doB ? u - OA::UNITS : 0;
    const int kof = OA::kof(ub);
    if (doA) ld.init<TA, C::BM>(A, lda, m0, M, kfirst, KSTEP, ub);
    else ld.init<!TB, C::BN>(B, ldb, n0, N, kfirst, KSTEP, ub);
    const int total = k_end > k_begin ? (int)((k_end - k_begin + KT - 1) / KT) : 0;
    const int nt = (total + C::WGK - 1) / C::WGK;           // rounds of the block
    const int mine = C::WGK == 2 ? (total - kg + 1) / 2 : total;
    const int left = (int)((k_end - k_begin) % KT);         // k values of a last k-tile cut short, or 0
    const int tail = left != 0 && (total - 1) % C::WGK == kg ? (total - 1) / C::WGK : -1;  // it, if mine

    // k-tiles in flight in registers: one where a round lasts longer than a
    // load (256 x 256: 2.2 us), two in the short rounds of the 128 x 128 tile
    // (0.84 -> 0.73 us a round)
    f32x4 v0[4], v1[4];
    auto load = [&](int t, f32x4 (&v)[4]) {
      if (!doA && !doB) return;
      if (!EDGE || t != tail) ld.load(v);
      else if (doA) ld.load_tail<TA>(kof, left, v);
      else ld.load_tail<!TB>(kof, left, v);
    };
    const uint32_t sign = (C::WGK == 2 ? kg == 1 : neg) ? 0x80000000u : 0u;  // A enters negated
    char* buf = lds + kg * 2 * SB;
    auto store = [&](int t, f32x4 (&v)[4]) {
      if (!doA && !doB) return;
      char* b = buf + (t & 1) * SB;
      if (EDGE && ld.edge) ld.place_rows(v);
      if (doA) {
        if (EDGE && t == tail) ld.place_tail<TA>(kof, left, v);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[j][e] = __uint_as_float(__float_as_uint(v[j][e]) ^ sign);
        OA::store(b, ub, v, range);
      } else {
        if (EDGE && t == tail) ld.place_tail<!TB>(kof, left, v);
        OB::store(b + OA::BYTES, ub, v, range);
      }
    };
    int wm, wn, wk;
    kp::wave_pos<C>(wm, wn, wk);
    const int lane = threadIdx.x & 63, h = lane >> 5, r = lane & 31;
    const int ra = wm * (C::WM * 32) + r, rb = wn * (C::WN * 32) + r;

    constexpr int PF = C::WM * C::WN == 4 ? 2 : 1;
    // one round: v holds k-tile t + 1
    auto round = [&](int t, f32x4 (&v)[4]) {
      bf16x8 a[C::WM][3], b[C::WN][3];
      // the fragment reads go first where registers allow: they arrive while
      // the next k-tile is split
      constexpr bool kReadsFirst = C::WM * C::WN == 4;
      if (kReadsFirst && t < mine) frags<C, OA, OB>(buf + (t & 1) * SB, a, b, ra, rb, h);
      if (t + 1 < mine) {
        store(t + 1, v);
        if (t + 1 + PF < mine) load(t + 1 + PF, v);
      }
      if (!kReadsFirst && t < mine) frags<C, OA, OB>(buf + (t & 1) * SB, a, b, ra, rb, h);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
      if (t < mine) {
        __builtin_amdgcn_s_setprio(1);
        mfmas<C>(a, b, acc);
        __builtin_amdgcn_s_setprio(0);
      }
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
    };
    if (mine > 0) load(0, v0);
    if (PF == 2 && mine > 1) load(1, v1);
    if (mine > 0) store(0, v0);
    if (mine > PF) load(PF, v0);
    __syncthreads();
    if (grp) __syncthreads();
    if constexpr (PF == 1) {
      for (int t = 0; t < nt; ++t) round(t, v0);
    } else {
      int t = 0;
      for (; t + 1 < nt; t += 2) {
        round(t, v1);
        round(t + 1, v0);
      }
      if (t < nt) round(t, v1);
    }
    if (!grp) __syncthreads();
    return __syncthreads_or(range.lo < kLossyCode);
  }

  // The block's largest staged |x|, for every thread; lds is free before and
  // after.
  __device__ __forceinline__ static float largest(char* lds, float hi) {
    uint32_t* m = reinterpret_cast<uint32_t*>(lds);
    if (threadIdx.x == 0) *m = 0;
    __syncthreads();
    atomicMax(m, __float_as_uint(hi));
    __syncthreads();
    hi = __uint_as_float(__builtin_amdgcn_readfirstlane(*m));
    __syncthreads();
    return hi;
  }

  // neg (WGK == 1, no place to park): form the negated sum first.  Returns the
  // smallest output that the terms serve: 2^24 times what the block's operands
  // may have lost in one (0 where they lost nothing).
  __device__ __forceinline__ static float run(const float* A, int64_t lda, const float* B, int64_t ldb, int64_t M,
                                             int64_t N, int64_t m0, int64_t n0, int64_t k_begin, int64_t k_end,
                                             char* lds, const Park& park, bool neg, f32x16 (&acc)[C::WM][C::WN]) {
    const bool inside = m0 + C::BM <= M && n0 + C::BN <= N;
    Range range;
    auto floor = [&](bool lossy) {
      return lossy ? largest(lds, range.hi) * ((float)(k_end - k_begin) * 0x1p-109f) : 0.f;
    };
    auto part = [&](int64_t k0, int64_t k1, bool minus) {
      return inside && (k1 - k0) % KT == 0 ? loop<false>(A, lda, B, ldb, M, N, m0, n0, k0, k1, lds, minus, range, acc)
                                           : loop<true>(A, lda, B, ldb, M, N, m0, n0, k0, k1, lds, minus, range, acc);
    };
    if constexpr (C::WGK == 2) {
      const float least = floor(part(k_begin, k_end, false));
      if (threadIdx.x >= NS) negate<C>(acc);
      kp::reduce_wgk<C>(reinterpret_cast<float*>(lds), acc);
      return least;
    }
    const int halves = park.C ? 2 : 1;
    const int64_t mid = park.C ? k_begin + (k_end - k_begin) / (2 * KT) * KT : k_end;
    bool lossy = false, minus = neg;
    int64_t k0 = k_begin, k1 = mid;
#pragma unroll 1
    for (int half = 0;; ++half) {
      lossy = part(k0, k1, minus);
      if (half + 1 == halves) break;
      minus = true;
      k0 = mid;
      k1 = k_end;
      each_run<C>(acc, park, [&](f32x16& x, int e0, int64_t m, int64_t n) {
        if (n >= park.N) return;
        float* q = park.C + m + park.ldc * n;
        if (m + 3 < park.M) {
          *reinterpret_cast<f32x4u*>(q) = f32x4{x[e0], x[e0 + 1], x[e0 + 2], x[e0 + 3]};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (m + e < park.M) q[e] = x[e0 + e];
        }
      });
      asm volatile("" ::: "memory");
      kp::zero_acc<C>(acc);
    }
    if (!park.C) {
      if (neg) negate<C>(acc);
      return floor(lossy);
    }
    each_run<C>(acc, park, [&](f32x16& x, int e0, int64_t m, int64_t n) {
      if (n >= park.N) return;
      const float* q = park.C + m + park.ldc * n;
      if (m + 3 < park.M) {
        const f32x4 y = *reinterpret_cast<const f32x4u*>(q);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e0 + e] = y[e] - x[e0 + e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (m + e < park.M) x[e0 + e] = q[e] - x[e0 + e];
      }
    });
    return floor(lossy);
  }

  // Whether this wave's outputs have to be formed with fp32 MFMAs: one is not
  // finite (an operand was not, or its bf16 term overflowed), or one is below
  // `least` (run), zeros included.
  __device__ __forceinline__ static bool needs_fp32(const f32x16 (&acc)[C::WM][C::WN], float least) {
    float s[4] = {0.f, 0.f, 0.f, 0.f};  // NaN once a value was not finite
#pragma unroll
    for (int i = 0; i < C::WM; ++i)
#pragma unroll
      for (int j = 0; j < C::WN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e & 3] = fmaf(acc[i][j][e], 0.f, s[e & 3]);
    const float sum = (s[0] + s[1]) + (s[2] + s[3]);
    if (least == 0.f) return __any(sum != sum);
    float lo = INFINITY;
#pragma unroll
    for (int i = 0; i < C::WM; ++i)
#pragma unroll
      for (int j = 0; j < C::WN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) lo = fminf(lo, fabsf(acc[i][j][e]));
    return __any(sum != sum || lo < least);
  }

  // n >= 4 ? X(row, k .. k + 3) : those before k + n, then zeros; p at X(row, k)
  template <bool KC, bool WHOLE>
  __device__ __forceinline__ static f32x4 quad(const float* p, int64_t ld, int64_t n) {
    f32x4 v;
    if (KC && WHOLE) {
      v = *reinterpret_cast<const f32x4u*>(p);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = WHOLE || e < n ? p[KC ? e : ld * e] : 0.f;
    }
    return v;
  }

  // The wave's outputs with v_mfma_f32_32x32x2f32, for the waves that
  // needs_fp32 names; operands straight from memory, 8 k (4 per half-wave) a
  // step and a stage of steps in flight behind the MFMAs, so the wave runs
  // near the fp32 matrix rate.  Rows past the last are read from the last,
  // their products never stored.
  __device__ __forceinline__ static void fp32(const float* A, int64_t lda, const float* B, int64_t ldb, int64_t M,
                                           int64_t N, int64_t m0, int64_t n0, int64_t k_begin, int64_t k_end,
                                           f32x16 (&acc)[C::WM][C::WN]) {
    constexpr int D = C::WM * C::WN >= 8 ? 1 : 2;  // steps of a stage
    struct Stage {
      f32x4 a[D][C::WM], b[D][C::WN];
    };
    int wm, wn, wk;
    kp::wave_pos<C>(wm, wn, wk);
    const int lane = threadIdx.x & 63, h = lane >> 5, r = lane & 31;
    const float *pa[C::WM], *pb[C::WN];
    const int64_t k0 = k_begin + 4 * h;
#pragma unroll
    for (int i = 0; i < C::WM; ++i) {
      const int64_t m = min(m0 + wm * (C::WM * 32) + 32 * i + r, M - 1);
      pa[i] = A + (TA ? k0 + lda * m : m + lda * k0);
    }
#pragma unroll
    for (int j = 0; j < C::WN; ++j) {
      const int64_t n = min(n0 + wn * (C::WN * 32) + 32 * j + r, N - 1);
      pb[j] = B + (!TB ? k0 + ldb * n : n + ldb * k0);
    }
    const int64_t sa = TA ? 8 : 8 * lda, sb = !TB ? 8 : 8 * ldb;
    auto step = [&](f32x4 (&a)[C::WM], f32x4 (&b)[C::WN], auto whole, int64_t left) {
#pragma unroll
      for (int i = 0; i < C::WM; ++i) {
        a[i] = quad<TA, decltype(whole)::value>(pa[i], lda, left);
        pa[i] += sa;
      }
#pragma unroll
      for (int j = 0; j < C::WN; ++j) {
        b[j] = quad<!TB, decltype(whole)::value>(pb[j], ldb, left);
        pb[j] += sb;
      }
    };
    auto load = [&](Stage& s) {
#pragma unroll
      for (int d = 0; d < D; ++d) step(s.a[d], s.b[d], std::true_type{}, 4);
    };
    auto multiply = [&](const f32x4 (&a)[C::WM], const f32x4 (&b)[C::WN]) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < C::WM; ++i)
#pragma unroll
          for (int j = 0; j < C::WN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
    };
    auto use = [&](const Stage& s) {
#pragma unroll
      for (int d = 0; d < D; ++d) multiply(s.a[d], s.b[d]);
    };
    kp::zero_acc<C>(acc);
    const int64_t stages = (k_end - k_begin) / (8 * D);
    Stage s0, s1;
    if (stages > 0) load(s0);
    int64_t t = 0;
#pragma unroll 1
    for (; t + 1 < stages; t += 2) {
      load(s1);
      use(s0);
      if (t + 2 < stages) load(s0);
      use(s1);
    }
    if (t < stages) use(s0);
#pragma unroll 1
    for (int64_t k = k0 + stages * (8 * D); k - 4 * h < k_end; k += 8) {
      f32x4 a[C::WM], b[C::WN];
      step(a, b, std::false_type{}, k_end - k);
      multiply(a, b);
    }
  }
};

}  // namespace sp
}  // namespace cnhip
