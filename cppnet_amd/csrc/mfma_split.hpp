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
// (needs_fp32 and large below) and that wave's outputs are formed again with
// fp32 MFMAs straight from memory: infinities and NaN (inf = inf + NaN + NaN
// would turn an infinite product into NaN), values whose bf16 rounding
// overflows, and values near the low end of the range.  The matrix cores keep
// subnormal bf16 inputs, products and sums (measured: 2^-70 * 2^-70 and
// 2^-130 * 2^10 come back exact), but the terms themselves lie on a grid of
// 2^-133, so a value below 2^-110 loses its low bits (2^-134 at most) and one
// of 2^-134 or less all of them.  A wave is formed again where some nonzero
// element of its block is below 2^-100 and an output is below 2^-60 or
// another operand value is 2^30 or more: otherwise what is lost,
// 2 * 2^-134 * 2^30 a product, is below 2^-24 of every output for
// contractions up to 2^18 terms.  Outputs that are nonzero and below 2^-84
// are formed again too.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

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

// Two elements adjacent in k, split: w[p] holds term p of both, the lower k
// in the low half.  tiny: running minimum over 2 |x| - 1 of the elements'
// bits, so zeros (2^32 - 1) do not count; below kTinyCode some nonzero element
// was under 2^-100.  It is taken from x itself and not from its first term,
// which is zero for |x| <= 2^-134.
constexpr uint32_t kTinyCode = 2u * (27u << 23);  // 2 * the bits of 2^-100

__device__ __forceinline__ uint32_t pack_bf16(float x, float y) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{x, y}, bf16x2));
}
__device__ __forceinline__ void split_pair(float x, float y, uint32_t (&w)[3], uint32_t& tiny) {
  tiny = min(tiny, min(2u * __float_as_uint(x) - 1u, 2u * __float_as_uint(y) - 1u));
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
  __device__ __forceinline__ static void store(char* lds, int u, const f32x4 (&v)[4], uint32_t& tiny) {
    char* p = lds + (u % 4 >> 1) * HS + (u & 1) * 8;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t lo[3], hi[3];
      if (KC) {
        split_pair(v[j][0], v[j][1], lo, tiny);
        split_pair(v[j][2], v[j][3], hi, tiny);
      } else {
        split_pair(v[0][j], v[1][j], lo, tiny);
        split_pair(v[2][j], v[3][j], hi, tiny);
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

  // Returns whether some staged element of the block was nonzero and below
  // 2^-100; ends with a barrier.
  template <bool EDGE>
  __device__ __forceinline__ static bool loop(const float* A, int64_t lda, const float* B, int64_t ldb, int64_t M,
                                             int64_t N, int64_t m0, int64_t n0, int64_t k_begin, int64_t k_end,
                                             char* lds, bool neg, f32x16 (&acc)[C::WM][C::WN]) {
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
    // load (256 x 256: 2.2 us), two in the short rounds of the smaller tiles
    // (128 x 128: 0.84 -> 0.73 us a round), one where two blocks share a CU
    f32x4 v0[4], v1[4];
    uint32_t tiny = 0xffffffffu;
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
        OA::store(b, ub, v, tiny);
      } else {
        if (EDGE && t == tail) ld.place_tail<!TB>(kof, left, v);
        OB::store(b + OA::BYTES, ub, v, tiny);
      }
    };
    int wm, wn, wk;
    kp::wave_pos<C>(wm, wn, wk);
    const int lane = threadIdx.x & 63, h = lane >> 5, r = lane & 31;
    const int ra = wm * (C::WM * 32) + r, rb = wn * (C::WN * 32) + r;

    constexpr int PF = C::WM * C::WN == 2 || C::WM * C::WN == 4 ? 2 : 1;
    // one round: v holds k-tile t + 1
    auto round = [&](int t, f32x4 (&v)[4]) {
      bf16x8 a[C::WM][3], b[C::WN][3];
      // the fragment reads go first where registers allow: they arrive while
      // the next k-tile is split
      constexpr bool kReadsFirst = C::WM * C::WN == 2 || C::WM * C::WN == 4;
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
    return __syncthreads_or(tiny < kTinyCode);
  }

  // neg (WGK == 1, no place to park): form the negated sum first.
  __device__ __forceinline__ static bool run(const float* A, int64_t lda, const float* B, int64_t ldb, int64_t M,
                                             int64_t N, int64_t m0, int64_t n0, int64_t k_begin, int64_t k_end,
                                             char* lds, const Park& park, bool neg, f32x16 (&acc)[C::WM][C::WN]) {
    const bool inside = m0 + C::BM <= M && n0 + C::BN <= N;
    auto part = [&](int64_t k0, int64_t k1, bool minus) {
      return inside && (k1 - k0) % KT == 0 ? loop<false>(A, lda, B, ldb, M, N, m0, n0, k0, k1, lds, minus, acc)
                                           : loop<true>(A, lda, B, ldb, M, N, m0, n0, k0, k1, lds, minus, acc);
    };
    if constexpr (C::WGK == 2) {
      const bool any = part(k_begin, k_end, false);
      if (threadIdx.x >= NS) negate<C>(acc);
      kp::reduce_wgk<C>(reinterpret_cast<float*>(lds), acc);
      return any;
    }
    const int halves = park.C ? 2 : 1;
    const int64_t mid = park.C ? k_begin + (k_end - k_begin) / (2 * KT) * KT : k_end;
    bool any = false, minus = neg;
    int64_t k0 = k_begin, k1 = mid;
#pragma unroll 1
    for (int half = 0;; ++half) {
      any |= part(k0, k1, minus);
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
      return any;
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
    return any;
  }

  // Whether this wave's outputs have to be formed with fp32 MFMAs: one is not
  // finite (an operand was not, or its bf16 term overflowed), or one is below
  // 2^-60 while some operand element was below 2^-100, or one is nonzero and
  // below 2^-84.
  __device__ __forceinline__ static bool needs_fp32(const f32x16 (&acc)[C::WM][C::WN], bool tiny) {
    float hi = 0.f, lo = INFINITY, lo_nz = INFINITY;
    bool nan = false;
#pragma unroll
    for (int i = 0; i < C::WM; ++i)
#pragma unroll
      for (int j = 0; j < C::WN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const float x = acc[i][j][e];
          nan |= x != x;
          hi = fmaxf(hi, fabsf(x));
          lo = fminf(lo, fabsf(x));
          lo_nz = fminf(lo_nz, x == 0.f ? INFINITY : fabsf(x));
        }
    const bool bad = nan || hi == INFINITY || (tiny && lo < 0x1p-60f) || lo_nz < 0x1p-84f;
    return __any(bad);
  }

  // f(a, b): the wave's operand values at k, k + 1, straight from memory
  // (zeros past the edges), over the whole contraction.
  template <class F>
  __device__ __forceinline__ static void each_k(const float* A, int64_t lda, const float* B, int64_t ldb, int64_t M,
                                             int64_t N, int64_t m0, int64_t n0, int64_t k_begin, int64_t k_end, F&& f) {
    int wm, wn, wk;
    kp::wave_pos<C>(wm, wn, wk);
    const int lane = threadIdx.x & 63, h = lane >> 5, r = lane & 31;
    for (int64_t k = k_begin; k < k_end; k += 2) {
      const int64_t kk = k + h;
      float a[C::WM], b[C::WN];
#pragma unroll
      for (int i = 0; i < C::WM; ++i) {
        const int64_t m = m0 + wm * (C::WM * 32) + 32 * i + r;
        a[i] = m < M && kk < k_end ? A[TA ? kk + lda * m : m + lda * kk] : 0.f;
      }
#pragma unroll
      for (int j = 0; j < C::WN; ++j) {
        const int64_t n = n0 + wn * (C::WN * 32) + 32 * j + r;
        b[j] = n < N && kk < k_end ? B[!TB ? kk + ldb * n : n + ldb * kk] : 0.f;
      }
      f(a, b);
    }
  }

  // Whether this wave's operands hold a value of 2^30 or more: beside what a
  // tiny value lost it can count in an output above 2^-60.
  // Only asked where some element was below 2^-100; its code beside the loop
  // and needs_fp32's test of small outputs cost the others up to 1.7%
  // (1001 x 785 x 515 forward and backward 82.5 -> 83.9 us; 4096^3 nothing).
  __device__ __forceinline__ static bool large(const float* A, int64_t lda, const float* B, int64_t ldb, int64_t M,
                                            int64_t N, int64_t m0, int64_t n0, int64_t k_begin, int64_t k_end) {
    float hi = 0.f;
    each_k(A, lda, B, ldb, M, N, m0, n0, k_begin, k_end, [&](const float (&a)[C::WM], const float (&b)[C::WN]) {
#pragma unroll
      for (int i = 0; i < C::WM; ++i) hi = fmaxf(hi, fabsf(a[i]));
#pragma unroll
      for (int j = 0; j < C::WN; ++j) hi = fmaxf(hi, fabsf(b[j]));
    });
    return __any(hi >= 0x1p30f);
  }

  // The wave's outputs with v_mfma_f32_32x32x2f32: slow, for the rare waves
  // that needs_fp32 or large names.
  __device__ __forceinline__ static void fp32(const float* A, int64_t lda, const float* B, int64_t ldb, int64_t M,
                                           int64_t N, int64_t m0, int64_t n0, int64_t k_begin, int64_t k_end,
                                           f32x16 (&acc)[C::WM][C::WN]) {
    kp::zero_acc<C>(acc);
    each_k(A, lda, B, ldb, M, N, m0, n0, k_begin, k_end, [&](const float (&a)[C::WM], const float (&b)[C::WN]) {
#pragma unroll
      for (int i = 0; i < C::WM; ++i)
#pragma unroll
        for (int j = 0; j < C::WN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    });
  }
};

}  // namespace sp
}  // namespace cnhip
