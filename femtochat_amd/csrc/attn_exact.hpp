// Building blocks of the exact-mode (fp32) kernels on gfx950.
//
// A float32 value is the sum of three bf16 values, x = h + m + l (8 + 8 + 8
// significant bits, each the rounded rest of the one before), so a float32
// product is six bf16 products with exact terms and fp32 accumulation:
//   x y ~ hh' + hm' + mh' + hl' + mm' + lh',
// the terms left out (m l' and l m' above all) being at most 2^-24 of |x y|,
// 2^-27.5 in the root mean square.  v_mfma_f32_32x32x16_bf16
// does 16 k values in half the time v_mfma_f32_32x32x2_f32 takes for 2, so the
// six together run at up to 2.7 times the fp32 rate, and round the running sum
// 48 times per 128 k values instead of 64: the 2-norm error against float64 of
// an 8 x 2048, H6, D128 causal step is 3.7e-7 (O), 5.2e-7 (dQ), 8.8e-7 (dK) and
// 8.6e-7 (dV), with fp32 MFMA 3.7-4.4e-7, 6.2e-7, 1.15e-6 and 1.15e-6.
//
// Every operand is multiplied by kSplitScale before it is split (and the
// results by its inverse powers, both exact): the bf16 spacing at 0 is 2^-133,
// the float32 spacing 2^-149, so the scaled parts hold every bit of every value
// down to subnormal ones (the matrix cores take subnormal bf16 as they are: at
// dS of 2^-120 the unscaled parts gave the error of gradual underflow).
// At the other end, a scaled value at or beyond 2^127 (an input beyond 2^111,
// an infinity or a NaN) has parts that are infinite or NaN, and so has any sum
// of products that leaves the float32 range with the scale on it (S and dP
// beyond 2^96, dQ, dK beyond 2^80): these reach the accumulators, and rows
// (in dK/dV a workgroup's) that end with one that is not finite are computed
// again with fp32 MFMA straight from global memory, unscaled, which makes them
// take four times as long.  Only a score of -inf would go unseen, as a
// probability of 0: a row whose scores are all -inf, or whose log-sum-exp is
// below -2^80, is computed again too.
#pragma once

#include "attn_fast.hpp"

namespace fc {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr float kSplitScale = 0x1p16f;         // of every operand
constexpr float kSplitScale2 = 0x1p32f;        // of a product of two
constexpr float kSplitInv = 0x1p-16f, kSplitInv2 = 0x1p-32f, kSplitInv3 = 0x1p-48f;
constexpr float kSplitLse = -0x1p80f;          // a log-sum-exp below it may go with scores of -inf

// Eight consecutive k values of one operand row in three bf16 parts.
struct Split8 {
  bf16x8 part[3];
};

__device__ inline uint32_t round2(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

__device__ inline Split8 split8(const float (&x)[8]) {
  uint32_t w[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      w[p][i] = round2(a, b);
      if (p < 2) {
        a -= __uint_as_float(w[p][i] << 16);
        b -= __uint_as_float(w[p][i] & 0xffff0000u);
      }
    }
  }
  Split8 s;
#pragma unroll
  for (int p = 0; p < 3; ++p) s.part[p] = __builtin_bit_cast(bf16x8, make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]));
  return s;
}

// Elements [8 H, 8 H + 8) of an accumulator.
template <int H>
__device__ inline Split8 split_acc(const f32x16& c) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = c[8 * H + e];
  return split8(x);
}

// The first N elements of an accumulator (8: its rows 0 .. 15) are finite.
template <int N = 16>
__device__ inline bool all_finite(const f32x16& c) {
  float m = __builtin_fabsf(c[0]);
#pragma unroll
  for (int r = 1; r < N; ++r) m = __builtin_elementwise_maximum(m, __builtin_fabsf(c[r]));  // propagates NaN
  return m < INFINITY;
}
// The same of D rows in blocks of 32.  (The last block's rows past the head dim
// come from LDS that nothing wrote.)
template <int D>
__device__ inline bool all_finite(const f32x16 (&c)[(D + 31) / 32]) {
  bool finite = true;
#pragma unroll
  for (int db = 0; db < D / 32; ++db) finite &= all_finite(c[db]);
  if (D % 32 != 0) finite &= all_finite<8>(c[(D + 31) / 32 - 1]);
  return finite;
}

// c += a b: the six products, the smallest first.
__device__ inline f32x16 mma_split(const Split8& a, const Split8& b, f32x16 c) {
  c = Mma<bf16>::mma(a.part[2], b.part[0], c);
  c = Mma<bf16>::mma(a.part[0], b.part[2], c);
  c = Mma<bf16>::mma(a.part[1], b.part[1], c);
  c = Mma<bf16>::mma(a.part[1], b.part[0], c);
  c = Mma<bf16>::mma(a.part[0], b.part[1], c);
  return Mma<bf16>::mma(a.part[0], b.part[0], c);
}

// Two sums at once, their products alternating: a product that adds to the
// result of the one before it starts 12 cycles late, which only a second wave on
// the SIMD would fill.
__device__ inline void mma_split_pair(const Split8& a0, const Split8& b0, f32x16& c0, const Split8& a1, const Split8& b1,
                                      f32x16& c1) {
  constexpr int kA[6] = {2, 0, 1, 1, 0, 0}, kB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    c0 = Mma<bf16>::mma(a0.part[kA[i]], b0.part[kB[i]], c0);
    c1 = Mma<bf16>::mma(a1.part[kA[i]], b1.part[kB[i]], c1);
  }
}

// A tile of 32 token rows x D in LDS: three swizzled bf16 tiles, one per part.
template <int D>
struct SplitTile {
  static constexpr int kW = tile_width(D);  // values past D are never written: rows they reach mean nothing
  using Tile = SwzTile<kW>;
  static constexpr int kPlane = 32 * Tile::kRowBytes;
  static constexpr int kBytes = 3 * kPlane;
};

// Natural fragment (chunk c, row l32) and transposed fragment (16-row chunk
// kc, column block db) of all three parts.
template <int D>
__device__ inline Split8 split_nat(const char* tile, const FragOffsets<tile_width(D)>& fo, int c) {
  Split8 s;
#pragma unroll
  for (int p = 0; p < 3; ++p) s.part[p] = as_bf16x8(lds_load16(tile + p * SplitTile<D>::kPlane, fo.nat(c)));
  return s;
}
template <int D>
__device__ inline Split8 split_tr(const char* tile, const FragOffsets<tile_width(D)>& fo, int kc, int db) {
  Split8 s;
#pragma unroll
  for (int p = 0; p < 3; ++p)
    s.part[p] = lds_tr_frag(tile + p * SplitTile<D>::kPlane + 16 * kc * 2 * SplitTile<D>::kW, fo.tr(0, db), fo.tr(1, db));
  return s;
}

// Loads 32 rows x D of float32 (two 16-byte loads per 8-value unit) and
// writes them to LDS, scaled, in parts.  Rows at or beyond T read row T - 1: what they
// give is masked or multiplied by zero.
template <int D>
struct SplitStage {
  static constexpr int kUPR = D / 8, kUnits = 32 * kUPR;
  static constexpr int kPer = (kUnits + kThreads - 1) / kThreads;
  f32x4 v[kPer][2];

  __device__ inline void load(const float* base, int64_t pitch, int row0, int T, int tid) {
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int unit = min(tid + i * kThreads, kUnits - 1);
      const float* p = base + (int64_t)min(row0 + unit / kUPR, T - 1) * pitch + 8 * (unit % kUPR);
      v[i][0] = *reinterpret_cast<const f32x4*>(p);
      v[i][1] = *reinterpret_cast<const f32x4*>(p + 4);
    }
  }
  __device__ inline void store_unit(char* tile, int tid, int i) const {
    const int unit = min(tid + i * kThreads, kUnits - 1);  // past the end: the same values to the same place again
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = v[i][e / 4][e % 4] * kSplitScale;
    const Split8 s = split8(x);
    const int at = SplitTile<D>::Tile::offset(unit / kUPR, unit % kUPR);
#pragma unroll
    for (int p = 0; p < 3; ++p) lds_store16(tile + p * SplitTile<D>::kPlane, at, __builtin_bit_cast(uint4, s.part[p]));
  }
  __device__ inline void store(char* tile, int tid) const {
#pragma unroll
    for (int i = 0; i < kPer; ++i) store_unit(tile, tid, i);
  }
};

// One wave's operand rows (row = lane l32) from global memory, scaled, in parts.
template <int D>
__device__ inline void split_rows(const float* row, bool valid, int g, Split8 (&f)[D / 16]) {
#pragma unroll
  for (int c = 0; c < D / 16; ++c) {
    float x[8];
    const f32x4 lo = valid ? *reinterpret_cast<const f32x4*>(row + 16 * c + 8 * g) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const f32x4 hi = valid ? *reinterpret_cast<const f32x4*>(row + 16 * c + 8 * g + 4) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = lo[e] * kSplitScale, x[4 + e] = hi[e] * kSplitScale;
    f[c] = split8(x);
  }
}

// For the recomputation: column d of 16 float32 rows from row0 as a fragment in
// accumulator k order (rows at or beyond T give zero).
template <int D>
__device__ inline void load_rows_f32(const float* base, int64_t pitch, int row0, int T, int d, int g, f32x8& f) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int row = row0 + 8 * (e >> 2) + 4 * g + (e & 3);
    f[e] = row < T ? base[(int64_t)row * pitch + min(d, D - 1)] : 0.0f;
  }
}

}  // namespace fc
