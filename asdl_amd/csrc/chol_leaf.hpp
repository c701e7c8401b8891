// Cholesky factorization + triangular inverse of one diagonal block of at most 128 x 128 by one work group of 16 waves,
// shared by the batched (one size) and the grouped (many sizes) damped inverse.
//
// The block is 8 x 8 tiles of 16 x 16 and lives in the accumulator registers of the waves for the whole factorization.
// With A = U^T U (U = L^T) the augmented matrix [A | I] is eliminated by block rows; for block row k
//   factor   one wave turns the diagonal tile into M_kk = L_kk^-1 in registers (leaf_tile_inverse)
//   panel    row_k <- M_kk row_k: tiles (k, j > k) become U_kj, tiles (k, j < k) row k of the inverse, which is final
//   update   tile(i, j) -= U_ki^T row_k(j) for the rows i > k: j >= i updates A, j <= k the inverse
// so both halves of a row obey one formula, every row is 8 tiles wide (position j < i: inverse, j > i: U), 64 tiles in
// all, and the inverse is complete when the factorization is: there is no second chain for it.  Only the finished row
// (16 x 128) and M_kk pass through the LDS.  A tile in the accumulator layout is the right operand of the next product as
// it is (v_mfma_f32_16x16x4_f32: register r of lane 16 g + c is row 4 g + r, column c; step r of a product contracts the
// rows {4 g + r}), which is why U and not L is kept.
//
// What bounds it: the chain of 8 x (factor -> barrier -> panel -> barrier -> update of the next diagonal tile), about 4 k
// cycles per link; the wave that owns diagonal tile k + 1 updates it first and factors it while the others still
// update.  The fp32 matrix instructions of all 224 tile products fill 7 k cycles of the four SIMDs beside it.
#pragma once
#include "common.hpp"

namespace ak {

constexpr int LEAF = 128;
constexpr int LT = 16;                       // tile
constexpr int LEAF_THREADS = 1024;
constexpr int LEAF_SLOTS = 5;                // tiles a wave holds at most
constexpr int LEAF_ROW_LD = LEAF + 4;        // 4 rows apart: 16 banks apart, so the rows 4 g + r of one step do not collide
constexpr int LEAF_INV_LD = LT + 4;

struct LeafShared {
  float row[LT * LEAF_ROW_LD];
  float inv[LT * LEAF_INV_LD];
  int bad;
};

__device__ __forceinline__ float lane_bcast(float v, int src_lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), src_lane));
}

// v_mfma_f32_16x16x4_f32: lane l feeds A[i = l%16][k = l/16] and B[k = l/16][j = l%16]; accumulator register r of
// lane l is C[i = 4*(l/16) + r][j = l%16].
__device__ __forceinline__ floatx4 mfma16(float a, float b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Lane 16 g + c receives register g of lane 16 q + c: the four registers of row group q, one to each row group (a
// column of the 4 x 4 transposition of registers and 16-lane rows: swap the halves, then the odd with the even rows).
template <int Q>
__device__ __forceinline__ float spread_row_group(const floatx4& v) {
  const auto bits = [](float x) { return __builtin_bit_cast(unsigned, x); };
  const auto s02 = __builtin_amdgcn_permlane32_swap(bits(v[0]), bits(v[2]), false, false);
  const auto s13 = __builtin_amdgcn_permlane32_swap(bits(v[1]), bits(v[3]), false, false);
  const auto t = __builtin_amdgcn_permlane16_swap(s02[Q >> 1], s13[Q >> 1], false, false);
  return __builtin_bit_cast(float, static_cast<unsigned>(t[Q & 1]));
}

// Pivots 4 Q ... 4 Q + 3 of leaf_tile_inverse.
template <int Q>
__device__ __forceinline__ void leaf_tile_step(floatx4& a, floatx4& inv, floatx4& piv, int& bad, int g, int c) {
  // the 4 x 4 block on the diagonal, in every lane: column i of its lower triangle sits in lane (Q, 4 Q + i)
  float d[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r <= i; ++r) d[i][r] = lane_bcast(a[r], 16 * Q + 4 * Q + i);
  float l[4][4], rec[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (!(d[k][k] > 0.f)) {                  // also catches NaN
      if (bad == 0) bad = 4 * Q + k + 1;
      d[k][k] = 1.f;
    }
    float r = __builtin_amdgcn_rcpf(d[k][k]);             // hardware reciprocal, then one Newton step
    r = __builtin_fmaf(__builtin_fmaf(-d[k][k], r, 1.f), r, r);
    rec[k] = r;
#pragma unroll
    for (int i = k + 1; i < 4; ++i) l[i][k] = d[i][k] * r;
#pragma unroll
    for (int i = k + 1; i < 4; ++i)
#pragma unroll
      for (int j = k + 1; j <= i; ++j) d[i][j] -= d[i][k] * l[j][k];
  }
  // x: the inverse of the unit lower triangle l
  const float x10 = -l[1][0], x21 = -l[2][1], x32 = -l[3][2];
  const float x20 = -l[2][0] - l[2][1] * x10, x31 = -l[3][1] - l[3][2] * x21;
  const float x30 = -l[3][0] - l[3][1] * x10 - l[3][2] * x20;
  // rows 4 Q + t of D L^T and of the unit inverse; meaningful in the lanes of row group Q, which hold those rows
  floatx4 z, w;
  z[0] = a[0];                                              w[0] = inv[0];
  z[1] = a[1] + x10 * a[0];                                 w[1] = inv[1] + x10 * inv[0];
  z[2] = a[2] + x21 * a[1] + x20 * a[0];                    w[2] = inv[2] + x21 * inv[1] + x20 * inv[0];
  z[3] = a[3] + x32 * a[2] + x31 * a[1] + x30 * a[0];       w[3] = inv[3] + x32 * inv[2] + x31 * inv[1] + x30 * inv[0];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    inv[r] = g == Q ? w[r] : inv[r];
    piv[r] = g == Q ? d[r][r] : piv[r];
  }
  if constexpr (Q < 3) {
    const float zq = spread_row_group<Q>(z), wq = spread_row_group<Q>(w);     // lane (g, c): row 4 Q + g, column c
    const float r = g < 2 ? (g == 0 ? rec[0] : rec[1]) : (g == 2 ? rec[2] : rec[3]);
    const float lq = c >= 4 * Q + 4 ? -zq * r : 0.f;                           // -L[c][4 Q + g]; finished rows are left alone
    a = mfma16(lq, zq, a);
    inv = mfma16(lq, wq, inv);
  }
}

// a: a symmetric 16 x 16 tile in the accumulator layout (only elements with column >= row are looked at), replaced by
// L^-1 of its Cholesky factor (zeros above the diagonal).  Returns 0 or the 1-based index of the first non-positive
// pivot.  L D L^T by blocks of 4 pivots: the 4 x 4 blocks are factored and inverted by every lane for itself (ten
// lane reads and a chain of four reciprocals; no square root before the end), and the rank-4 updates of the tile and of
// its inverse are one matrix instruction each.
__device__ __forceinline__ int leaf_tile_inverse(floatx4& a, int lane) {
  const int g = lane >> 4, c = lane & 15;
  int bad = 0;
  floatx4 inv, piv = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
  for (int r = 0; r < 4; ++r) inv[r] = 4 * g + r == c ? 1.f : 0.f;
  leaf_tile_step<0>(a, inv, piv, bad, g, c);
  leaf_tile_step<1>(a, inv, piv, bad, g, c);
  leaf_tile_step<2>(a, inv, piv, bad, g, c);
  leaf_tile_step<3>(a, inv, piv, bad, g, c);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float s = __builtin_amdgcn_rsqf(piv[r]);
    s = __builtin_fmaf(0.5f * s, __builtin_fmaf(-piv[r] * s, s, 1.f), s);      // one Newton step
    a[r] = inv[r] * s;
  }
  return bad;
}

// Tile of slot s of a wave: waves 0 ... 7 hold the diagonal tile of their own row in slot 0 and two tiles of the row above
// (finished when they factor), waves 8 ... 15 five tiles each, spread over the rows.  row = 8: none.
__device__ __forceinline__ void leaf_slot(int wave, int s, int& row, int& col) {
  int t;
  if (wave < 8) {
    if (s == 0) { row = col = wave; return; }
    row = s < 3 ? (wave + 7) & 7 : 8;
    t = s - 1;
  } else {
    const int u = 8 * s + wave - 8;
    row = u / 5;
    t = 2 + u % 5;
  }
  col = t < row ? t : t + 1;
}

// The n x n block at `blk` (row stride ld, lower triangle) is replaced by the inverse of its Cholesky factor (zeros
// above the diagonal).  Returns the 1-based index of the first non-positive pivot inside the block, or 0, to every
// thread.  All 1024 threads of the work group call it.  (26 us for n = 128 as a recursion on an LDS-resident block that
// handled 16 x 16 blocks one row per lane; 16.7 us in this form, launch included.)
__device__ __forceinline__ int leaf_block(float* __restrict__ blk, int64_t ld, int n, LeafShared& sh, int tid) {
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int nb = (n + LT - 1) / LT;
  const bool vec = (ld & 3) == 0 && (reinterpret_cast<uintptr_t>(blk) & 15) == 0 && (n & 3) == 0;
  int row[LEAF_SLOTS], col[LEAF_SLOTS];
  floatx4 acc[LEAF_SLOTS];
#pragma unroll
  for (int s = 0; s < LEAF_SLOTS; ++s) {
    leaf_slot(wave, s, row[s], col[s]);
    if (row[s] >= nb || col[s] >= nb) row[s] = 8;
    acc[s] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (row[s] < 8 && col[s] >= row[s]) {
      // element (16 row + 4 g + r, 16 col + c) of U's side is element (16 col + c, 16 row + 4 g + r) of the lower triangle
      const int i = LT * col[s] + c, j = LT * row[s] + 4 * g;
      const float* src = blk + static_cast<int64_t>(i) * ld + j;
      if (vec) {
        if (i < n && j < n && j <= i) acc[s] = *reinterpret_cast<const floatx4*>(src);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (i < n && j + r <= i) acc[s][r] = src[r];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (i >= n) acc[s][r] = i == j + r ? 1.f : 0.f;      // identity padding
        if (j + r > i) acc[s][r] = 0.f;
      }
    }
  }
  if (tid == 0) sh.bad = 0;
#pragma unroll 1
  for (int k = 0; k < nb; ++k) {
    if (wave == k) {
      __builtin_amdgcn_s_setprio(3);
      const int bad = leaf_tile_inverse(acc[0], lane);
#pragma unroll
      for (int r = 0; r < 4; ++r) sh.inv[(4 * g + r) * LEAF_INV_LD + c] = acc[0][r];
      if (bad != 0 && lane == 0 && sh.bad == 0) sh.bad = LT * k + bad;
      __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < LEAF_SLOTS; ++s) {
      if (row[s] != k) continue;
      if (col[s] != k) {
        const floatx4 m = *reinterpret_cast<const floatx4*>(sh.inv + c * LEAF_INV_LD + 4 * g);
        floatx4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int r = 0; r < 4; ++r) p = mfma16(m[r], acc[s][r], p);
        acc[s] = p;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) sh.row[(4 * g + r) * LEAF_ROW_LD + LT * col[s] + c] = acc[s][r];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < LEAF_SLOTS; ++s) {
      if (row[s] > k && row[s] < 8 && (col[s] >= row[s] || col[s] <= k)) {
        const float* pa = sh.row + 4 * g * LEAF_ROW_LD + LT * row[s] + c;
        const float* pb = sh.row + 4 * g * LEAF_ROW_LD + LT * col[s] + c;
        float av[4], bv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          av[r] = -pa[r * LEAF_ROW_LD];
          bv[r] = pb[r * LEAF_ROW_LD];
        }
        __builtin_amdgcn_sched_barrier(0);       // all eight reads before the first product: one wait, not one per step
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[s] = mfma16(av[r], bv[r], acc[s]);
      }
    }
  }
  // every element of the block was read before the first barrier released the last row of tiles that needed it
#pragma unroll
  for (int s = 0; s < LEAF_SLOTS; ++s) {
    if (row[s] >= 8) continue;
    const int j = LT * col[s] + c;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = LT * row[s] + 4 * g + r;
      if (i < n && j < n) blk[static_cast<int64_t>(i) * ld + j] = col[s] > row[s] ? 0.f : acc[s][r];
    }
  }
  return sh.bad;
}

}  // namespace ak
