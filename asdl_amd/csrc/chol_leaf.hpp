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
// What bounds it: the chain factor k -> U_k,k+1 -> update of diagonal tile k + 1 -> factor k + 1.  Wave 0 runs nothing
// but this chain, at the highest priority; eight waves on the other three SIMDs hold one column of tiles each, form
// row k and update the rows below beside the next factor, and publish the two tiles that the chain needs next.  The right
// operand of every product of a column is that column's own tile of row k, in registers.  1.4 us per row of tiles, the
// factor 0.9 of it; with all waves in step (panel and update of all tiles between two factors) it was 2.2 us.
#pragma once
#include "common.hpp"

namespace ak {

constexpr int LEAF = 128;
constexpr int LT = 16;                       // tile
constexpr int LEAF_THREADS = 1024;
constexpr int LEAF_TILES = LEAF / LT;
constexpr int LEAF_ROW_LD = LEAF + 4;        // 4 rows apart: 16 banks apart, so the rows 4 g + r of one step do not collide
constexpr int LEAF_INV_LD = LT + 4;

struct LeafShared {
  float row[LT * LEAF_ROW_LD];
  float inv[LT * LEAF_INV_LD];
  floatx4 first[64], super[64], diag[64];      // published tiles: (0, 0), (k, k + 1), (k + 1, k + 1)
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
__device__ __forceinline__ void leaf_tile_step(floatx4& a, floatx4& inv, floatx4& piv, int g, int c) {
  // the 4 x 4 block on the diagonal, in every lane: column i of its lower triangle sits in lane (Q, 4 Q + i)
  float d[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r <= i; ++r) d[i][r] = lane_bcast(a[r], 16 * Q + 4 * Q + i);
  float l[4][4], rec[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float p = fmaxf(d[k][k], 1e-36f);               // a pivot that is not positive (or NaN) is reported by the caller
    const float r = __builtin_amdgcn_rcpf(p);             // hardware reciprocal; its error e corrects the quotients
    const float e = __builtin_fmaf(-p, r, 1.f);
    rec[k] = __builtin_fmaf(e, r, r);
#pragma unroll
    for (int i = k + 1; i < 4; ++i) {
      const float q = d[i][k] * r;
      l[i][k] = __builtin_fmaf(q, e, q);
    }
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
// L^-1 of its Cholesky factor (zeros above the diagonal).  L D L^T by blocks of 4 pivots: the 4 x 4 blocks are factored and
// inverted by every lane for itself (ten lane reads and a chain of four reciprocals; no square root before the end), and
// the rank-4 updates of the tile and of its inverse are one matrix instruction each.  piv: the pivots, register r of the
// lanes of row group g holds pivot 4 g + r.
template <class AfterFirst>
__device__ __forceinline__ void leaf_tile_inverse(floatx4& a, floatx4& piv, int lane, AfterFirst&& after_first_step) {
  const int g = lane >> 4, c = lane & 15;
  floatx4 inv;
  piv = floatx4{1.f, 1.f, 1.f, 1.f};
#pragma unroll
  for (int r = 0; r < 4; ++r) inv[r] = 4 * g + r == c ? 1.f : 0.f;
  leaf_tile_step<0>(a, inv, piv, g, c);
  after_first_step();
  leaf_tile_step<1>(a, inv, piv, g, c);
  leaf_tile_step<2>(a, inv, piv, g, c);
  leaf_tile_step<3>(a, inv, piv, g, c);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float p = fmaxf(piv[r], 1e-36f);
    float s = __builtin_amdgcn_rsqf(p);
    s = __builtin_fmaf(0.5f * s, __builtin_fmaf(-p * s, s, 1.f), s);      // one Newton step
    a[r] = inv[r] * s;
  }
}

// 0 or the 1-based index of the first pivot of leaf_tile_inverse that is not positive.
__device__ __forceinline__ int leaf_first_bad(const floatx4& piv) {
  const bool ok = piv[0] > 0.f && piv[1] > 0.f && piv[2] > 0.f && piv[3] > 0.f;
  const uint64_t bad = __ballot(!ok);
  if (bad == 0) return 0;
  const int at = __builtin_ctzll(bad);                 // a lane of the first row group with a bad pivot
  const int r = !(piv[0] > 0.f) ? 1 : !(piv[1] > 0.f) ? 2 : !(piv[2] > 0.f) ? 3 : 4;
  return 4 * (at >> 4) + __builtin_amdgcn_readlane(r, at);
}

// The column of tiles a wave holds (8: none).  None of the waves shares a SIMD with wave 0, beside whose priority it would
// be the last one at every barrier; the columns are dealt so that the three SIMDs have about the same number of updates.
__device__ __forceinline__ int leaf_column(int wave) {
  constexpr uint64_t kColumn = 0x8888821854380678ull;       // wave 0 in the lowest hex digit
  return static_cast<int>((kColumn >> (4 * wave)) & 15);
}

// The elimination itself.  load(i, j): tile (i, j), i <= j, of U's side of the block in the accumulator layout; store(i, j,
// tile): takes tile (i, j) of L^-1, i >= j (both called by the wave that holds column j, with constant i, all loads before the
// first barrier and all stores after the last product).  nb: rows of tiles of the block.  Returns the 1-based index of the
// first non-positive pivot inside the block, or 0, to every thread.  All branches meet the same barriers in the same
// order: one before the loop, B_k after the factor of row k, C_k (k + 1 < nb) once row k is complete, one at the end.
template <class Load, class Store>
__device__ __forceinline__ int leaf_eliminate(int nb, LeafShared& sh, int wave, int lane, Load&& load, Store&& store) {
  const int j = leaf_column(wave);
  const int g = lane >> 4, c = lane & 15;
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  if (wave == 0) {
    __builtin_amdgcn_s_setprio(3);
    __syncthreads();
    floatx4 a = sh.first[lane], piv;
    int first_bad = 0;
#pragma unroll 1
    for (int k = 0; k < nb; ++k) {
      leaf_tile_inverse(a, piv, lane, [k]() {
        if (k > 0) __syncthreads();                            // C_(k - 1): here the chain has not got to wait for it
      });
#pragma unroll
      for (int r = 0; r < 4; ++r) sh.inv[(4 * g + r) * LEAF_INV_LD + c] = a[r];
      __syncthreads();                                         // B_k
      if (k + 1 < nb) {
        const floatx4 m = *reinterpret_cast<const floatx4*>(sh.inv + c * LEAF_INV_LD + 4 * g);
        const floatx4 t = sh.super[lane], d = sh.diag[lane];
        // two chains of two products each time: half the latency of one of four
        const floatx4 u = mfma16(m[1], t[1], mfma16(m[0], t[0], zero)) + mfma16(m[3], t[3], mfma16(m[2], t[2], zero));
        a = mfma16(-u[1], u[1], mfma16(-u[0], u[0], d)) + mfma16(-u[3], u[3], mfma16(-u[2], u[2], zero));
      }
      const int bad = leaf_first_bad(piv);
      if (bad != 0 && first_bad == 0) first_bad = LT * k + bad;
    }
    if (lane == 0) sh.bad = first_bad;
    __builtin_amdgcn_s_setprio(0);
  } else if (j < nb) {
    floatx4 acc[LEAF_TILES];
#pragma unroll
    for (int i = 0; i < LEAF_TILES; ++i) {
      acc[i] = zero;
      if (i <= j) acc[i] = load(i, j);
    }
    if (j == 0) sh.first[lane] = acc[0];
    if (j == 1) {
      sh.super[lane] = acc[0];
      sh.diag[lane] = acc[1];
    }
    __syncthreads();
    float* row = sh.row + 4 * g * LEAF_ROW_LD + c;
#pragma unroll
    for (int k = 0; k < LEAF_TILES; ++k) {
      if (k >= nb) break;
      __syncthreads();                                         // B_k
      if (j != k) {
        const floatx4 m = *reinterpret_cast<const floatx4*>(sh.inv + c * LEAF_INV_LD + 4 * g), t = acc[k];
        acc[k] = mfma16(m[1], t[1], mfma16(m[0], t[0], zero)) + mfma16(m[3], t[3], mfma16(m[2], t[2], zero));
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[k][r] = sh.inv[(4 * g + r) * LEAF_INV_LD + c];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) row[r * LEAF_ROW_LD + LT * j] = acc[k][r];
      if (k + 1 == nb) break;
      __syncthreads();                                         // C_k
      float u[LEAF_TILES][4];            // all left operands requested before the first product
#pragma unroll
      for (int i = k + 1; i < LEAF_TILES; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) u[i][r] = row[r * LEAF_ROW_LD + LT * i];
      const floatx4 b = -acc[k];
#pragma unroll
      for (int i = k + 1; i < LEAF_TILES; ++i) {
        if (j >= i || j <= k) {
          acc[i] = mfma16(u[i][1], b[1], mfma16(u[i][0], b[0], acc[i])) + mfma16(u[i][3], b[3], mfma16(u[i][2], b[2], zero));
          if (i == k + 2 && j == k + 2) {
            sh.super[lane] = acc[k + 1];
            sh.diag[lane] = acc[k + 2];
          }
        }
      }
    }
#pragma unroll
    for (int i = 0; i < LEAF_TILES; ++i)
      if (i >= j && i < nb) store(i, j, acc[i]);
  } else {
    __syncthreads();
#pragma unroll 1
    for (int k = 0; k < nb; ++k) {
      __syncthreads();                                         // B_k
      if (k + 1 < nb) __syncthreads();                         // C_k
    }
  }
  __syncthreads();
  return sh.bad;
}

// The n x n block at `blk` (row stride ld, lower triangle) is replaced by the inverse of its Cholesky factor (zeros
// above the diagonal).  Returns the 1-based index of the first non-positive pivot inside the block, or 0, to every
// thread.  All 1024 threads of the work group call it.
__device__ __forceinline__ int leaf_block(float* __restrict__ blk, int64_t ld, int n, LeafShared& sh, int tid) {
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 4, c = lane & 15;
  const int nb = (n + LT - 1) / LT;
  const bool vec = (ld & 3) == 0 && (reinterpret_cast<uintptr_t>(blk) & 15) == 0 && (n & 3) == 0;
  return leaf_eliminate(
      nb, sh, wave, lane,
      [&](int s, int col) {
        // element (16 s + 4 g + r, 16 col + c) of U's side is element (16 col + c, 16 s + 4 g + r) of the lower triangle
        const int i = LT * col + c, j = LT * s + 4 * g;
        const float* src = blk + static_cast<int64_t>(i) * ld + j;
        floatx4 v = {0.f, 0.f, 0.f, 0.f};
        if (vec) {
          if (i < n && j < n && j <= i) v = *reinterpret_cast<const floatx4*>(src);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (i < n && j + r <= i) v[r] = src[r];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (i >= n) v[r] = i == j + r ? 1.f : 0.f;      // identity padding
          if (j + r > i) v[r] = 0.f;
        }
        return v;
      },
      [&](int s, int col, const floatx4& v) {
        const int j = LT * col + c;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = LT * s + 4 * g + r;
          if (i < n && j < n) {
            blk[static_cast<int64_t>(i) * ld + j] = v[r];
            if (s != col) blk[static_cast<int64_t>(j) * ld + i] = 0.f;
          }
        }
      });
}

}  // namespace ak
