// 256 x 128 tile of a product of fp32 matrices on two fp16 pieces per element (gemm_x3.hpp's pieces, layouts and order of sums:
// the same bits as its 128 x 128 tile), for launches that fill the device with tiles of this size.
//
// With 64 x 64 per wave the LDS is as busy as the matrix pipes: per k-tile of 32 and CU 128 KB of fragments and 64 KB of pieces,
// 1536 cycles at 128 B each, as the 24 matrix instructions of two waves per SIMD.  128 x 64 per wave reads 24 KB for 48 matrix
// instructions: 1152 cycles of 1536, and each element of B is split half as often.  Two work groups per CU, single-buffered as
// there: one splits while the other multiplies. 
// Measured, 128 x 128 and this tile: 4096^3 465 and 408 us (1000 TFLOP/s of piece products), a 12-layer decoder's
// preconditioning products 1240 and 1120 us.
#pragma once
#include "gemm_x3.hpp"

namespace ak {

constexpr int HT_BT = 256;
constexpr int HT_LDS = 2 * (2 + 1) * X3_PLANE;       // two planes of A's two halves and of B

// Tile at rows i0 ... i0 + 255 (which begins inside the matrix) and column tile tj; TILE_ALL, K_FULL, alpha and beta = 0.
template <bool A_KC, bool B_KC>
__device__ __forceinline__ void gemm_half_tall_tile(const GemmParams& p, int i0, int tj, AK_LDS3 unsigned char* lds) {
  constexpr int BK = X3_BK;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wr = wave >> 1, wc = wave & 1, l32 = lane & 31;
  const int j0 = tj * X3_BT, nk = (p.K + BK - 1) / BK;
  const float* __restrict__ A = p.A;
  const float* __restrict__ B = p.B;
  AK_LDS3 unsigned char* panelB = lds + 4 * X3_PLANE;
  floatx16 acc[4][2];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;

  auto mainloop = [&](auto interior_tag) {
    constexpr bool INTERIOR = decltype(interior_tag)::value;
    X3Fetch ra[2], rb;
    auto fetch = [&](int kt) {
      const int k0 = kt * BK;
#pragma unroll
      for (int s = 0; s < 2; ++s) x3_fetch<INTERIOR>(ra[s], A, p.lda, A_KC, i0 + 128 * s, p.M, k0, p.K, tid);
      x3_fetch<INTERIOR>(rb, B, p.ldb, B_KC, j0, p.N, k0, p.K, tid);
    };
    auto stash = [&] {
#pragma unroll
      for (int s = 0; s < 2; ++s) x3_stash<2, true>(ra[s], lds + 2 * s * X3_PLANE, A_KC, tid, p.scaleA);
      x3_stash<2, true>(rb, panelB, B_KC, tid, p.scaleB);
    };
    auto multiply = [&] {
      AK_LDS3 unsigned char* pa = lds + 2 * wr * X3_PLANE;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        bf16x8 fb[2][2];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int b = 0; b < 2; ++b) fb[b][s] = x3_frag(panelB + s * X3_PLANE, B_KC, 64 * wc + 32 * b + l32, h, lane);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const bf16x8 f0 = x3_frag(pa, A_KC, 32 * a + l32, h, lane), f1 = x3_frag(pa + X3_PLANE, A_KC, 32 * a + l32, h, lane);
          // smallest terms first
#pragma unroll
          for (int b = 0; b < 2; ++b) acc[a][b] = x3_mfma<true>(f0, fb[b][1], acc[a][b]);
#pragma unroll
          for (int b = 0; b < 2; ++b) acc[a][b] = x3_mfma<true>(f1, fb[b][0], acc[a][b]);
#pragma unroll
          for (int b = 0; b < 2; ++b) acc[a][b] = x3_mfma<true>(f0, fb[b][0], acc[a][b]);
        }
      }
    };
    if (nk > 0) {
      fetch(0);
      stash();
    }
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
      if (kt + 1 < nk) fetch(kt + 1);       // next k-tile's global loads fly during this one's MFMAs
      multiply();
      __syncthreads();                      // everybody is done reading this k-tile
      if (kt + 1 < nk) stash();
      __syncthreads();
    }
  };
  if (i0 + HT_BT <= p.M && j0 + X3_BT <= p.N && p.K % BK == 0) mainloop(std::true_type{});
  else mainloop(std::false_type{});

  float vmax = 0.f;
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int gj = j0 + 64 * wc + 32 * b + l32;
    if (gj >= p.N) continue;
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gi = i0 + 128 * wr + 32 * a + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (gi >= p.M) continue;
        const float v = p.alpha * acc[a][b][r];
        vmax = gemm_fold_absmax(vmax, v, false, 0);
        p.C[static_cast<int64_t>(gi) * p.ldc + gj] = v;
      }
  }
  if (p.absmax_out != nullptr) gemm_store_absmax(p.absmax_out, vmax, lane);
}

// gemm_x3_grouped_kernel<2, true> for launches of many tiles: two tile rows per work group.  Products with beta, symmetric
// ones and a last odd tile row go tile by tile.
static __global__ __launch_bounds__(256, 2) void gemm_half_grouped_kernel(const int64_t* __restrict__ table, int count) {
  __shared__ __attribute__((aligned(16))) unsigned char smem[HT_LDS];
  GemmParams p;
  int ti, tj;
  if (!grouped_lookup(table, count, blockIdx.x, p, ti, tj)) return;
  AK_LDS3 unsigned char* lds = (AK_LDS3 unsigned char*)smem;
  bool tall = false;
  if (p.beta == 0.f && p.tile_mode == TILE_ALL) {
    // the product's first work groups take the pairs of tile rows, the next ones a last odd row, the rest none: side by side,
    // so that the XCDs, which take work groups in turn, get as many of them each
    const int tm = (p.M + X3_BT - 1) / X3_BT, tn = (p.N + X3_BT - 1) / X3_BT, local = ti * tn + tj, pairs = tm / 2 * tn;
    tall = local < pairs;
    if (!tall && local - pairs >= (tm & 1) * tn) return;
    ti = tall ? 2 * (local / tn) : tm - 1;
    tj = tall ? local % tn : local - pairs;
  }
  grouped_half_scales(table, count, blockIdx.x, p);
  if (tall) {
    if (p.transA == 0) {
      if (p.transB != 0) gemm_half_tall_tile<true, true>(p, ti * X3_BT, tj, lds);
      else gemm_half_tall_tile<true, false>(p, ti * X3_BT, tj, lds);
    } else {
      if (p.transB != 0) gemm_half_tall_tile<false, true>(p, ti * X3_BT, tj, lds);
      else gemm_half_tall_tile<false, false>(p, ti * X3_BT, tj, lds);
    }
  } else if (p.transA == 0) {
    if (p.transB != 0) gemm_x3_tile<2, false, 1, 1, true>(p, ti, tj, 0, lds);
    else gemm_x3_tile<2, false, 1, 0, true>(p, ti, tj, 0, lds);
  } else {
    if (p.transB != 0) gemm_x3_tile<2, false, 0, 1, true>(p, ti, tj, 0, lds);
    else gemm_x3_tile<2, false, 0, 0, true>(p, ti, tj, 0, lds);
  }
}

}  // namespace ak
