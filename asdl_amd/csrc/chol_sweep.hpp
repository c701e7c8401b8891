// Damped inverses of many small and medium matrices by a block sweep: one launch per 128 columns.  Included by
// chol_group.hip, whose plan leaves groups of three rounds of tiles a step and more to the chain of chol_chain.hpp where that saves enough (cg_build).
//
// In-place block Gauss-Jordan elimination on the Cholesky factors.  With M_k = L_kk^-1 of the updated diagonal block,
// step k is ONE symmetric rank-128 update of the whole lower triangle,
//     v_i = Y_i M_k^T   (Y_i: block (i, k) for i > k, block (k, i) transposed for i < k, the identity for i = k)
//     X_ij <- X_ij - v_i v_j^T  for i > k,      X_ij <- X_ij + v_i v_j^T  for i <= k       (j <= i; old X_ij = 0 in row / column k)
// For i > k v_i is block (i, k) of the Cholesky factor; for i <= k it is block (k, i) of L^-1, transposed.  So the three
// parts of the triangle hold the Schur complement (i, j > k), the partial sums of L^-1's rows (i > k >= j) and of the result
// (i, j <= k): factorization, triangular inverse and L^-T L^-1 advance together, d^3 FLOP in all as POTRF + POTRI, in
// ceil(d / 128) dependent steps instead of 3 ceil(d / 128) + 2 log2 + 1 launches.
//
// What bounds it: the chain leaf -> update of the next diagonal block -> leaf, 22 us per step: 2 for the operands, 4.2 for
// v_k+1, 4.6 for the block's update, 12 for the leaf (54k cycles).  Every other work group needs less (two v and a 128 x 128
// tile: 14 to 18 us) and runs beside it as long as the tiles of all matrices fit the device once.  That is why each work group
// forms the v_i and v_j that it needs for itself (the same value in every work group) instead of waiting for a launch that forms
// them once, and why the work group of the next diagonal block goes on to factor it in registers (chol_leaf.hpp).
// Three bf16 pieces per operand (chol_step.hpp) instead of true fp32 products: (784, 4 x 512, 10) 206 -> 180 us, (1153, 512)
// 284 -> 249, 512 alone 123 -> 110, 2 x 2048 768 -> 566; error against 64 bits of the inverses 2.0e-7 to 3.7e-7 (fp32: 2.0e-7 to
// 3.7e-7), of rank-deficient ones (16 of 512, 64 of 1153) 7.8e-4 and 4.6e-4 (1.2e-3 and 8.1e-4).
//
// No work group reads what another one of the same launch writes: the row and column of the next step are written to
// the other half of the Y buffer, M alternates likewise, an X tile is read and written by its own work group only.
#pragma once
#include "chol_step.hpp"

namespace ak {

constexpr int SW_TILE = ST_TILE;

struct SwTask {               // one 128 x 128 tile of a lower triangle; of a leaf list: one matrix (x_off: its first tile)
  int64_t x_off, y_off, m_off;     // floats from the workspace base: X tile, Y (2 x [nb][128][128]), M (2 x [128][128])
  int32_t mat, d, nb, bi, bj, pad0;
};

struct SwArgs {
  float* ws;
  const float* const* A_list;
  float* const* out_list;
  const float* lam;
  const int* skip;
  int* info;
  int lam_stride, skip_stride;
};

// Step k (-1: only the first diagonal block of every matrix is factored).  Work groups 0 ... nleaf - 1: the next
// diagonal block of a matrix, updated and factored; the others: one tile each.
static __global__ __launch_bounds__(LEAF_THREADS) void cg_sweep_kernel(SwArgs a, const SwTask* __restrict__ leaves,
                                                                       const SwTask* __restrict__ tiles, int nleaf, int k) {
  hold_cu();
  __shared__ __attribute__((aligned(16))) unsigned char st_smem[ST_LDS];
  __shared__ __attribute__((aligned(16))) LeafShared sh;
  AK_LDS3 unsigned char* lds = (AK_LDS3 unsigned char*)st_smem;
  const bool leaf = static_cast<int>(blockIdx.x) < nleaf;
  const SwTask& t = leaf ? leaves[blockIdx.x] : tiles[blockIdx.x - nleaf];
  const int bi = leaf ? k + 1 : t.bi, bj = leaf ? k + 1 : t.bj;
  if (!leaf && k + 1 < t.nb && bi == k + 1 && bj == k + 1) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31;
  // column blocks over the groups of four waves: one wave of each column block, whose contractions differ in length, per SIMD
  const int wr = wave & 3, wc = wave >> 2;
  const bool ik = bi == k, jk = bj == k, diag = bi == bj;
  const float* __restrict__ A = a.A_list[t.mat];
  const float* __restrict__ Y = a.ws + t.y_off + static_cast<int64_t>(k & 1) * t.nb * SW_TILE;
  const float* __restrict__ M = a.ws + t.m_off + (k & 1) * SW_TILE;
  const int kcols = min(LEAF, t.d);
  const int rows_i = t.d - LEAF * bi, rows_j = t.d - LEAF * bj;
  float* __restrict__ X = a.ws + t.x_off + (leaf ? static_cast<int64_t>(bi) * (bi + 3) / 2 * SW_TILE : 0);
  auto fetch_y = [&](StPart& y, int b, int rows) {
    if (k == 0) st_fetch(y, A + static_cast<int64_t>(LEAF) * b * t.d, t.d, rows, kcols, tid);
    else st_fetch(y, Y + static_cast<int64_t>(b) * SW_TILE, LEAF, LEAF, LEAF, tid);
  };
  auto stage_m = [&](const StPart& m) {
    st_stash(m.v[0], lds, false, tid);
    st_stash(m.v[1], lds + ST_HALF, false, tid);
  };

  if (leaf) {
    const int n = min(LEAF, rows_i);
    const float l = a.lam[static_cast<int64_t>(t.mat) * a.lam_stride];
    StPart m, y;
    if (k >= 0) {
      st_fetch(m, M, LEAF, LEAF, LEAF, tid);
      fetch_y(y, bi, rows_i);
    }
    floatx16 upd;
    st_leaf_fetch(upd, [&](int i, int j) {
      if (k > 0) return *reinterpret_cast<const floatx4*>(X + i * LEAF + j);
      const float* src = A + static_cast<int64_t>(LEAF * bi + i) * t.d + LEAF * bi + j;
      floatx4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = src[min(r, i - min(i, j))] + (j + r == i ? l : 0.f);      // (what lies above the diagonal is dropped)
      return v;
    }, n, tid);
    floatx16 v;
    if (k >= 0) {
      stage_m(m);
      v = st_panel(y, false, lds, wr, wc, tid);
    }
    float* __restrict__ Mn = a.ws + t.m_off + ((k + 1) & 1) * SW_TILE;
    const int bad = st_leaf(upd, [](int, int, const floatx4&) {}, v, k >= 0, n, Mn, lds, sh, wr, wc, tid);
    if (tid == 0 && (a.skip == nullptr || a.skip[static_cast<int64_t>(t.mat) * a.skip_stride] != 0)) {
      const int where = bad != 0 && LEAF * bi + bad <= t.d ? LEAF * bi + bad : 0;
      if (k < 0) a.info[t.mat] = where;
      else if (where != 0 && a.info[t.mat] == 0) a.info[t.mat] = where;
    }
    return;
  }

  StPart m, y;
  st_fetch(m, M, LEAF, LEAF, LEAF, tid);
  if (!ik) fetch_y(y, bi, rows_i);
  stage_m(m);
  floatx16 vi, vj;
  if (!ik) vi = st_panel(y, false, lds, wr, wc, tid);
  if (!diag && !jk) {
    fetch_y(y, bj, rows_j);
    __syncthreads();
    vj = st_panel(y, false, lds, wr, wc, tid);
  }
  if (ik) vi = st_own(M, tid);             // v_k = M_k^T
  if (jk && !diag) vj = st_own(M, tid);

  const bool last = k + 1 == t.nb, upper = diag && wr < wc;      // the blocks above the diagonal are not needed
  const int i0 = 32 * wr + 4 * g, j = 32 * wc + l32;             // element r of a wave's block: (i0 + 8 (r / 4) + r % 4, j)
  floatx16 old;
#pragma unroll
  for (int r = 0; r < 16; ++r) old[r] = 0.f;
  if (!ik && !jk && !upper) {
    if (k == 0) {
      const float l = a.lam[static_cast<int64_t>(t.mat) * a.lam_stride];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = i0 + 8 * (r >> 2) + (r & 3);
        if (i < rows_i && j < rows_j && (!diag || i >= j))
          old[r] = A[static_cast<int64_t>(LEAF * bi + i) * t.d + LEAF * bj + j] + (diag && i == j ? l : 0.f);
      }
    } else if (diag) {
#pragma unroll
      for (int r = 0; r < 16; ++r) old[r] = X[(i0 + 8 * (r >> 2) + (r & 3)) * LEAF + j];
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx4 v = reinterpret_cast<const floatx4*>(X)[1024 * q + tid];
#pragma unroll
        for (int e = 0; e < 4; ++e) old[4 * q + e] = v[e];
      }
    }
  }
  floatx16 sum = st_outer(vi, ik, vj, jk, diag, lds, wr, wc, tid);
  if (upper) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) sum[r] = bi <= k ? old[r] + sum[r] : old[r] - sum[r];

  if (last) {
    if (a.skip != nullptr && a.skip[static_cast<int64_t>(t.mat) * a.skip_stride] == 0) return;
    float* __restrict__ C = a.out_list[t.mat];
    const int gj = LEAF * bj + j;
    if (gj >= t.d) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int gi = LEAF * bi + i0 + 8 * q;
      const floatx4 v = {sum[4 * q], sum[4 * q + 1], sum[4 * q + 2], sum[4 * q + 3]};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (gi + e < t.d && gi + e >= gj) C[static_cast<int64_t>(gi + e) * t.d + gj] = v[e];
      float* dst = C + static_cast<int64_t>(gj) * t.d + gi;     // the mirror image
      if (gi > gj && gi + 4 <= t.d) *reinterpret_cast<floatx4u*>(dst) = v;
      else
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (gi + e > gj && gi + e < t.d) dst[e] = v[e];
    }
    return;
  }
  float* __restrict__ Yn = a.ws + t.y_off + static_cast<int64_t>((k + 1) & 1) * t.nb * SW_TILE;
  if (bj == k + 1) {             // column k + 1 below the diagonal
    float* __restrict__ dst = Yn + static_cast<int64_t>(bi) * SW_TILE + j;
#pragma unroll
    for (int r = 0; r < 16; ++r) dst[(i0 + 8 * (r >> 2) + (r & 3)) * LEAF] = sum[r];
  } else if (bi == k + 1) {      // row k + 1, transposed
    float* __restrict__ dst = Yn + static_cast<int64_t>(bj) * SW_TILE + j * LEAF + i0;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<floatx4*>(dst + 8 * q) = floatx4{sum[4 * q], sum[4 * q + 1], sum[4 * q + 2], sum[4 * q + 3]};
  } else if (diag) {
#pragma unroll
    for (int r = 0; r < 16; ++r) X[(i0 + 8 * (r >> 2) + (r & 3)) * LEAF + j] = sum[r];
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      reinterpret_cast<floatx4*>(X)[1024 * q + tid] = floatx4{sum[4 * q], sum[4 * q + 1], sum[4 * q + 2], sum[4 * q + 3]};
  }
}

}  // namespace ak
