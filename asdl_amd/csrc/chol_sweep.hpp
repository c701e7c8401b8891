// Damped inverses of many small and medium matrices by a block sweep: one launch per 128 columns.  Included by
// chol_group.hip, whose plan picks between this and the right-looking factorization by their estimated times.
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
// What bounds it: the chain leaf -> update of the next diagonal block -> leaf, 25 us per step: 3 for the operands, 5.5 for
// v_k+1, 4.5 for the block's update, 12 for the leaf.  Every other work group needs less (two v and a 128 x 128 tile: 20 us)
// and runs beside it as long as the tiles of all matrices fit the device once.  That is why each work group forms the
// v_i and v_j that it needs for itself (the same value in every work group) instead of waiting for a launch that forms them
// once, and why the work group of the next diagonal block goes on to factor it in registers (chol_leaf.hpp).  True fp32
// products, sums in chunks.  Against the right-looking factorization: (784, 4 x 512, 10) 361 -> 206 us, (1153, 512)
// 526 -> 284 us, (577, 1000) 427 -> 229 us, 512 alone 180 -> 123 us.
//
// No work group reads what another one of the same launch writes: the row and column of the next step are written to
// the other half of the Y buffer, M alternates likewise, an X tile is read and written by its own work group only.
#pragma once
#include "gemm_f32.hpp"
#include "chol_leaf.hpp"

namespace ak {

constexpr int SW_LD = LEAF + 4;              // LDS row: 4 banks further per row, 16-byte reads of 8 rows do not collide
constexpr int SW_TILE = LEAF * LEAF;

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

// 128 x 128 floats at P (row stride ld, rows x cols inside), 16 values per thread, zeros outside.
__device__ __forceinline__ void sw_fetch(floatx4 (&reg)[4], const float* __restrict__ P, int ld, int rows, int cols, int tid) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int r = (tid >> 5) + 32 * u, c = 4 * (tid & 31);
    floatx4 v = {0.f, 0.f, 0.f, 0.f};
    const float* src = P + (r * ld + c);       // (at most 128 rows of at most 32768)
    if (r < rows && c + 4 <= cols) {
      v = *reinterpret_cast<const floatx4u*>(src);
    } else if (r < rows) {
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (c + e < cols) v[e] = src[e];
    }
    reg[u] = v;
  }
}

__device__ __forceinline__ void sw_stash(const floatx4 (&reg)[4], float* __restrict__ lds, bool transposed, int tid) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int r = (tid >> 5) + 32 * u, c = 4 * (tid & 31);
    if (!transposed) {
      *reinterpret_cast<floatx4*>(lds + r * SW_LD + c) = reg[u];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) lds[(c + e) * SW_LD + r] = reg[u][e];
    }
  }
}

// 32 x 32 block of a product of two [row][k] panels over k < kmax, in four accumulators: the matrix instruction rounds
// its accumulator once per two k, and long runs of roundings show in the inverses of ill-conditioned factors.
__device__ __forceinline__ floatx16 sw_dot(const float* __restrict__ pa, const float* __restrict__ pb, int kmax) {
  floatx16 part[4];
#pragma unroll
  for (int r = 0; r < 16; ++r) part[0][r] = part[1][r] = part[2][r] = part[3][r] = 0.f;
#pragma unroll 1
  for (int q = 0; q < kmax; q += 16) {
    const floatx4 a = *reinterpret_cast<const floatx4*>(pa + q), b = *reinterpret_cast<const floatx4*>(pb + q);
    const floatx4 c = *reinterpret_cast<const floatx4*>(pa + q + 8), d = *reinterpret_cast<const floatx4*>(pb + q + 8);
#pragma unroll
    for (int e = 0; e < 4; ++e) part[e] = mfma_f32(a[e], b[e], part[e]);
#pragma unroll
    for (int e = 0; e < 4; ++e) part[e] = mfma_f32(c[e], d[e], part[e]);
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) part[0][r] = (part[0][r] + part[1][r]) + (part[2][r] + part[3][r]);
  return part[0];
}

__device__ __forceinline__ void sw_put(const floatx16& v, float* __restrict__ lds, int wr, int wc, int g, int l32) {
#pragma unroll
  for (int r = 0; r < 16; ++r) lds[(32 * wr + 8 * (r >> 2) + 4 * g + (r & 3)) * SW_LD + 32 * wc + l32] = v[r];
}

// Step k (-1: only the first diagonal block of every matrix is factored).  Work groups 0 ... nleaf - 1: the next
// diagonal block of a matrix, updated and factored; the others: one tile each.
static __global__ __launch_bounds__(LEAF_THREADS) void cg_sweep_kernel(SwArgs a, const SwTask* __restrict__ leaves,
                                                                       const SwTask* __restrict__ tiles, int nleaf, int k) {
  __shared__ __attribute__((aligned(16))) float L0[LEAF * SW_LD];
  __shared__ __attribute__((aligned(16))) float L1[LEAF * SW_LD];
  __shared__ __attribute__((aligned(16))) LeafShared sh;
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
  const float* pa = L0 + (32 * wr + l32) * SW_LD + 4 * g;
  const float* pm = L1 + (32 * wc + l32) * SW_LD + 4 * g;
  const int rows_i = t.d - LEAF * bi, rows_j = t.d - LEAF * bj;
  float* __restrict__ X = a.ws + t.x_off + (leaf ? static_cast<int64_t>(bi) * (bi + 3) / 2 * SW_TILE : 0);

  if (leaf) {
    const int n = min(LEAF, rows_i), nb = (n + LT - 1) / LT, g4 = lane >> 4, c = lane & 15;
    const float l = a.lam[static_cast<int64_t>(t.mat) * a.lam_stride];
    if (k >= 0) {
      floatx4 rm[4], ry[4];
      sw_fetch(rm, M, LEAF, LEAF, LEAF, tid);
      if (k == 0) sw_fetch(ry, A + static_cast<int64_t>(LEAF) * bi * t.d, t.d, rows_i, kcols, tid);
      else sw_fetch(ry, Y + static_cast<int64_t>(bi) * SW_TILE, LEAF, LEAF, LEAF, tid);
      sw_stash(rm, L1, false, tid);
      sw_stash(ry, L0, false, tid);
    }
    // Tiles (s, col) of 16 x 16, s <= col: element (16 s + 4 g + r, 16 col + c) is element (16 col + c, 16 s + 4 g + r) of the
    // lower triangle.  They are dealt to all waves for the update and handed to the waves of the columns through the LDS.
    constexpr int kMine = 3;
    int ts[kMine], tc[kMine];
    floatx4 upd[kMine];          // the block's old values: under way while the product runs
#pragma unroll
    for (int u = 0; u < kMine; ++u) {
      const int id = wave + 16 * u;           // (integers only: the waves' branches below have to be scalar)
      tc[u] = (id >= 1) + (id >= 3) + (id >= 6) + (id >= 10) + (id >= 15) + (id >= 21) + (id >= 28) + (id >= 36);
      ts[u] = id - tc[u] * (tc[u] + 1) / 2;
      upd[u] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (tc[u] >= nb) continue;
      const int i = LT * tc[u] + c, j = LT * ts[u] + 4 * g4;
      if (k > 0) {
        upd[u] = *reinterpret_cast<const floatx4*>(X + i * LEAF + j);
      } else {
        const float* src = A + static_cast<int64_t>(LEAF * bi + i) * t.d + LEAF * bi + j;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (i < n && j + r <= i) upd[u][r] = src[r] + (j + r == i ? l : 0.f);
      }
    }
    if (k >= 0) {
      __syncthreads();
      const floatx16 v = sw_dot(pa, pm, 32 * (wc + 1));
      __syncthreads();
      sw_put(v, L0, wr, wc, g, l32);
      __syncthreads();
    }
    floatx4* handed = reinterpret_cast<floatx4*>(L1);
#pragma unroll
    for (int u = 0; u < kMine; ++u) {
      if (tc[u] >= nb) continue;
      const int i = LT * tc[u] + c, j = LT * ts[u] + 4 * g4;
      if (k >= 0) {
        const float* pr = L0 + (LT * ts[u] + c) * SW_LD + 4 * g4;
        const float* pc = L0 + (LT * tc[u] + c) * SW_LD + 4 * g4;
        floatx4 p0 = {0.f, 0.f, 0.f, 0.f}, p1 = p0;
#pragma unroll 2
        for (int q = 0; q < LEAF; q += 32) {
          const floatx4 u0 = *reinterpret_cast<const floatx4*>(pr + q), w0 = *reinterpret_cast<const floatx4*>(pc + q);
          const floatx4 u1 = *reinterpret_cast<const floatx4*>(pr + q + 16), w1 = *reinterpret_cast<const floatx4*>(pc + q + 16);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            p0 = mfma16(u0[e], w0[e], p0);
            p1 = mfma16(u1[e], w1[e], p1);
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) upd[u][r] -= p0[r] + p1[r];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (i >= n) upd[u][r] = i == j + r ? 1.f : 0.f;      // identity padding
        if (j + r > i) upd[u][r] = 0.f;
      }
      handed[(tc[u] * (tc[u] + 1) / 2 + ts[u]) * 64 + lane] = upd[u];
    }
    __syncthreads();
    float* __restrict__ Mn = a.ws + t.m_off + ((k + 1) & 1) * SW_TILE;
    const int bad = leaf_eliminate(
        nb, sh, wave, lane, [&](int s, int col) { return handed[(col * (col + 1) / 2 + s) * 64 + lane]; },
        [&](int s, int col, const floatx4& v) {
#pragma unroll
          for (int r = 0; r < 4; ++r) Mn[(LT * s + 4 * g4 + r) * LEAF + LT * col + c] = v[r];
          if (s != col) *reinterpret_cast<floatx4*>(Mn + (LT * col + c) * LEAF + LT * s + 4 * g4) = floatx4{0.f, 0.f, 0.f, 0.f};
        });
    if (nb < LEAF_TILES) {         // the identity beyond the matrix
      for (int e = tid; e < SW_TILE; e += LEAF_THREADS) {
        const int i = e / LEAF, j = e % LEAF;
        if (i >= LT * nb || j >= LT * nb) Mn[e] = i == j ? 1.f : 0.f;
      }
    }
    if (tid == 0 && (a.skip == nullptr || a.skip[static_cast<int64_t>(t.mat) * a.skip_stride] != 0)) {
      const int where = bad != 0 && LEAF * bi + bad <= t.d ? LEAF * bi + bad : 0;
      if (k < 0) a.info[t.mat] = where;
      else if (where != 0 && a.info[t.mat] == 0) a.info[t.mat] = where;
    }
    return;
  }

  floatx4 rm[4], ry[4];
  sw_fetch(rm, M, LEAF, LEAF, LEAF, tid);
  if (!ik) {
    if (k == 0) sw_fetch(ry, A + static_cast<int64_t>(LEAF) * bi * t.d, t.d, rows_i, kcols, tid);
    else sw_fetch(ry, Y + static_cast<int64_t>(bi) * SW_TILE, LEAF, LEAF, LEAF, tid);
    sw_stash(ry, L0, false, tid);
  }
  sw_stash(rm, L1, false, tid);
  const bool second = !diag && !jk;
  if (second) {
    if (k == 0) sw_fetch(ry, A + static_cast<int64_t>(LEAF) * bj * t.d, t.d, rows_j, kcols, tid);
    else sw_fetch(ry, Y + static_cast<int64_t>(bj) * SW_TILE, LEAF, LEAF, LEAF, tid);
  }
  __syncthreads();
  floatx16 vi, vj;
  if (!ik) vi = sw_dot(pa, pm, 32 * (wc + 1));       // M_k is lower triangular
  if (second) {
    __syncthreads();
    sw_stash(ry, L0, false, tid);
    __syncthreads();
    vj = sw_dot(pa, pm, 32 * (wc + 1));
  }
  if (ik || jk) sw_fetch(rm, M, LEAF, LEAF, LEAF, tid);      // v_k = M_k^T
  __syncthreads();
  if (ik) sw_stash(rm, L0, true, tid);
  else sw_put(vi, L0, wr, wc, g, l32);
  if (!diag) {
    if (jk) sw_stash(rm, L1, true, tid);
    else sw_put(vj, L1, wr, wc, g, l32);
  }

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
  __syncthreads();
  if (upper) return;
  floatx16 sum = sw_dot(L0 + (32 * wr + l32) * SW_LD + 4 * g, (diag ? L0 : L1) + (32 * wc + l32) * SW_LD + 4 * g, LEAF);
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
