// Damped inverses of groups that are too large for the block sweep (chol_sweep.hpp; cg_build): the same elimination, with all but the
// columns of the current group of CG_GROUP blocks left to one product of that depth.  Included by chol_group.hip.
//
// The sweep's step k updates the whole triangle by v v^T of 128 columns (v_i = Y_i M_k^T): beyond one round of tiles on the
// device its updates cost more than the chain leaf -> v -> leaf they run beside, at a sixteenth of an operation per byte of the
// triangle.  Here the steps k of a group [g0, ge) update only what the group's further steps read,
//     tiles (i, j) with g0 <= k < j < ge, i >= j: the columns that follow;   tiles (r, i) with k < r < ge, i <= k: the rows that follow;
//     tile (ge, ge): the next group's first diagonal block, so that its leaf need not wait for the product,
// and keep every v_i as rows of V [d][128 CG_GROUP].  Each of those tiles forms the two v that it needs for itself (three products
// instead of one, but no second launch); where they are more than the device takes at once, the launch forms the v only and
// the tiles are products of a launch of their own.  At the end of the group all tiles get their update from V at once (the
// products of CgOp: X -+ V V^T, 512 deep, on the split-operand tiles of the grouped products).  Work: d^3 in all, as in the sweep;
// chain: 26 to 30 us per 128 columns while a step has up to a tile per CU, and one product per 512.
//
// W: the work matrix (lower triangle, row-major, dp columns), lam added by cg_copy_in_kernel.  Tiles (r, i) inside a group live in
// E from the step that makes them (i = k), because their place in W is column k, which the same launch reads.  M alternates
// between two buffers by k, V by the group (the next group's first leaf writes M^T there while this group's V is read).
// Bound by the chain (26 to 30 us a step: the leaf 12, its v and update 9, its operands from a row-major matrix 3) and by the
// products (80 us per 512 columns for 2 x 4096, 0.65 PFLOP/s of 16-bit work: 1056 tiles, two a CU, that split their operands).
// Against a factorization with leaf, panel and update launches, a triangular inverse by levels and M^T M (3 launches a block and two a
// level): 4096 1825 -> 1250 us, 2 x 4096 2110 -> 1625, 16 decoder factors of 768 ... 3073 2545 -> 1835, the 108 factors of
// ResNet-50 4715 -> 4150, 24 x 1100 870 -> 673.
#pragma once
#include "chol_step.hpp"

namespace ak {

constexpr int CG_GROUP = 4;                           // block columns of a group
constexpr int CC_VLD = CG_GROUP * LEAF;
enum { CC_LEAF = 0, CC_TILE = 1, CC_PANEL = 2 };

struct CcTask {
  int64_t w_off, v_off, e_off, m_off;        // floats from the workspace base; V: two of [dp][CC_VLD], E: six tiles, M: two
  int32_t mat, d, dp, nb;
  int32_t kind, bi, bj, g0;                  // g0: first block of the group of step k
};

struct CcArgs {
  float* ws;
  const int* skip;
  int* info;
  int skip_stride;
};

// Step k (-1: the first diagonal blocks are factored), one work group per task.
static __global__ __launch_bounds__(LEAF_THREADS) void cg_chain_kernel(CcArgs a, const CcTask* __restrict__ tasks, int k) {
  __shared__ __attribute__((aligned(16))) unsigned char st_smem[ST_LDS];
  __shared__ __attribute__((aligned(16))) LeafShared sh;
  AK_LDS3 unsigned char* lds = (AK_LDS3 unsigned char*)st_smem;
  const CcTask& t = tasks[blockIdx.x];
  const int kind = t.kind, bi = t.bi, bj = t.bj, g0 = t.g0, dp = t.dp, ge = min(g0 + CG_GROUP, t.nb);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31, wr = wave & 3, wc = wave >> 2;
  float* __restrict__ W = a.ws + t.w_off;
  float* __restrict__ E = a.ws + t.e_off;
  float* __restrict__ V = a.ws + t.v_off + static_cast<int64_t>(g0 / CG_GROUP & 1) * dp * CC_VLD;
  const float* __restrict__ M = a.ws + t.m_off + (k & 1) * ST_TILE;
  auto in_group = [&](int r, int i) { const int rr = r - g0; return E + (rr * (rr - 1) / 2 + i - g0) * ST_TILE; };
  auto at = [&](int r, int c) { return W + static_cast<int64_t>(LEAF) * r * dp + LEAF * c; };
  // Y_i: block (i, k), or block (k, i) transposed; the latter comes with the threads of a transposed operand
  auto fetch_y = [&](StPart& y, int i) {
    const int kcols = dp - LEAF * k;
    if (i > k) st_fetch(y, at(i, k), dp, dp - LEAF * i, kcols, tid);
    else if (i < g0) st_fetch_t(y, at(k, i), dp, kcols, tid);
    else st_fetch_t(y, in_group(k, i), LEAF, kcols, tid);
  };
  auto store_v = [&](const floatx16& v, int i) {
    const int row = LEAF * i + 32 * wr + l32;
    if (row >= dp) return;
    float* __restrict__ dst = V + static_cast<int64_t>(row) * CC_VLD + LEAF * (k - g0) + 32 * wc + 4 * g;
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<floatx4*>(dst + 8 * q) = floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
  };
  StPart m, y;
  auto stage_m = [&] {
    st_stash(m.v[0], lds, false, tid);
    st_stash(m.v[1], lds + ST_HALF, false, tid);
  };

  if (kind == CC_LEAF) {
    const int n = min(LEAF, dp - LEAF * bi);
    floatx16 upd, v;
    if (k >= 0) {
      st_fetch(m, M, LEAF, LEAF, LEAF, tid);
      st_fetch(y, at(bi, k), dp, dp - LEAF * bi, LEAF, tid);
    }
    st_leaf_fetch(upd, [&](int i, int j) { return *reinterpret_cast<const floatx4*>(at(bi, bi) + static_cast<int64_t>(i) * dp + j); }, n, tid);
    if (k >= 0) {
      stage_m();
      v = st_panel(y, false, lds, wr, wc, tid);
      store_v(v, bi);
    }
    float* __restrict__ Mn = a.ws + t.m_off + ((k + 1) & 1) * ST_TILE;
    // M^T is v_k of the block's own column, in the buffer of its own group
    const int gn = bi / CG_GROUP * CG_GROUP;
    float* __restrict__ Vn = a.ws + t.v_off + static_cast<int64_t>(gn / CG_GROUP & 1) * dp * CC_VLD + static_cast<int64_t>(LEAF) * bi * CC_VLD + LEAF * (bi - gn);
    const int bad = st_leaf(upd, [&](int i, int j, const floatx4& x) {
      const int c = lane & 15;
      if (i + c < n) *reinterpret_cast<floatx4*>(Vn + i * CC_VLD + j + static_cast<uint32_t>(c * CC_VLD + 4 * (lane >> 4))) = x;
    }, v, k >= 0, n, Mn, lds, sh, wr, wc, tid);
    if (tid == 0 && (a.skip == nullptr || a.skip[static_cast<int64_t>(t.mat) * a.skip_stride] != 0)) {
      const int where = bad != 0 && LEAF * bi + bad <= t.d ? LEAF * bi + bad : 0;
      if (where != 0 && a.info[t.mat] == 0) a.info[t.mat] = where;
    }
    return;
  }

  st_fetch(m, M, LEAF, LEAF, LEAF, tid);
  fetch_y(y, bi);
  stage_m();
  floatx16 vi = st_panel(y, bi < k, lds, wr, wc, tid), vj;
  if (kind == CC_PANEL) {
    store_v(vi, bi);
    return;
  }
  const bool diag = bi == bj, jk = bj == k;
  if (jk) {
    vj = st_own(M, tid);
  } else if (!diag) {
    fetch_y(y, bj);
    __syncthreads();
    vj = st_panel(y, bj < k, lds, wr, wc, tid);
  }
  // who stores v: the tiles of column and row k + 1
  if (bj == k + 1 && !diag) store_v(vi, bi);
  if (bi == k + 1 && bj < k) store_v(vj, bj);

  const bool inside = bj >= g0 && bj <= k;               // a row that follows, column of this group: in E
  float* __restrict__ X = inside ? in_group(bi, bj) : at(bi, bj);
  const int ld = inside ? LEAF : dp, rows = dp - LEAF * bi, cols = inside ? LEAF : dp - LEAF * bj;
  const int i0 = 32 * wr + 4 * g, j = 32 * wc + l32;     // element r of a wave's block: (i0 + 8 (r / 4) + r % 4, j)
  const uint32_t lane_at = static_cast<uint32_t>(i0 * ld + j);       // (a wave's rows differ by uniform offsets)
  const bool whole = inside || (rows >= LEAF && cols >= LEAF);
  floatx16 old;
#pragma unroll
  for (int r = 0; r < 16; ++r) old[r] = 0.f;
  if (!jk) {
    if (whole) {
#pragma unroll
      for (int r = 0; r < 16; ++r) old[r] = (X + (8 * (r >> 2) + (r & 3)) * ld)[lane_at];
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) old[r] = X[min(i0 + 8 * (r >> 2) + (r & 3), rows - 1) * ld + min(j, cols - 1)];
    }
  }
  const floatx16 sum = st_outer(vi, false, vj, jk, diag, lds, wr, wc, tid);
  if (whole) {
#pragma unroll
    for (int r = 0; r < 16; ++r) (X + (8 * (r >> 2) + (r & 3)) * ld)[lane_at] = old[r] - sum[r];
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int i = i0 + 8 * (r >> 2) + (r & 3);
      if (i < rows && j < cols) X[i * ld + j] = old[r] - sum[r];
    }
  }
}

}  // namespace ak
