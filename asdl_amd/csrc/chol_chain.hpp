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
// the tiles are products of a launch of their own.  At the end of the group every tile gets its update from V, 512 deep: at once what
// the steps of the next group read, its columns and rows and the diagonal block behind it, in a launch of products; the others beside
// those steps, in their launches, as long as these are not longer for it (cg_build_chain).  Work: d^3 in all, as in the sweep.
//
// W: the work matrix (lower triangle, row-major, dp columns), lam added by cg_copy_in_kernel.  Tiles (r, i) inside a group live in
// E from the step that makes them (i = k), because their place in W is column k, which the same launch reads.  M alternates
// between two buffers by k, V by the group (the steps of a group write one while the products of the group before read the other).
// V is kept as the two fp16 pieces of its scaled values, which every tile of the products would form again, where 22 bits do.
// Bound by the chain (25 to 30 us a step: the leaf 12, its v and update 9, its operands from a row-major matrix 3): with the products
// beside it, 2 x 4096 takes 33 steps of 25 to 33 us, 7 launches of 244 urgent tiles of 19 us each, and 77 us for the last 1056 (1.2 PFLOP/s of
// fp16 products would take 43).  All products in launches of their own, 80 us per 512 columns, pieces formed by every tile, and now: 2 x 4096
// 1720 -> 1250 us, 4096 1265 -> 1020, the 42 factors of ResNet-18 2975 -> 2640, 16 decoder factors of 768 ... 3073 1725 -> 1480,
// 12 x 1537 825 -> 745, 24 x 1100 665 -> 625, 8192 4080 -> 3410.
// Cross products on an accumulator of their own, and three bf16 pieces in the tiles of the steps, round less than one accumulator for all:
// error against 64 bits, full rank 5.5e-7 -> 4.5e-7, ReLU rows of rank d / 8 at a / lam = 2^12 4096 1.9e-2 -> 7e-3, 2048 8.8e-3 -> 4e-3.
#pragma once
#include "chol_step.hpp"
#include "syrk_dtl_tile.hpp"

namespace ak {

// What an operand of a product holds, for the fp16-piece products.  With
// a = the largest diagonal element of A + lam I, every element is bounded in magnitude: of the Cholesky factor L by sqrt(a),
// of M = L^-1 by 1 / sqrt(lam).
constexpr int CG_KIND_L = 1, CG_KIND_M = 2;
constexpr int CG_SCALE_FLOATS = 4;                    // per matrix: the fp16 switch, the scales of both kinds, padding
constexpr int CG_GROUP = 4;                           // block columns of a group
constexpr int CC_VLD = CG_GROUP * LEAF;
enum { CC_LEAF = 0, CC_TILE = 1, CC_PANEL = 2, CC_OWN = 3, CC_STEP = 4, CC_PRODUCT = 5 };

struct CcTask {
  int64_t w_off, v_off, e_off, m_off;        // floats from the workspace base; V: two of [dp][CC_VLD], E: six tiles, M: two
  int32_t mat, d, dp, nb;
  int32_t kind, bi, bj, g0;                  // g0: first block of the group of step k (CC_PRODUCT: of the group whose V it takes)
};

// V holds rows of fp32, or (scales[0] of the matrix) two fp16 pieces of the scaled values, by blocks of 16 columns: [32][dp rows][16 upper, 16
// lower ones], so that 16 rows of a block, what a wave brings into the LDS at once, are eight whole lines of memory.
struct CcArgs {
  float* ws;
  const int* skip;
  int* info;
  const float* scales;                       // CG_SCALE_FLOATS per matrix (cg_scale_kernel)
  const float* const* A_list;                // the matrices themselves: what the first group's products update
  const float* lam;
  int skip_stride, lam_stride;
};
// W holds of A + lam I what the first group's steps read: CC_VLD columns and the diagonal block behind them.
constexpr int CC_COPIED = CC_VLD + LEAF;     // rows that are copied beyond column CC_VLD

// (said of pointers that are chosen between or read from memory: else their accesses are flat ones)
#define CC_GLOBAL __attribute__((address_space(1)))

// X <- old -+ V_i V_j^T, one 128 x 128 tile over columns 64 h0 ... 64 h1 - 1 of V; rows, cols: of the tile inside the matrix.
struct CcProduct {
  const float* V;
  CC_GLOBAL float* X;
  CC_GLOBAL const float* old;                // of old_rows x old_cols, rows old_ld apart; beyond it zeros and `pad` on the diagonal
  int dp, bi, bj, ld, rows, cols, h0, h1, old_ld, old_rows, old_cols;
  float alpha, lam, pad;                     // lam is added to the old diagonal
  bool half, same, anew;                     // V on fp16 pieces; one operand; no old value
};

constexpr int CC_BLOCK = 16;                 // columns of a block of V on fp16 pieces
constexpr int CC_PANEL_BYTES = LEAF * 64;    // a block's 128 rows of one operand
// Elements (row, 16 b + ...) of V on fp16 pieces, in bytes from its start; dp below 2^15: 32 bits.
__host__ __device__ __forceinline__ uint32_t cc_v_at(int dp, int row, int b) {
  return (static_cast<uint32_t>(b) * static_cast<uint32_t>(dp) + static_cast<uint32_t>(row)) * 64u;
}
__device__ __forceinline__ u32x4 cc_descriptor(CC_GLOBAL const void* at) {
  const uint64_t b = reinterpret_cast<uint64_t>(at);
  u32x4 d;
  d[0] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b));
  d[1] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b >> 32) & 0xffffu);
  d[2] = kDtlRange;
  d[3] = 0x00020000u;
  return d;
}
// Byte offset in V of what a lane loads of rows 16 part ... + 15 of operand block `blk` (rows beyond the matrix: its last one).  16-byte
// chunks (two of upper, two of lower pieces) are permuted inside a row by row / 4, in the LDS: reads of 32 rows without conflicts.
__device__ __forceinline__ uint32_t cc_lane_at(int dp, int blk, int rows, int part, int lane) {
  const int row = 16 * part + (lane >> 2), chunk = (lane & 3) ^ ((row >> 2) & 3);
  return cc_v_at(dp, LEAF * blk + min(row, rows - 1), 0) + 16u * chunk;
}
struct CcFragments { bf16x8 x[2]; };         // the two pieces (fp16 patterns) of 32 rows
__device__ __forceinline__ CcFragments cc_read(AK_LDS3 const unsigned char* panel, int row, int g) {
  const int swap = (row >> 2) & 3;
  CcFragments f;
#pragma unroll
  for (int q = 0; q < 2; ++q) f.x[q] = *reinterpret_cast<AK_LDS3 const bf16x8*>(panel + row * 64 + 16 * ((2 * q + g) ^ swap));
  return f;
}

// A wave's 32 x 32 block at (r0, c0) of the tile.  (Whole tiles: a wave's rows differ by uniform offsets, one 32-bit offset per lane.)
__device__ __forceinline__ void cc_update(const CcProduct& p, const floatx16& sum, int r0, int c0, int lane) {
  const int i0 = r0 + 4 * (lane >> 5), j = c0 + (lane & 31);
  floatx16 old;
  if (p.old_rows >= LEAF && p.old_cols >= LEAF && !(p.same && p.lam != 0.f)) {        // (the tile has no less)
    CC_GLOBAL float* X = p.X;                // (behind the first group the old values lie in X itself)
    CC_GLOBAL const float* Y = p.old;
    const int ld = p.ld, old_ld = p.old_ld;
    const uint32_t at = static_cast<uint32_t>(i0 * ld + j), from = static_cast<uint32_t>(i0 * old_ld + j);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      old[e] = 0.f;
      if (!p.anew) old[e] = (Y + (8 * (e >> 2) + (e & 3)) * old_ld)[from];
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) (X + (8 * (e >> 2) + (e & 3)) * ld)[at] = old[e] + p.alpha * sum[e];
    return;
  }
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int i = i0 + 8 * (e >> 2) + (e & 3);
    old[e] = 0.f;
    if (!p.anew) {
      const float x = p.old[static_cast<uint32_t>(min(i, p.old_rows - 1) * p.old_ld + min(j, p.old_cols - 1))];
      const bool diagonal = p.same && i == j;
      old[e] = i < p.old_rows && j < p.old_cols ? x + (diagonal ? p.lam : 0.f) : diagonal ? p.pad : 0.f;
    }
  }
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int i = i0 + 8 * (e >> 2) + (e & 3);
    if (i < p.rows && j < p.cols) p.X[static_cast<uint32_t>(i * p.ld + j)] = old[e] + p.alpha * sum[e];
  }
}

// V on fp16 pieces, by the 16 waves of a step's work group: the operands go from memory straight to the LDS, a stage of 32 k ahead of
// three others.  Three matrix instructions per product, the cross products on an accumulator of their own.
__device__ __forceinline__ floatx16 cc_sum_half(const CcProduct& p, AK_LDS3 unsigned char* lds, int tid) {
  constexpr int OPERAND = 2 * CC_PANEL_BYTES, STAGE = 2 * OPERAND, STAGES = 4;
  static_assert(STAGES * STAGE + 16384 <= ST_LDS, "stages");
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, l32 = lane & 31, wr = wave & 3, wc = wave >> 2;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
  const u32x4 d = cc_descriptor((CC_GLOBAL const void*)p.V);
  // a wave brings 16 rows of one block of 16 k of either operand
  const int blk = wave >> 3, part = wave & 7;
  const uint32_t oi = cc_lane_at(p.dp, p.bi, p.rows, part, lane), oj = cc_lane_at(p.dp, p.bj, p.cols, part, lane);
  const uint32_t to = lds0 + blk * CC_PANEL_BYTES + part * 1024;
  const int s0 = 2 * p.h0, s1 = 2 * p.h1;
  auto issue = [&](int s) {
    const uint32_t at = to + (s & (STAGES - 1)) * STAGE, block = cc_v_at(p.dp, 0, 2 * s + blk);
    load_to_lds(d, at, oi + block);
    if (!p.same) load_to_lds(d, at + OPERAND, oj + block);
  };
  StSum sum;
  sum.clear();
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
    if (s0 + t < s1) issue(s0 + t);
  // The old tile, if there is one, a word of every 64 bytes: on its way to the L2 while the last stages run (their registers leave no room
  // for it; ahead of the first stages it would hold those up).  The spare LDS takes what comes.  (Its descriptor is formed here, in the loop.)
  auto touch = [&] {
    const uint32_t i = min(tid >> 3, p.old_rows - 1), j = min(16 * (tid & 7), p.old_cols - 4);
    load_to_lds<true>(cc_descriptor(p.old), lds0 + STAGES * STAGE + wave * 1024, p.anew || p.old_cols < 4 ? kDtlOob : (i * p.old_ld + j) * 4);
  };
  if (s1 - s0 < STAGES - 1) touch();
  struct Operands { CcFragments a, b; };
  auto read = [&](Operands& f, int s, int t) {
    AK_LDS3 const unsigned char* at = lds + (s & (STAGES - 1)) * STAGE + t * CC_PANEL_BYTES;
    f.a = cc_read(at, 32 * wr + l32, g);
    f.b = cc_read(p.same ? at : at + OPERAND, 32 * wc + l32, g);
  };
  auto multiply = [&](const Operands& f) {
    sum.small = x3_mfma<true>(f.a.x[1], f.b.x[0], sum.small);
    sum.big = x3_mfma<true>(f.a.x[0], f.b.x[0], sum.big);
    sum.small = x3_mfma<true>(f.a.x[0], f.b.x[1], sum.small);
  };
  Operands first, second;
  for (int s = s0; s < s1; ++s) {
    // stage s has landed for this wave, then for all; and all have read stage s - 1, which the next loads overwrite
    const int ahead = min(s1 - 1 - s, STAGES - 2);
    if (ahead == 2) {
      if (p.same) wait_vmcnt<2>();
      else wait_vmcnt<4>();
    } else if (ahead == 1) {
      if (p.same) wait_vmcnt<2>();           // (and the old tile's)
      else wait_vmcnt<3>();
    } else {
      wait_vmcnt<1>();
    }
    __syncthreads();
    if (s + STAGES - 1 < s1) issue(s + STAGES - 1);
    if (s + STAGES - 1 == s1) touch();
    read(first, s, 0);
    if (s > s0) multiply(second);
    read(second, s, 1);
    multiply(first);
  }
  multiply(second);
  wait_vmcnt<0>();                           // (the old tile's words, before the LDS is released)
  return sum.value();
}

// V in fp32 (a / lam beyond what 22 bits serve): three bf16 pieces, formed on the way to the LDS.
__device__ __forceinline__ floatx16 cc_sum_full(const CcProduct& p, AK_LDS3 unsigned char* lds, int wr, int wc, int tid) {
  const int lane = tid & 63;
  StPart a, b;
  StSum s;
  auto fetch = [&](int h) {                  // (halves beyond the last one are not used)
    st_fetch(a, p.V + static_cast<int64_t>(LEAF) * p.bi * CC_VLD + 64 * h, CC_VLD, p.rows, CC_VLD - 64 * h, tid);
    if (!p.same) st_fetch(b, p.V + static_cast<int64_t>(LEAF) * p.bj * CC_VLD + 64 * h, CC_VLD, p.cols, CC_VLD - 64 * h, tid);
  };
  s.clear();
  for (int h = p.h0; h < p.h1; h += 2) {
    fetch(h);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      __syncthreads();
      st_stash(a.v[u], lds, false, tid);
      if (!p.same) st_stash(b.v[u], lds + ST_HALF, false, tid);
      __syncthreads();
      if (h + u < p.h1) st_mma<4>(s, lds, 32 * wr, p.same ? lds : lds + ST_HALF, 32 * wc, lane);
    }
  }
  return s.value();
}

__device__ __forceinline__ void cc_product(const CcProduct& p, AK_LDS3 unsigned char* lds, int wr, int wc, int tid) {
  const floatx16 sum = p.half ? cc_sum_half(p, lds, tid) : cc_sum_full(p, lds, wr, wc, tid);
  cc_update(p, sum, 32 * wr, 32 * wc, tid & 63);
}

// CC_STEP: a tile of step k, whose launch formed V alone; CC_PRODUCT: a tile of the products of the group, whose own rows and columns are
// formed anew, from their own column on.
__device__ __forceinline__ CcProduct cc_task_product(const CcArgs& a, const CcTask& t, int k) {
  const int g0 = t.g0, bi = t.bi, bj = t.bj, dp = t.dp, ge = min(g0 + CG_GROUP, t.nb);
  const bool step = t.kind == CC_STEP, own_row = bi >= g0 && bi < ge, own_col = bj >= g0 && bj < ge;
  const int last = step ? k : ge - 1, from = step ? k - g0 : max(own_row ? bi - g0 : 0, own_col ? bj - g0 : 0);
  const int width = min(CC_VLD, dp - LEAF * g0), rr = bi - g0;
  const bool inside = step && bj >= g0 && bj <= k;
  const float* __restrict__ scales = a.scales + static_cast<int64_t>(t.mat) * CG_SCALE_FLOATS;
  CcProduct p;
  p.V = a.ws + t.v_off + static_cast<int64_t>(g0 / CG_GROUP & 1) * dp * CC_VLD;
  p.X = (CC_GLOBAL float*)(inside ? a.ws + t.e_off + (rr * (rr - 1) / 2 + bj - g0) * ST_TILE : a.ws + t.w_off + static_cast<int64_t>(LEAF) * bi * dp + LEAF * bj);
  p.dp = dp; p.bi = bi; p.bj = bj;
  p.ld = inside ? LEAF : dp;
  p.rows = min(LEAF, dp - LEAF * bi);
  p.cols = min(LEAF, dp - LEAF * bj);
  p.h0 = 2 * from;
  p.h1 = (width + 63) / 64;
  if (step) p.h1 = min(p.h1, p.h0 + 2);
  p.half = scales[0] != 0.f;
  p.same = bi == bj;
  p.anew = step ? bj == k : own_row || own_col;
  p.old = p.X; p.old_ld = p.ld; p.old_rows = p.rows; p.old_cols = p.cols;
  p.lam = p.pad = 0.f;
  if (!step && g0 == 0 && !p.anew) {         // never written before
    const int d = t.d;
    p.old = (CC_GLOBAL const float*)a.A_list[t.mat] + static_cast<int64_t>(LEAF) * bi * d + LEAF * bj;
    p.old_ld = d;
    p.old_rows = min(LEAF, d - LEAF * bi);
    p.old_cols = min(LEAF, d - LEAF * bj);
    p.lam = a.lam[static_cast<int64_t>(t.mat) * a.lam_stride];
    p.pad = p.lam > 0.f ? p.lam : 1.f;
  }
  p.alpha = bi > last ? -1.f : 1.f;
  if (p.half) p.alpha /= scales[bi > last ? CG_KIND_L : CG_KIND_M] * scales[bj > last ? CG_KIND_L : CG_KIND_M];        // (powers of two)
  return p;
}

// Step k (-1: the first diagonal blocks are factored), or products in a launch of their own; one work group per task.
// (Products of 8 waves, two work groups a CU, 1056 tiles in 66 us: 2 x 4096 1250 us as here, ResNet-18's factors 2520, here 2660, ResNet-50's
// 3350, here 3570.  They left half a CU to other kernels' waves: hold_cu.)
static __global__ __launch_bounds__(LEAF_THREADS) void cg_chain_kernel(CcArgs a, const CcTask* __restrict__ tasks, int k) {
  hold_cu();
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
  const float* __restrict__ scales = a.scales + static_cast<int64_t>(t.mat) * CG_SCALE_FLOATS;
  const bool half = scales[0] != 0.f;
  const float scale_l = scales[CG_KIND_L], scale_m = scales[CG_KIND_M];
  // values (row, c ... c + 3) of V
  auto put_v = [&](int row, int c, floatx4 x, float scale) {
    if (half) {
      typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
      typedef float f32x4 __attribute__((ext_vector_type(4)));
      f32x4 y = {x[0], x[1], x[2], x[3]};
      y *= scale;
      const f16x4 hi = __builtin_convertvector(y, f16x4);
      const f16x4 lo = __builtin_convertvector(y - __builtin_convertvector(hi, f32x4), f16x4);
      unsigned char* __restrict__ to = reinterpret_cast<unsigned char*>(V) + (cc_v_at(dp, row, c >> 4) + 2u * (c & 15));
      *reinterpret_cast<f16x4*>(to) = hi;
      *reinterpret_cast<f16x4*>(to + 32) = lo;
    } else {
      *reinterpret_cast<floatx4*>(V + static_cast<int64_t>(row) * CC_VLD + c) = x;
    }
  };
  auto store_v = [&](const floatx16& v, int i) {
    const int row = LEAF * i + 32 * wr + l32;
    if (row >= dp) return;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      put_v(row, LEAF * (k - g0) + 32 * wc + 4 * g + 8 * q, floatx4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]}, i > k ? scale_l : scale_m);
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
    const int bad = st_leaf(upd, [](int, int, const floatx4&) {}, v, k >= 0, n, Mn, lds, sh, wr, wc, tid);
    if (tid == 0 && (a.skip == nullptr || a.skip[static_cast<int64_t>(t.mat) * a.skip_stride] != 0)) {
      const int where = bad != 0 && LEAF * bi + bad <= t.d ? LEAF * bi + bad : 0;
      if (where != 0 && a.info[t.mat] == 0) a.info[t.mat] = where;
    }
    return;
  }

  if (kind == CC_OWN) {
    // M^T is v_k of the step's own column
    st_fetch_t(m, M, LEAF, LEAF, tid);
    const int row = LEAF * k + (tid & 127);
    if (row >= dp) return;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      put_v(row, LEAF * (k - g0) + 64 * (q >> 1) + 8 * (tid >> 7) + 4 * (q & 1),
            floatx4{m.v[q >> 1][4 * (q & 1)], m.v[q >> 1][4 * (q & 1) + 1], m.v[q >> 1][4 * (q & 1) + 2], m.v[q >> 1][4 * (q & 1) + 3]}, scale_m);
    return;
  }
  if (kind == CC_STEP || kind == CC_PRODUCT) {
    cc_product(cc_task_product(a, t, k), lds, wr, wc, tid);
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
