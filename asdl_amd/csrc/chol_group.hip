// out_m <- (A_m + lam_m I)^-1 for many symmetric positive definite fp32 matrices of DIFFERENT sizes in one call.
//
// A block elimination on Cholesky factors of 128 x 128 diagonal blocks that advances factorization, triangular inverse and
// L^-T L^-1 together (d^3 FLOP, as POTRF + POTRI), in one of two forms:
//   chol_sweep.hpp   every step updates the whole triangle: one launch per 128 columns, for groups whose tiles fit the device
//   chol_chain.hpp   the steps update the block columns that the next steps need, one product per 512 columns the rest
// The plan takes the chain where it saves enough (cg_build).  Explicit inverses are taken of 128 x 128 diagonal blocks only, so a panel is
// as accurate as a triangular solve with a block of that size (measured against fp64 on rank-deficient factors: the sweep at 0.8 to 0.9,
// the chain at 1.4 to 1.7 times the error of LAPACK's fp32 potrf + potri; a recursion that multiplied by the inverse of a whole half
// was at 3 to 8 times that).
//
// The steps of all matrices are merged: step k of the chain is one launch for all matrices that have a block k, and so are the products
// that are due at the end of a group; products that are not due yet go along with the steps.
//
// The plan (descriptor tables, launch sequence) depends on the sizes only; every address in it is an offset into the
// workspace.  The caller builds it once per size set on the host (ak_chol_group_plan), keeps a device copy, and
// passes both to every call.
//
// Matrices are padded to a multiple of 4 columns with an identity block (the padded rows and columns drop out of the
// result), which keeps every operand 16-byte aligned.  Only the lower triangle of the input is
// read; the strictly upper 128-blocks of W are never touched.
#include <algorithm>
#include <cstring>
#include <utility>
#include <vector>
#include "gemm_f32.hpp"
#include "chol_sweep.hpp"
#include "chol_chain.hpp"

namespace ak {

constexpr int64_t CG_MAGIC = 0x3647524c4f4843ll;     // "CHOLGR6"
constexpr int CG_COPY = 0, CG_CHAIN = 1, CG_SWEEP = 2, CG_OUT = 3;

#ifdef AK_TUNING_HOOKS
static float CG_HALF_MAX_COND = 65536.f;              // tuning builds: ak_debug_set_chol_half_max_cond
#else
constexpr float CG_HALF_MAX_COND = 65536.f;           // a / lam beyond 2^16: the matrix keeps the bf16 three-piece products
#endif
constexpr int CG_COPY_ROWS = 8;                       // rows of W one work group of the copy-in kernel writes

struct CgHeader {
  int64_t magic;
  int64_t total_bytes;
  int64_t ws_floats;
  int64_t scales_off;       // floats from the workspace base: CG_SCALE_FLOATS per matrix
  int64_t mats_off, steps_off, tasks_off, tiles_off;      // byte offsets of the tables inside the plan (tiles: of the sweep)
  int32_t count, nsteps, copy_blocks, out_blocks;
  double us;                // estimated time of one call (cg_build)
};

struct CgMat {
  int64_t w_off;            // work matrix [dp, dp], offset in floats from the workspace base
  int32_t d, dp;
  int32_t first_copy_block, first_out_block;
};

struct CgStep {
  int32_t type, first, count, grid;    // chain: first task, step k, tasks
};

struct CgArgs {
  const unsigned char* plan;        // device copy of the plan
  float* ws;
  const float* const* A_list;
  float* const* out_list;
  const float* lam;
  const int* skip;
  int* info;
  int lam_stride, skip_stride;
  float* scales;                    // ws + scales_off
};

__device__ __forceinline__ bool cg_skipped(const CgArgs& a, int mat) {
  return a.skip != nullptr && a.skip[static_cast<int64_t>(mat) * a.skip_stride] == 0;
}

// W_m <- what the chain's first group of lower(A_m) + lam_m I reads before its products, which take the rest from A_m itself
// (cc_task_product); padded rows carry the identity; info_m <- 0.  One work group per CG_COPY_ROWS rows of one matrix (bisection on
// first_copy_block); a row is read and written up to its diagonal element at most.  Bound by the memory: two matrices of 4096 columns 15 us,
// where all of them took 40 (the whole of ResNet-18's 42 factors took 120 us less, a decoder's 65, 8192 130).
static __global__ __launch_bounds__(256) void cg_copy_in_kernel(CgArgs a, int count) {
  const CgHeader* __restrict__ h = reinterpret_cast<const CgHeader*>(a.plan);
  const CgMat* __restrict__ mats = reinterpret_cast<const CgMat*>(a.plan + h->mats_off);
  const int w = blockIdx.x;
  int lo = 0, hi = count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (mats[mid].first_copy_block <= w) lo = mid;
    else hi = mid - 1;
  }
  const CgMat m = mats[lo];
  if (cg_skipped(a, lo)) return;
  const int r0 = (w - m.first_copy_block) * CG_COPY_ROWS;
  if (r0 == 0 && threadIdx.x == 0) a.info[lo] = 0;
  const float* __restrict__ A = a.A_list[lo];
  float* __restrict__ W = a.ws + m.w_off;
  const float l = a.lam[static_cast<int64_t>(lo) * a.lam_stride];
  const bool vec = (m.d % 4 == 0) && ((reinterpret_cast<uintptr_t>(A) & 15) == 0);
#pragma unroll 1
  for (int e = 0; e < CG_COPY_ROWS; ++e) {
    const int r = r0 + e;
    if (r >= m.dp) break;
    float* __restrict__ dst = W + static_cast<int64_t>(r) * m.dp;
    const int last = r < CC_COPIED ? r : CC_VLD - 1;
    if (r >= m.d) {
      // padding: a diagonal block that drops out of the result.  Its value lam (1 when lam <= 0) stays inside the
      // magnitude bounds the fp16-piece products scale their operands by (lam <= a, 1 / sqrt(lam) for the inverse).
      const float pad = l > 0.f ? l : 1.f;
      for (int c = threadIdx.x; c <= last; c += 256) dst[c] = (c == r) ? pad : 0.f;
      continue;
    }
    const float* __restrict__ src = A + static_cast<int64_t>(r) * m.d;
    if (vec) {
      for (int c = 4 * threadIdx.x; c <= last; c += 1024) {
        floatx4 v = *reinterpret_cast<const floatx4*>(src + c);
        if (r >= c && r < c + 4) v[r - c] += l;
        *reinterpret_cast<floatx4*>(dst + c) = v;       // the elements right of the diagonal are never read
      }
    } else {
      for (int c = threadIdx.x; c <= last; c += 256) dst[c] = src[c] + ((c == r) ? l : 0.f);
    }
  }
}

// Per matrix: the powers of two that bring each kind of operand into the range of fp16 (largest possible magnitude
// -> (2^13, 2^14]), from a = max_i (A_ii + lam) and lam; and whether the matrix takes the fp16-piece products at
// all: a > 0, lam > 0 and a / lam <= 2^16 (elements that are much smaller than their kind's bound lose relative, not
// absolute accuracy; within that ratio the elements that matter keep 22 bits, and the condition number, at most d a / lam,
// leaves the two bits the fp16 pieces have less than fp32 to spare before the factorization breaks down).  One work group
// per matrix.
static __global__ __launch_bounds__(256) void cg_scale_kernel(CgArgs a, int count, float max_cond) {
  __shared__ float red[4];
  const int m = blockIdx.x;
  const CgHeader* __restrict__ h = reinterpret_cast<const CgHeader*>(a.plan);
  const CgMat cm = reinterpret_cast<const CgMat*>(a.plan + h->mats_off)[m];
  float* __restrict__ sc = a.scales + static_cast<int64_t>(m) * CG_SCALE_FLOATS;
  float amax = -3.0e38f;
  const bool live = !cg_skipped(a, m);
  if (live) {
    const float* __restrict__ A = a.A_list[m];
    for (int i = threadIdx.x; i < cm.d; i += 256) amax = fmaxf(amax, A[static_cast<int64_t>(i) * cm.d + i]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = amax;
  __syncthreads();
  if (threadIdx.x != 0) return;
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float lam = live ? a.lam[static_cast<int64_t>(m) * a.lam_stride] : 0.f;
  amax += lam;
  const bool half = live && lam > 0.f && amax > 0.f && amax < 3.0e38f && amax <= max_cond * lam;
  auto scale = [&](float bound) {
    int e;
    frexpf(bound, &e);                   // bound <= 2^e
    return half ? ldexpf(1.f, 14 - e) : 1.f;
  };
  sc[0] = half ? 1.f : 0.f;
  sc[CG_KIND_L] = scale(sqrtf(amax));
  sc[CG_KIND_M] = scale(1.f / sqrtf(lam));
}

// out_m <- both triangles of W_m, one work group per 64 x 64 tile of its lower triangle (bisection on first_out_block).
static __global__ __launch_bounds__(256) void cg_out_kernel(CgArgs a, int count) {
  __shared__ float tile[64][65];
  const CgHeader* __restrict__ h = reinterpret_cast<const CgHeader*>(a.plan);
  const CgMat* __restrict__ mats = reinterpret_cast<const CgMat*>(a.plan + h->mats_off);
  const int w = blockIdx.x;
  int lo = 0, hi = count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (mats[mid].first_out_block <= w) lo = mid;
    else hi = mid - 1;
  }
  const CgMat m = mats[lo];
  if (cg_skipped(a, lo)) return;
  int ti, tj;
  decode_lower_tile(w - m.first_out_block, ti, tj);
  const float* __restrict__ W = a.ws + m.w_off;
  float* __restrict__ out = a.out_list[lo];
  const int c = 4 * (threadIdx.x & 15), r0 = threadIdx.x >> 4;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int r = r0 + 16 * u, i = 64 * ti + r, j = 64 * tj + c;
    const floatx4 v = *reinterpret_cast<const floatx4*>(W + static_cast<int64_t>(min(i, m.dp - 1)) * m.dp + min(j, m.dp - 4));
#pragma unroll
    for (int e = 0; e < 4; ++e) tile[r][c + e] = v[e];
  }
  __syncthreads();
  const int x = threadIdx.x & 63, y0 = threadIdx.x >> 6;
#pragma unroll 4
  for (int u = 0; u < 16; ++u) {
    const int y = y0 + 4 * u;
    const bool upper = ti == tj && x > y;              // of a diagonal tile: the mirror image
    const int i = 64 * ti + y, j = 64 * tj + x;
    if (i < m.d && j < m.d) out[static_cast<int64_t>(i) * m.d + j] = upper ? tile[x][y] : tile[y][x];
    const int mi = 64 * tj + y, mj = 64 * ti + x;
    if (ti != tj && mj < m.d) out[static_cast<int64_t>(mi) * m.d + mj] = tile[x][y];
  }
}

// ---- host: the plan ------------------------------------------------------------------------------------------

static inline int64_t cg_align64(int64_t x) { return (x + 63) / 64 * 64; }

// Products in launches of their own, on 128 x 128 tiles of split operands or on deep fp32 tiles of 64 x 64: what the rule between sweep and
// chain was measured with (cg_build).
struct CgShape {
  int64_t tiles, deep_tiles, K;
};
static void cg_add_shape(std::vector<CgShape>& ps, int64_t M, int64_t N, int64_t K, bool lower) {
  if (M <= 0 || N <= 0) return;
  const int64_t m = (M + 127) / 128, n = (N + 127) / 128, dm = (M + 63) / 64, dn = (N + 63) / 64;
  ps.push_back(lower ? CgShape{m * (m + 1) / 2, dm * (dm + 1) / 2, K} : CgShape{m * n, dm * dn, K});
}
// Microseconds of one launch: as long as its longest tile, or as its work spread over the CUs.
static double cg_shapes_us(const std::vector<CgShape>& ps) {
  if (ps.empty()) return 0.0;
  double longest = 0, sum = 0, deep_longest = 0, deep_sum = 0;
  for (const CgShape& p : ps) {
    const double c = static_cast<double>((p.K + 31) / 32), d = static_cast<double>((p.K + 127) / 128);
    longest = std::max(longest, c);
    sum += c * static_cast<double>(p.tiles);
    deep_longest = std::max(deep_longest, d);
    deep_sum += d * static_cast<double>(p.deep_tiles);
  }
  return 4 + std::min(2.0 * std::max(deep_longest, deep_sum / 256), std::max(1.6 * longest, 1.05 * sum / 256));
}
// Of the products at the end of the group of columns [c0, c1) of one matrix; of the tiles of step k.
static void cg_group_shapes(std::vector<CgShape>& ps, int64_t dp, int64_t c0, int64_t c1) {
  const int64_t width = c1 - c0, below = dp - c1;
  cg_add_shape(ps, below, below, width, true);
  cg_add_shape(ps, below, width, width, false);
  cg_add_shape(ps, below, c0, width, false);
  cg_add_shape(ps, width, c0, width, false);
  cg_add_shape(ps, width, width, width, true);
  cg_add_shape(ps, c0, c0, width, true);
}
static void cg_step_shapes(std::vector<CgShape>& ps, int64_t dp, int k, int g0, int ge) {
  const int64_t c0 = static_cast<int64_t>(g0) * LEAF, c1 = static_cast<int64_t>(k + 1) * LEAF, c2 = std::min<int64_t>(static_cast<int64_t>(ge) * LEAF, dp);
  const int64_t next = std::min<int64_t>(LEAF, dp - c2);
  cg_add_shape(ps, c2 - c1, c2 - c1, LEAF, true);
  cg_add_shape(ps, dp - c2, c2 - c1, LEAF, false);
  cg_add_shape(ps, next, next, LEAF, true);
  cg_add_shape(ps, c2 - c1, c0, LEAF, false);
  for (int r = k + 1; r < ge; ++r)
    for (int i = g0; i <= k; ++i) cg_add_shape(ps, std::min<int64_t>(LEAF, dp - static_cast<int64_t>(r) * LEAF), LEAF, LEAF, false);
}

struct CgPlan {
  CgHeader h;
  std::vector<CgMat> mats;
  std::vector<CgStep> steps;
  std::vector<CcTask> tasks;
  std::vector<SwTask> sweep_leaves, sweep_tiles;
};

static inline int64_t cg_align(int64_t x, int64_t a) { return (x + a - 1) / a * a; }

static bool cg_dims_ok(const int64_t* dims, int count) {
  if (dims == nullptr || count <= 0 || count > (1 << 20)) return false;
  for (int i = 0; i < count; ++i)
    if (dims[i] <= 0 || dims[i] > 32768) return false;
  return true;
}

// The sweep: per step the leaf's work group, or the rounds of tiles that the device needs (one work group per CU); rounds: of all
// steps, of which so many are filled.  Estimated and measured, us: 3072 864 and 868, 6 x 1700 811 and 800, 20 x 1142 712 and 710, 64 x 630 412 and 438,
// 4 x 2400 with 8 x 512 1216 and 1230.
static double cg_sweep_us(const int64_t* dims, int count, int64_t& rounds, double& filled) {
  int64_t nb_max = 0, all = 0;
  for (int m = 0; m < count; ++m) nb_max = std::max<int64_t>(nb_max, (dims[m] + LEAF - 1) / LEAF);
  double us = 14;
  rounds = 0;
  for (int64_t k = 0; k < nb_max; ++k) {
    int64_t groups = 0;
    for (int m = 0; m < count; ++m) {
      const int64_t nb = (dims[m] + LEAF - 1) / LEAF;
      if (nb > k) groups += nb * (nb + 1) / 2 + (nb > k + 1 ? 1 : 0);
    }
    const int64_t r = (groups + 255) / 256;
    us += std::max(22.0, 14.0 * static_cast<double>(r) + 6.0 * static_cast<double>(groups) / 256);
    rounds += r;
    all += groups;
  }
  filled = static_cast<double>(all) / 256;
  return us;
}

// The tables of the sweep: matrices in the order of their number of block columns, so that those still at work in step k
// are the first ones of both lists.
static void cg_build_sweep(const int64_t* dims, int count, CgPlan& plan) {
  std::vector<int> order(count);
  for (int m = 0; m < count; ++m) order[m] = m;
  auto blocks = [&](int m) { return static_cast<int>((dims[m] + LEAF - 1) / LEAF); };
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return blocks(x) > blocks(y); });
  int64_t off = 0;
  for (int m : order) {
    const int nb = blocks(m);
    SwTask t;
    std::memset(&t, 0, sizeof(t));
    t.mat = m; t.d = static_cast<int>(dims[m]); t.nb = nb;
    t.x_off = off;
    t.y_off = off + static_cast<int64_t>(nb) * (nb + 1) / 2 * SW_TILE;
    t.m_off = t.y_off + static_cast<int64_t>(2) * nb * SW_TILE;
    off = t.m_off + 2 * SW_TILE;
    plan.sweep_leaves.push_back(t);
    const int64_t x0 = t.x_off;
    for (t.bi = 0; t.bi < nb; ++t.bi)
      for (t.bj = 0; t.bj <= t.bi; ++t.bj) {
        t.x_off = x0 + (static_cast<int64_t>(t.bi) * (t.bi + 1) / 2 + t.bj) * SW_TILE;
        plan.sweep_tiles.push_back(t);
      }
  }
  const int nb_max = blocks(order[0]);
  for (int k = -1; k < nb_max; ++k) {
    int leaves = 0, tiles = 0;
    for (int m : order) {
      if (blocks(m) > k + 1) ++leaves;
      if (k >= 0 && blocks(m) > k) tiles += blocks(m) * (blocks(m) + 1) / 2;
    }
    plan.steps.push_back(CgStep{CG_SWEEP, k, leaves, leaves + tiles});
  }
  CgHeader& h = plan.h;
  std::memset(&h, 0, sizeof(h));
  h.magic = CG_MAGIC;
  h.ws_floats = off;
  h.count = count;
  h.nsteps = static_cast<int>(plan.steps.size());
  int64_t b = cg_align(sizeof(CgHeader), 64);
  h.steps_off = b; b = cg_align(b + plan.steps.size() * sizeof(CgStep), 64);
  h.tasks_off = b; b = cg_align(b + plan.sweep_leaves.size() * sizeof(SwTask), 64);
  h.tiles_off = b; b = cg_align(b + plan.sweep_tiles.size() * sizeof(SwTask), 64);
  h.mats_off = b;
  h.total_bytes = b;
}

#ifdef AK_TUNING_HOOKS
static int CG_FORCE = 0;               // tuning builds: 1 the sweep, 2 the chain, 3 (4) with (without) launches of their own for its tiles
#else
constexpr int CG_FORCE = 0;
#endif

// The tiles of a lower triangle along a Z curve: neighbours in the list read the same rows of V.
static std::vector<std::pair<int, int>> cg_blocked_tiles(int nb) {
  std::vector<std::pair<int, int>> tiles;
  int side = 1;
  while (side < nb) side *= 2;
  for (int64_t z = 0; z < static_cast<int64_t>(side) * side; ++z) {
    int bi = 0, bj = 0;
    for (int bit = 0; (1 << bit) < side; ++bit) {
      bj |= static_cast<int>(z >> (2 * bit) & 1) << bit;
      bi |= static_cast<int>(z >> (2 * bit + 1) & 1) << bit;
    }
    if (bi < nb && bj <= bi) tiles.emplace_back(bi, bj);
  }
  return tiles;
}
// Appends a list to the tasks of the launch that starts at task `first` so that every XCD (work group number modulo 8) gets a
// contiguous eighth of it, whose rows of V its L2 then holds (the 42 factors of ResNet-18 took 175 us less).
static void cg_append_by_xcd(std::vector<CcTask>& tasks, int first, const std::vector<CcTask>& list) {
  const size_t n = list.size(), base = tasks.size() - static_cast<size_t>(first);
  size_t next[8], at = 0;
  for (size_t x = 0; x < 8; ++x) {
    next[x] = at;
    at += (n + 7 - (x + 8 - base % 8) % 8) / 8;          // places of the list on this XCD
  }
  for (size_t i = 0; i < n; ++i) {
    const size_t x = (base + i) % 8;
    tasks.push_back(list[next[x]++]);
  }
}

constexpr size_t kProductChunk = 16;   // tiles that stay together
// us of a CU: a tile of a group's products, a tile of a step in a launch of its own;
// what a step's launch takes along without being longer for it: its leaf takes 26.  (Tiles beyond that in the steps' launches, each of which
// asks for a whole CU: 24 x 1100 605 -> 625 us, ResNet-18's step, beside the loss backward pass, 1 % more.)
constexpr double kProductUs = 18.0, kStepUs = 5.0, kBesideUs = 26.0;
// The chain's tables.  Returns the time that the rule goes by: 26 us a step, or 9 and 18 per round of tiles (of panels alone: 9) where that is
// more, all products in launches of their own (cg_shapes_us), the copies by their bytes.
static double cg_build_chain(const int64_t* dims, int count, CgPlan& plan) {
  struct Mat { int64_t w, v, e, m; int d, dp, nb; };
  std::vector<Mat> mats(count);
  int64_t off = 0;
  int copy_blocks = 0, out_blocks = 0, nb_max = 0;
  double bytes = 0;
  plan.mats.resize(count);
  for (int i = 0; i < count; ++i) {
    Mat& x = mats[i];
    x.d = static_cast<int>(dims[i]);
    x.dp = (x.d + 3) / 4 * 4;
    x.nb = (x.dp + LEAF - 1) / LEAF;
    nb_max = std::max(nb_max, x.nb);
    auto take = [&](int64_t floats) { const int64_t at = off; off += cg_align64(floats); return at; };
    x.w = take(static_cast<int64_t>(x.dp) * x.dp);
    x.v = take(static_cast<int64_t>(2) * x.dp * CC_VLD);
    x.e = take(static_cast<int64_t>(CG_GROUP * (CG_GROUP - 1) / 2) * ST_TILE);
    x.m = take(static_cast<int64_t>(2) * ST_TILE);
    plan.mats[i] = CgMat{x.w, x.d, x.dp, copy_blocks, out_blocks};
    copy_blocks += (x.dp + CG_COPY_ROWS - 1) / CG_COPY_ROWS;
    const int t = (x.d + 63) / 64;
    out_blocks += t * (t + 1) / 2;
    bytes += 2.5 * 4 * x.d * x.d;
  }
  double us = 24 + bytes / 3.5e6;
  plan.steps.push_back(CgStep{CG_COPY, 0, count, copy_blocks});
  auto each = [&](int k, auto&& f) {             // the matrices at work in step k
    for (int i = 0; i < count; ++i)
      if (mats[i].nb > std::max(k, 0)) f(i, mats[i]);
  };
  auto group_of = [](int k) { return std::max(k, 0) / CG_GROUP * CG_GROUP; };
  std::vector<char> split(nb_max, 0);            // V alone in a step's launch, its tiles in another one
  std::vector<double> load(nb_max, 0.0);         // us of one CU that the work groups of a step's launch take
  std::vector<double> alone(nb_max, 26.0);       // the launch without products
  std::vector<double> apart(nb_max, 0.0);        // the launch of the tiles
  double rule_us = us + 18;
  for (int k = 0; k < nb_max; ++k) {
    int tiles = 0, rows = 0, leaves = 0;
    std::vector<CgShape> ps;
    const int g0 = group_of(k);
    each(k, [&](int, const Mat& x) {
      const int ge = std::min(g0 + CG_GROUP, x.nb), left = ge - k - 1;
      rows += x.nb;
      tiles += left * (x.nb - k - 1) - left * (left - 1) / 2 + left * (k + 1);
      leaves += k + 1 < x.nb ? 1 : 0;
      if (left > 0) cg_step_shapes(ps, x.dp, k, g0, ge);
    });
    const double panels = std::max(26.0, 9.0 + 9.0 * rows / 256), fused = std::max(26.0, 9.0 + 18.0 * tiles / 256);
    apart[k] = 4.0 + kStepUs * std::max(1.0, tiles / 256.0);
    split[k] = tiles > 0 && (panels + apart[k] < fused || CG_FORCE == 3) && CG_FORCE != 4;
    alone[k] = split[k] || tiles == 0 ? panels : fused;
    load[k] = 26.0 * leaves + (split[k] || tiles == 0 ? 9.0 * rows : 15.0 * tiles);
    rule_us += tiles == 0 ? panels : std::min(fused, panels + cg_shapes_us(ps));
    ps.clear();
    each(k, [&](int, const Mat& x) {
      const int ge = std::min(g0 + CG_GROUP, x.nb);
      if (k + 1 == ge) cg_group_shapes(ps, x.dp, static_cast<int64_t>(g0) * LEAF, std::min<int64_t>(static_cast<int64_t>(ge) * LEAF, x.dp));
    });
    rule_us += cg_shapes_us(ps);
  }
  std::vector<std::vector<CcTask>> beside(nb_max);      // products that step k's launch takes along
  for (int k = -1; k < nb_max; ++k) {
    CgStep st{CG_CHAIN, static_cast<int>(plan.tasks.size()), k, 0};
    const int g0 = group_of(k);
    auto task = [&](int i, int kind, int bi, int bj) {
      const Mat& x = mats[i];
      return CcTask{x.w, x.v, x.e, x.m, i, x.d, x.dp, x.nb, kind, bi, bj, g0};
    };
    auto put = [&](int i, int kind, int bi, int bj) { plan.tasks.push_back(task(i, kind, bi, bj)); };
    each(k, [&](int i, const Mat& x) {
      if (k + 1 < x.nb) put(i, CC_LEAF, k + 1, k + 1);
    });
    auto tiles = [&](int kind) {
      each(k, [&](int i, const Mat& x) {
        const int ge = std::min(g0 + CG_GROUP, x.nb);
        for (int j = k + 1; j < ge; ++j)
          for (int b = j; b < x.nb; ++b)
            if (b != k + 1 || j != k + 1) put(i, kind, b, j);
        for (int r = k + 1; r < ge; ++r)
          for (int b = 0; b <= k; ++b) put(i, kind, r, b);
        if (k + 1 < ge && ge < x.nb) put(i, kind, ge, ge);
      });
    };
    if (k >= 0) {
      each(k, [&](int i, const Mat& x) {
        if (k + 1 != std::min(g0 + CG_GROUP, x.nb) && !split[k]) return;
        for (int b = 0; b < x.nb; ++b)                   // V only
          if (b != k && b != k + 1) put(i, CC_PANEL, b, b);
      });
      if (!split[k]) tiles(CC_TILE);
      each(k, [&](int i, const Mat&) { put(i, CC_OWN, k, k); });
      cg_append_by_xcd(plan.tasks, st.first, beside[k]);
      us += std::max(alone[k], 9.0 + load[k] / 256);
    } else {
      us += 18;
    }
    st.grid = static_cast<int>(plan.tasks.size()) - st.first;
    if (st.grid > 0) plan.steps.push_back(st);
    if (k < 0) continue;
    if (split[k]) {
      CgStep own{CG_CHAIN, static_cast<int>(plan.tasks.size()), k, 0};
      tiles(CC_STEP);
      own.grid = static_cast<int>(plan.tasks.size()) - own.first;
      plan.steps.push_back(own);
      us += apart[k];
    }
    // The products of the matrices whose group ends here.  What the steps of the next group read, its columns, its rows and the
    // diagonal block behind it, is due now; every other tile goes along with the launches of those steps, or, of a matrix that is
    // done, of any step to come: that with the least work so far.  (V of this group is overwritten with the group after the next.)
    std::vector<CcTask> now, later;
    each(k, [&](int i, const Mat& x) {
      const int ge = std::min(g0 + CG_GROUP, x.nb), after = std::min(ge + CG_GROUP, x.nb);
      if (k + 1 != ge) return;
      for (const auto& [bi, bj] : cg_blocked_tiles(x.nb)) {
          if (ge < x.nb && bi == ge && bj == ge) continue;                 // that block is factored
          const bool due = ge < x.nb && ((bi >= ge && bi < after) || (bj >= ge && bj < after) || (bi == after && bj == after));
          (due ? now : later).push_back(task(i, CC_PRODUCT, bi, bj));
      }
      const int last = ge == x.nb ? nb_max - 1 : after - 1;
      if (last <= k) now.insert(now.end(), later.begin(), later.end());
      else
        for (size_t from = 0; from < later.size(); from += kProductChunk) {
          const size_t to = std::min(later.size(), from + kProductChunk);
          int at = k + 1;
          for (int step = k + 2; step <= last; ++step)
            if (load[step] < load[at]) at = step;
          const double more = kProductUs * static_cast<double>(to - from);
          if (load[at] + more > kBesideUs * 256) {
            now.insert(now.end(), later.begin() + from, later.begin() + to);
            continue;
          }
          beside[at].insert(beside[at].end(), later.begin() + from, later.begin() + to);
          load[at] += more;
        }
      later.clear();
    });
    if (!now.empty()) {
      plan.steps.push_back(CgStep{CG_CHAIN, static_cast<int>(plan.tasks.size()), k, static_cast<int>(now.size())});
      cg_append_by_xcd(plan.tasks, static_cast<int>(plan.tasks.size()), now);
      us += 4.0 + kProductUs * std::max(1.0, static_cast<double>(now.size()) / 256);
    }
  }
  plan.steps.push_back(CgStep{CG_OUT, 0, count, out_blocks});
  CgHeader& h = plan.h;
  std::memset(&h, 0, sizeof(h));
  h.magic = CG_MAGIC;
  h.scales_off = off;
  off += cg_align64(static_cast<int64_t>(count) * CG_SCALE_FLOATS);
  h.ws_floats = off;
  h.count = count;
  h.nsteps = static_cast<int>(plan.steps.size());
  h.copy_blocks = copy_blocks;
  h.out_blocks = out_blocks;
  h.us = us;
  int64_t b = cg_align(sizeof(CgHeader), 64);
  h.mats_off = b; b = cg_align(b + plan.mats.size() * sizeof(CgMat), 64);
  h.steps_off = b; b = cg_align(b + plan.steps.size() * sizeof(CgStep), 64);
  h.tasks_off = b; b = cg_align(b + plan.tasks.size() * sizeof(CcTask), 64);
  h.total_bytes = b;
  return rule_us;
}

// The sweep holds more: its sums are 128 long and its operands have all their bits, the chain's products sum 512 and take two
// fp16 pieces (22 bits).  Error against 64 bits of the inverses, sweep and chain: ReLU rows of rank d / 8, a / lam = 2^12, 3072 4.8e-3 and
// 5.2e-3, 1700 2.7e-3 and 3.2e-3; full rank 3072 2.8e-7 and 3.6e-7.  It takes half the memory, too (3072: 23 and 51 MB).  So the chain is for groups whose steps take three rounds of tiles
// and more, and of matrices of 15 block columns and more whose third round is used (the 2.3) it has to save a quarter: up to there
// the sweep served when it was as slow as fp32 products make it, so that no size has lost accuracy since.  The rule goes by the chain with its
// products in launches of their own, as it was when it was measured (it takes up to a tenth less now).  Measured then, sweep and
// chain, us: two rounds 3072 868 and 846, 2600 with 2304, 2048, 1500, 700, 600 1030 and 930; three and more 4 x 2048 855 and 652,
// 3 x 2304 886 and 704, 4 x 2400 with 8 x 512 1230 and 880, 60 x 513 373 and 346.  The bound of 4096 tiles keeps the tables of
// hopeless cases from being built.
static void cg_build(const int64_t* dims, int count, CgPlan& plan) {
  int64_t tiles = 0, nb_max = 0, rounds;
  for (int m = 0; m < count; ++m) {
    const int64_t nb = (dims[m] + LEAF - 1) / LEAF;
    nb_max = std::max(nb_max, nb);
    tiles += nb * (nb + 1) / 2;
  }
  double filled;
  const double sweep_us = cg_sweep_us(dims, count, rounds, filled);
  bool sweep = CG_FORCE == 1 || (CG_FORCE == 0 && tiles <= 4096 && rounds < 3 * nb_max);
  if (!sweep) {
    const double us = cg_build_chain(dims, count, plan);
    const double worth = nb_max >= 15 && filled >= 2.3 * static_cast<double>(nb_max) ? 0.73 : 0.92;
    sweep = CG_FORCE == 0 && tiles <= 4096 && us >= worth * sweep_us;
  }
  if (!sweep) return;
  plan = CgPlan();
  cg_build_sweep(dims, count, plan);
  plan.h.us = sweep_us;
}

// The plan of the sizes that this thread asked for last: a caller asks for the bytes, the workspace and the plan one after the other,
// and the tables are given back with the plan.
struct CgKept {
  std::vector<int64_t> key;
  CgPlan plan;
};
static CgKept& cg_kept() {
  thread_local CgKept kept;
  return kept;
}
static const CgPlan& cg_plan(const int64_t* dims, int count) {
  CgKept& kept = cg_kept();
  std::vector<int64_t> asked(dims, dims + count);
  asked.push_back(CG_FORCE);
  if (kept.key != asked) {
    kept = CgKept();                   // (nothing is kept if the tables do not fit the memory)
    cg_build(dims, count, kept.plan);
    kept.key.swap(asked);
  }
  return kept.plan;
}

}  // namespace ak

extern "C" size_t ak_chol_group_plan_bytes(const int64_t* dims, int count) {
  if (!ak::cg_dims_ok(dims, count)) return 0;
  return static_cast<size_t>(ak::cg_plan(dims, count).h.total_bytes);
}

extern "C" size_t ak_chol_group_ws_bytes(const int64_t* dims, int count) {
  if (!ak::cg_dims_ok(dims, count)) return 0;
  return static_cast<size_t>(ak::cg_plan(dims, count).h.ws_floats) * sizeof(float);
}

extern "C" int ak_chol_group_plan(const int64_t* dims, int count, void* plan_host, size_t plan_bytes) {
  using namespace ak;
  if (!cg_dims_ok(dims, count) || plan_host == nullptr) return AK_ERR_ARG;
  const CgPlan& plan = cg_plan(dims, count);
  if (plan_bytes < static_cast<size_t>(plan.h.total_bytes)) return AK_ERR_WORKSPACE;
  unsigned char* out = static_cast<unsigned char*>(plan_host);
  std::memset(out, 0, static_cast<size_t>(plan.h.total_bytes));
  std::memcpy(out, &plan.h, sizeof(CgHeader));
  if (!plan.mats.empty()) std::memcpy(out + plan.h.mats_off, plan.mats.data(), plan.mats.size() * sizeof(CgMat));
  std::memcpy(out + plan.h.steps_off, plan.steps.data(), plan.steps.size() * sizeof(CgStep));
  if (!plan.tasks.empty()) std::memcpy(out + plan.h.tasks_off, plan.tasks.data(), plan.tasks.size() * sizeof(CcTask));
  if (!plan.sweep_leaves.empty()) {
    std::memcpy(out + plan.h.tasks_off, plan.sweep_leaves.data(), plan.sweep_leaves.size() * sizeof(SwTask));
    std::memcpy(out + plan.h.tiles_off, plan.sweep_tiles.data(), plan.sweep_tiles.size() * sizeof(SwTask));
  }
  cg_kept() = CgKept();
  return AK_OK;
}

extern "C" int ak_chol_group_plan_launches(const void* plan_host) {
  if (plan_host == nullptr) return AK_ERR_ARG;
  const ak::CgHeader* h = static_cast<const ak::CgHeader*>(plan_host);
  return h->magic == ak::CG_MAGIC ? h->nsteps : AK_ERR_ARG;
}

extern "C" double ak_chol_group_plan_us(const void* plan_host) {
  if (plan_host == nullptr) return -1.0;
  const ak::CgHeader* h = static_cast<const ak::CgHeader*>(plan_host);
  return h->magic == ak::CG_MAGIC ? h->us : -1.0;
}

extern "C" int ak_chol_inv_grouped(const void* plan_host, const void* plan_dev, const float* const* A_list,
                                   float* const* out_list, const float* lam, int lam_stride, const int* skip_flags,
                                   int skip_stride, int* info, void* ws, size_t ws_bytes, ak_stream_t stream) {
  using namespace ak;
  if (plan_host == nullptr || plan_dev == nullptr || A_list == nullptr || out_list == nullptr || lam == nullptr ||
      info == nullptr)
    return AK_ERR_ARG;
  const unsigned char* ph = static_cast<const unsigned char*>(plan_host);
  const CgHeader* h = reinterpret_cast<const CgHeader*>(ph);
  if (h->magic != CG_MAGIC || h->count <= 0 || h->nsteps <= 0) return AK_ERR_ARG;
  if (ws == nullptr || (reinterpret_cast<uintptr_t>(ws) & 255) != 0 ||
      ws_bytes < static_cast<size_t>(h->ws_floats) * sizeof(float))
    return AK_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  CgArgs a;
  a.plan = static_cast<const unsigned char*>(plan_dev);
  a.ws = static_cast<float*>(ws);
  a.A_list = A_list; a.out_list = out_list;
  a.lam = lam; a.skip = skip_flags; a.info = info;
  a.lam_stride = lam_stride; a.skip_stride = skip_stride;
  a.scales = a.ws + h->scales_off;
  const CgStep* steps = reinterpret_cast<const CgStep*>(ph + h->steps_off);
  for (int i = 0; i < h->nsteps; ++i) {
    const CgStep& st = steps[i];
    if (st.grid <= 0) continue;
    if (st.type == CG_SWEEP) {
      const SwArgs w{a.ws, A_list, out_list, lam, skip_flags, info, lam_stride, skip_stride};
      hipLaunchKernelGGL(cg_sweep_kernel, dim3(st.grid), dim3(LEAF_THREADS), 0, s, w,
                         reinterpret_cast<const SwTask*>(a.plan + h->tasks_off),
                         reinterpret_cast<const SwTask*>(a.plan + h->tiles_off), st.count, st.first);
    } else if (st.type == CG_COPY) {
      hipLaunchKernelGGL(cg_copy_in_kernel, dim3(st.grid), dim3(256), 0, s, a, h->count);
      hipLaunchKernelGGL(cg_scale_kernel, dim3(h->count), dim3(256), 0, s, a, h->count, CG_HALF_MAX_COND);
    } else if (st.type == CG_OUT) {
      hipLaunchKernelGGL(cg_out_kernel, dim3(st.grid), dim3(256), 0, s, a, h->count);
    } else {
      const CcArgs c{a.ws, skip_flags, info, a.scales, A_list, lam, skip_stride, lam_stride};
      const CcTask* tasks = reinterpret_cast<const CcTask*>(a.plan + h->tasks_off) + st.first;
      hipLaunchKernelGGL(cg_chain_kernel, dim3(st.grid), dim3(LEAF_THREADS), 0, s, c, tasks, st.count);
    }
  }
  return check_launch();
}

#ifdef AK_TUNING_HOOKS
// Tuning builds only: the bound a / lam up to which a matrix takes the fp16-piece products (0: never).
extern "C" void ak_debug_set_chol_half_max_cond(float v) { ak::CG_HALF_MAX_COND = v; }
// Tuning builds only: the plan (CG_FORCE), 0: the rule.
extern "C" void ak_debug_force_chol_plan(int v) { ak::CG_FORCE = v; }
#endif
