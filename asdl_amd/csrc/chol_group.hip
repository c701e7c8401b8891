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
// The steps of all matrices are merged: step k of the chain is one launch for all matrices that have a block k, the products
// at the end of a group are one launch for all matrices (one work group per tile of any product, descriptor found through a
// tile -> product map; 128 x 128 split-operand MFMA tiles of gemm_x3.hpp, or the smaller fp32 tiles of gemm_deep.hpp where
// those would leave the device idle: cg_prefer_deep).
//
// The plan (descriptor tables, launch sequence) depends on the sizes only; every address in it is an offset into the
// workspace.  The caller builds it once per size set on the host (ak_chol_group_plan), keeps a device copy, and
// passes both to every call.
//
// Matrices are padded to a multiple of 4 columns with an identity block (the padded rows and columns drop out of the
// result), which keeps every operand of the split kernel 16-byte aligned.  Only the lower triangle of the input is
// read; the strictly upper 128-blocks of W are never touched.
#include <algorithm>
#include <cstring>
#include <vector>
#include "gemm_f32.hpp"
#include "chol_sweep.hpp"
#include "chol_chain.hpp"

namespace ak {

constexpr int64_t CG_MAGIC = 0x3447524c4f4843ll;     // "CHOLGR4"
constexpr int CG_COPY = 0, CG_CHAIN = 1, CG_PROD = 2, CG_PROD_DEEP = 3, CG_SWEEP = 4, CG_OUT = 5;

// What an operand of a product holds, for the fp16-piece products (bits 4-5 of CgProd::flags: A, bits 6-7: B).  With
// a = the largest diagonal element of A + lam I, every element is bounded in magnitude: of the Cholesky factor L by sqrt(a),
// of M = L^-1 by 1 / sqrt(lam).
constexpr int CG_KIND_L = 1, CG_KIND_M = 2;
constexpr int CG_SCALE_FLOATS = 4;                    // per matrix: the fp16 switch, the scales of both kinds, padding
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
  int64_t mats_off, steps_off, tasks_off, prods_off, map_off;      // byte offsets of the tables inside the plan
  int32_t count, nsteps, copy_blocks, out_blocks;
  double us;                // estimated time of one call (cg_build)
};

struct CgMat {
  int64_t w_off;            // work matrix [dp, dp], offset in floats from the workspace base
  int32_t d, dp;
  int32_t first_copy_block, first_out_block;
};

struct CgStep {
  int32_t type, first, count, grid;    // chain: first task, step k, tasks; products: first product, products, tiles
  int32_t first_tile, pad0;            // products: where the step's tile -> product map starts
};

struct CgProd {
  int64_t a_off, b_off, c_off;
  int32_t lda, ldb, ldc;
  int32_t M, N, K;
  int32_t flags, kmode, tile_mode;
  float alpha, beta;
  int32_t mat;
  int32_t first_tile, tiles_m, tiles_n;
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

// W_m <- lower(A_m) + lam_m I, padded rows carry the identity; info_m <- 0.  One work group per CG_COPY_ROWS rows of
// one matrix (bisection on first_copy_block); a row is read and written up to its diagonal element only.
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
    if (r >= m.d) {
      // padding: a diagonal block that drops out of the result.  Its value lam (1 when lam <= 0) stays inside the
      // magnitude bounds the fp16-piece products scale their operands by (lam <= a, 1 / sqrt(lam) for the inverse).
      const float pad = l > 0.f ? l : 1.f;
      for (int c = threadIdx.x; c <= r; c += 256) dst[c] = (c == r) ? pad : 0.f;
      continue;
    }
    const float* __restrict__ src = A + static_cast<int64_t>(r) * m.d;
    if (vec) {
      for (int c = 4 * threadIdx.x; c <= r; c += 1024) {
        floatx4 v = *reinterpret_cast<const floatx4*>(src + c);
        if (r >= c && r < c + 4) v[r - c] += l;
        *reinterpret_cast<floatx4*>(dst + c) = v;       // the elements right of the diagonal are never read
      }
    } else {
      for (int c = threadIdx.x; c <= r; c += 256) dst[c] = src[c] + ((c == r) ? l : 0.f);
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

// Tile (ti, tj) number `local` of a product, longest contraction first where the range depends on the tile.
__device__ __forceinline__ void cg_decode_tile(const CgProd& d, int local, int& ti, int& tj) {
  if (d.tile_mode != TILE_ALL) {     // tiles on and below the diagonal, row by row (K_GE_MAXIJ: longest first)
    ti = static_cast<int>((__builtin_sqrtf(8.f * static_cast<float>(local) + 1.f) - 1.f) * 0.5f);
    while ((ti + 1) * (ti + 2) / 2 <= local) ++ti;
    while (ti * (ti + 1) / 2 > local) --ti;
    tj = local - ti * (ti + 1) / 2;
    return;
  }
  if (d.kmode == K_GE_J) {           // k >= column tile: first column first
    tj = local / d.tiles_m;
    ti = local % d.tiles_m;
  } else {
    ti = local / d.tiles_n;
    tj = local % d.tiles_n;
  }
}

// One work group per 128 x 128 tile of any product of the step; tile_map[w] = the product of work group w.
static __global__ __launch_bounds__(256, 2) void cg_prod_kernel(CgArgs a, const CgProd* __restrict__ prods,
                                                             const int32_t* __restrict__ tile_map) {
  __shared__ __attribute__((aligned(16))) unsigned char x3_smem[2 * 3 * X3_PLANE];
  const int w = blockIdx.x;
  const CgProd d = prods[tile_map[w]];
  // (a skipped matrix's work area holds whatever the last call left there; its steps still run and touch nothing else)
  int ti, tj;
  cg_decode_tile(d, w - d.first_tile, ti, tj);
  GemmParams p;
  p.A = a.ws + d.a_off;
  p.B = a.ws + d.b_off;
  p.C = a.ws + d.c_off;
  p.C_list = nullptr;
  p.lda = d.lda; p.ldb = d.ldb; p.ldc = d.ldc;
  p.sA = p.sB = p.sC = 0;
  p.M = d.M; p.N = d.N; p.K = d.K;
  p.transA = 0; p.transB = 1;
  p.alpha = d.alpha; p.beta = d.beta;
  p.kmode = d.kmode; p.tile_mode = d.tile_mode;
  p.active = nullptr; p.active_stride = 0;
  p.split = 3;
  p.scaleA = p.scaleB = 1.f;
  const float* __restrict__ sc = a.scales + static_cast<int64_t>(d.mat) * CG_SCALE_FLOATS;
  if (sc[0] != 0.f) {
    // fp16 pieces: two per operand element, three matrix instructions per product instead of six
    p.scaleA = sc[(d.flags >> 4) & 3];
    p.scaleB = sc[(d.flags >> 6) & 3];
    p.alpha = d.alpha / (p.scaleA * p.scaleB);      // powers of two: exact
    if (d.beta != 0.f) gemm_x3_tile<2, false, 1, 1, true, false, true>(p, ti, tj, 0, (AK_LDS3 unsigned char*)x3_smem);
    else gemm_x3_tile<2, false, 1, 1, true>(p, ti, tj, 0, (AK_LDS3 unsigned char*)x3_smem);
  } else {
    gemm_x3_tile<3, false, 1, 1>(p, ti, tj, 0, (AK_LDS3 unsigned char*)x3_smem);
  }
}

// The same for the steps whose 128 x 128 tiles would leave most of the device idle: deep fp32 tiles of 64 x 64 (gemm_deep.hpp).
static __global__ __launch_bounds__(256, 2) void cg_prod_deep_kernel(CgArgs a, const CgProd* __restrict__ prods,
                                                                  const int32_t* __restrict__ tile_map) {
  __shared__ __attribute__((aligned(16))) float lds[deep_lds_floats<64, 64, 128>()];
  const int w = blockIdx.x;
  const CgProd d = prods[tile_map[w]];
  int ti, tj;
  cg_decode_tile(d, w - d.first_tile, ti, tj);
  GemmParams p;
  p.A = a.ws + d.a_off;
  p.B = a.ws + d.b_off;
  p.C = a.ws + d.c_off;
  p.lda = d.lda; p.ldb = d.ldb; p.ldc = d.ldc;
  p.M = d.M; p.N = d.N; p.K = d.K;
  p.transA = 0; p.transB = 1;
  p.alpha = d.alpha; p.beta = d.beta;
  p.kmode = d.kmode; p.tile_mode = d.tile_mode;
  gemm_deep_tile<64, 64, 128>(p, ti, tj, 0, lds);
}

// ---- host: the plan ------------------------------------------------------------------------------------------

static inline int64_t cg_align64(int64_t x) { return (x + 63) / 64 * 64; }

static int64_t cg_tiles(const CgProd& p) {
  return p.tile_mode == TILE_ALL ? static_cast<int64_t>(p.tiles_m) * p.tiles_n
                                 : static_cast<int64_t>(p.tiles_m) * (p.tiles_m + 1) / 2;
}

// Tiles of the deep kernel instead of 128 x 128.
static void cg_make_deep(CgProd& p) {
  p.tiles_m = (p.M + 63) / 64;
  p.tiles_n = (p.N + 63) / 64;
}

// Microseconds of the products of one super-step (cg_prefer_deep), its launch not counted.
static double cg_product_us(const std::vector<CgProd>& ps, bool deep) {
  double longest = 0, sum = 0;
  for (const CgProd& p : ps) {
    CgProd q = p;
    if (deep) cg_make_deep(q);
    const double c = deep ? (p.K + 127) / 128 : (p.K + 31) / 32;
    longest = std::max(longest, c);
    sum += c * static_cast<double>(cg_tiles(q));
  }
  return deep ? 2.0 * std::max(longest, sum / 256) : std::max(1.6 * longest, 1.05 * sum / 256);
}

// Which kernel a super-step's products take.  The split kernel's 128 x 128 tiles have three times the rate once they
// fill the device (about 1 us per k-tile of 32 and CU), but a tile takes 1.6 us per k-tile however few there are; the
// deep tiles take 2 us per chunk of 128 k.  The step is as long as its longest tile or as its work spread over the CUs.
static bool cg_prefer_deep(const std::vector<CgProd>& ps) { return cg_product_us(ps, true) < cg_product_us(ps, false); }

// C = beta C + alpha A B^T
static CgProd cg_prod(int mat, int kind_a, int kind_b, int M, int N, int K, float alpha, int64_t a, int lda,
                      int64_t b, int ldb, float beta, int64_t c, int ldc, int kmode, int tile_mode) {
  CgProd p;
  std::memset(&p, 0, sizeof(p));
  p.a_off = a; p.b_off = b; p.c_off = c;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = M; p.N = N; p.K = K;
  p.flags = (kind_a << 4) | (kind_b << 6); p.kmode = kmode; p.tile_mode = tile_mode;
  p.alpha = alpha; p.beta = beta;
  p.mat = mat;
  p.tiles_m = (M + 127) / 128;
  p.tiles_n = (N + 127) / 128;
  return p;
}

// The products at the end of the group of columns [c0, c1) of one matrix: X -+ V V^T.  Rows and columns of the group, whose
// old values have become V, are formed anew.
static void cg_group_products(std::vector<CgProd>& ps, int mat, int64_t w, int64_t v, int dp, int c0, int c1) {
  const int width = c1 - c0, below = dp - c1;
  auto at = [&](int r, int c) { return w + static_cast<int64_t>(r) * dp + c; };
  auto put = [&](int kind_a, int kind_b, int r, int M, int c, int N, float alpha, float beta, int kmode, int tile_mode) {
    if (M <= 0 || N <= 0) return;
    ps.push_back(cg_prod(mat, kind_a, kind_b, M, N, width, alpha, v + static_cast<int64_t>(r) * CC_VLD, CC_VLD,
                         v + static_cast<int64_t>(c) * CC_VLD, CC_VLD, beta, at(r, c), dp, kmode, tile_mode));
  };
  put(CG_KIND_L, CG_KIND_L, c1, below, c1, below, -1.f, 1.f, K_FULL, TILE_LOWER);
  put(CG_KIND_L, CG_KIND_M, c1, below, c0, width, -1.f, 0.f, K_GE_J, TILE_ALL);
  put(CG_KIND_L, CG_KIND_M, c1, below, 0, c0, -1.f, 1.f, K_FULL, TILE_ALL);
  put(CG_KIND_M, CG_KIND_M, c0, width, 0, c0, 1.f, 0.f, K_GE_I, TILE_ALL);
  put(CG_KIND_M, CG_KIND_M, c0, width, c0, width, 1.f, 0.f, K_GE_MAXIJ, TILE_LOWER);
  put(CG_KIND_M, CG_KIND_M, 0, c0, 0, c0, 1.f, 1.f, K_FULL, TILE_LOWER);
}

// The tiles of step k of one matrix (chol_chain.hpp) as products of 128 columns of V, for launches of their own.
static void cg_step_products(std::vector<CgProd>& ps, int mat, int64_t w, int64_t v, int64_t e, int dp, int k, int g0, int ge) {
  const int c0 = g0 * LEAF, c1 = (k + 1) * LEAF, c2 = std::min(ge * LEAF, dp);
  auto at = [&](int r, int c) { return w + static_cast<int64_t>(r) * dp + c; };
  auto row = [&](int r) { return v + static_cast<int64_t>(r) * CC_VLD + (k - g0) * LEAF; };
  auto put = [&](int kind_b, int r, int M, int c, int N, float beta, int64_t to, int ld, int tile_mode) {
    if (M > 0 && N > 0)
      ps.push_back(cg_prod(mat, CG_KIND_L, kind_b, M, N, LEAF, -1.f, row(r), CC_VLD, row(c), CC_VLD, beta, to, ld, K_FULL, tile_mode));
  };
  put(CG_KIND_L, c1, c2 - c1, c1, c2 - c1, 1.f, at(c1, c1), dp, TILE_LOWER);
  put(CG_KIND_L, c2, dp - c2, c1, c2 - c1, 1.f, at(c2, c1), dp, TILE_ALL);
  put(CG_KIND_L, c2, std::min(LEAF, dp - c2), c2, std::min(LEAF, dp - c2), 1.f, at(c2, c2), dp, TILE_LOWER);
  put(CG_KIND_M, c1, c2 - c1, 0, c0, 1.f, at(c1, 0), dp, TILE_ALL);
  for (int r = k + 1; r < ge; ++r)
    for (int i = g0; i <= k; ++i)
      put(CG_KIND_M, r * LEAF, std::min(LEAF, dp - r * LEAF), i * LEAF, LEAF, i < k ? 1.f : 0.f,
          e + static_cast<int64_t>((r - g0) * (r - g0 - 1) / 2 + i - g0) * ST_TILE, LEAF, TILE_ALL);
}

struct CgPlan {
  CgHeader h;
  std::vector<CgMat> mats;
  std::vector<CgStep> steps;
  std::vector<CcTask> tasks;
  std::vector<CgProd> prods;
  std::vector<int32_t> tile_map;
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
    plan.steps.push_back(CgStep{CG_SWEEP, k, leaves, leaves + tiles, 0, 0});
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
  h.prods_off = b; b = cg_align(b + plan.sweep_tiles.size() * sizeof(SwTask), 64);
  h.mats_off = h.map_off = b;
  h.total_bytes = b;
}

#ifdef AK_TUNING_HOOKS
static int CG_FORCE = 0;               // tuning builds: 1 the sweep, 2 the chain, 3 (4) with (without) launches of their own for its tiles
#else
constexpr int CG_FORCE = 0;
#endif

// The chain's tables.  Returns its estimated time: 26 us a step, or 9 and 18 per round of tiles (of panels alone: 9) where that is
// more, the products by cg_product_us, the copies by their bytes.
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
  // one launch of products, if any: its estimated time; written to the plan or not
  auto products = [&](std::vector<CgProd> ps, bool write) {
    if (ps.empty()) return 0.0;
    CgStep pr{CG_PROD, static_cast<int>(plan.prods.size()), static_cast<int>(ps.size()), 0, static_cast<int>(plan.tile_map.size()), 0};
    const bool deep = cg_prefer_deep(ps);
    if (deep) {
      pr.type = CG_PROD_DEEP;
      for (CgProd& p : ps) cg_make_deep(p);
    }
    const double time = 4 + cg_product_us(ps, deep);
    if (!write) return time;
    // longest contraction first: the long tiles start early, the short ones (those that start in the middle of it) fill the tail
    auto depth = [](const CgProd& p) { return p.kmode == K_FULL ? 2 * p.K : p.K; };
    std::stable_sort(ps.begin(), ps.end(), [&](const CgProd& x, const CgProd& y) { return depth(x) > depth(y); });
    int64_t n = 0;
    for (size_t i = 0; i < ps.size(); ++i) {
      ps[i].first_tile = static_cast<int>(n);
      const int64_t mine = cg_tiles(ps[i]);
      n += mine;
      plan.tile_map.insert(plan.tile_map.end(), static_cast<size_t>(mine), static_cast<int32_t>(i));
    }
    pr.grid = static_cast<int>(n);
    plan.prods.insert(plan.prods.end(), ps.begin(), ps.end());
    plan.steps.push_back(pr);
    return time;
  };
  plan.steps.push_back(CgStep{CG_COPY, 0, count, copy_blocks, 0, 0});
  for (int k = -1; k < nb_max; ++k) {
    CgStep st{CG_CHAIN, static_cast<int>(plan.tasks.size()), k, 0, 0, 0};
    auto each = [&](auto&& f) {
      for (int i = 0; i < count; ++i)
        if (mats[i].nb > std::max(k, 0)) f(i, mats[i]);
    };
    auto put = [&](int i, int kind, int bi, int bj) {
      const Mat& x = mats[i];
      const int g0 = std::max(k, 0) / CG_GROUP * CG_GROUP;
      plan.tasks.push_back(CcTask{x.w, x.v, x.e, x.m, i, x.d, x.dp, x.nb, kind, bi, bj, g0});
    };
    each([&](int i, const Mat& x) {
      if (k + 1 < x.nb) put(i, CC_LEAF, k + 1, k + 1);
    });
    const int g0 = std::max(k, 0) / CG_GROUP * CG_GROUP;
    std::vector<CgProd> ps;
    bool split = false;
    if (k >= 0) {
      int tiles = 0, rows = 0;
      each([&](int i, const Mat& x) {
        const int ge = std::min(g0 + CG_GROUP, x.nb), left = ge - k - 1;
        rows += x.nb;
        tiles += left * (x.nb - k - 1) - left * (left - 1) / 2 + left * (k + 1);
        if (left > 0) cg_step_products(ps, i, x.w, x.v + static_cast<int64_t>(g0 / CG_GROUP & 1) * x.dp * CC_VLD, x.e, x.dp, k, g0, ge);
      });
      const double fused = std::max(26.0, 9.0 + 18.0 * tiles / 256), apart = std::max(26.0, 9.0 + 9.0 * rows / 256) + products(ps, false);
      split = !ps.empty() && (apart < fused || CG_FORCE == 3) && CG_FORCE != 4;
      us += split || ps.empty() ? std::max(26.0, 9.0 + 9.0 * rows / 256) : fused;
      each([&](int i, const Mat& x) {
        const int ge = std::min(g0 + CG_GROUP, x.nb);
        if (k + 1 == ge || split) {                      // V only
          for (int b = 0; b < x.nb; ++b)
            if (b != k && b != k + 1) put(i, CC_PANEL, b, b);
          return;
        }
        for (int j = k + 1; j < ge; ++j)
          for (int b = j; b < x.nb; ++b)
            if (b != k + 1 || j != k + 1) put(i, CC_TILE, b, j);
        for (int r = k + 1; r < ge; ++r)
          for (int b = 0; b <= k; ++b) put(i, CC_TILE, r, b);
        if (ge < x.nb) put(i, CC_TILE, ge, ge);
      });
    } else {
      us += 18;
    }
    st.grid = static_cast<int>(plan.tasks.size()) - st.first;
    if (st.grid > 0) plan.steps.push_back(st);
    if (split) us += products(ps, true);
    ps.clear();
    // the group's products, by the matrices whose group ends here
    if (k >= 0) {
      each([&](int i, const Mat& x) {
        if (k + 1 != std::min(g0 + CG_GROUP, x.nb)) return;
        const int64_t v = x.v + static_cast<int64_t>(g0 / CG_GROUP & 1) * x.dp * CC_VLD;
        cg_group_products(ps, i, x.w, v, x.dp, g0 * LEAF, std::min((k + 1) * LEAF, x.dp));
      });
    }
    us += products(ps, true);
  }
  plan.steps.push_back(CgStep{CG_OUT, 0, count, out_blocks, 0, 0});
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
  h.prods_off = b; b = cg_align(b + plan.prods.size() * sizeof(CgProd), 64);
  h.map_off = b; b = cg_align(b + plan.tile_map.size() * sizeof(int32_t), 64);
  h.total_bytes = b;
  return us;
}

// The sweep holds more: its sums are 128 long and its operands have all their bits, the chain's products sum 512 and take two
// fp16 pieces (22 bits).  Error against 64 bits of the inverses, sweep and chain: ReLU rows of rank d / 8, a / lam = 2^12, 3072 4.8e-3 and
// 1.4e-2, 6 x 1700 2.7e-3 and 6.1e-3; full rank 3072 2.8e-7 and 3.8e-7.  (Three bf16 pieces in the chain's products: 1.7e-2, more
// roundings.)  It takes half the memory, too (3072: 23 and 51 MB).  So the chain is for groups whose steps take three rounds of tiles
// and more, and of matrices of 15 block columns and more whose third round is used (the 2.3) it has to save a quarter: up to there
// the sweep served when it was as slow as fp32 products make it, so that no size has lost accuracy since.  Measured, sweep and
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
  if (!plan.prods.empty()) std::memcpy(out + plan.h.prods_off, plan.prods.data(), plan.prods.size() * sizeof(CgProd));
  if (!plan.sweep_leaves.empty()) {
    std::memcpy(out + plan.h.tasks_off, plan.sweep_leaves.data(), plan.sweep_leaves.size() * sizeof(SwTask));
    std::memcpy(out + plan.h.prods_off, plan.sweep_tiles.data(), plan.sweep_tiles.size() * sizeof(SwTask));
  }
  if (!plan.tile_map.empty())
    std::memcpy(out + plan.h.map_off, plan.tile_map.data(), plan.tile_map.size() * sizeof(int32_t));
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
                         reinterpret_cast<const SwTask*>(a.plan + h->prods_off), st.count, st.first);
    } else if (st.type == CG_COPY) {
      hipLaunchKernelGGL(cg_copy_in_kernel, dim3(st.grid), dim3(256), 0, s, a, h->count);
      hipLaunchKernelGGL(cg_scale_kernel, dim3(h->count), dim3(256), 0, s, a, h->count, CG_HALF_MAX_COND);
    } else if (st.type == CG_OUT) {
      hipLaunchKernelGGL(cg_out_kernel, dim3(st.grid), dim3(256), 0, s, a, h->count);
    } else if (st.type == CG_CHAIN) {
      hipLaunchKernelGGL(cg_chain_kernel, dim3(st.grid), dim3(LEAF_THREADS), 0, s, CcArgs{a.ws, skip_flags, info, skip_stride},
                         reinterpret_cast<const CcTask*>(a.plan + h->tasks_off) + st.first, st.count);
    } else
      hipLaunchKernelGGL(st.type == CG_PROD ? cg_prod_kernel : cg_prod_deep_kernel, dim3(st.grid), dim3(256), 0, s, a,
                         reinterpret_cast<const CgProd*>(a.plan + h->prods_off) + st.first,
                         reinterpret_cast<const int32_t*>(a.plan + h->map_off) + st.first_tile);
  }
  return check_launch();
}

#ifdef AK_TUNING_HOOKS
// Tuning builds only: the bound a / lam up to which a matrix takes the fp16-piece products (0: never).
extern "C" void ak_debug_set_chol_half_max_cond(float v) { ak::CG_HALF_MAX_COND = v; }
// Tuning builds only: the plan (CG_FORCE), 0: the rule.
extern "C" void ak_debug_force_chol_plan(int v) { ak::CG_FORCE = v; }
#endif
