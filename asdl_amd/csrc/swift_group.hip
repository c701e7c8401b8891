// Inverses of many low-rank factors at once: (x^T x / n + lam I)^-1 = (I - x^T (x x^T + n lam I)^-1 x) / lam for [n, d] row matrices
// with few rows.  Four launches around one grouped inverse of the n x n Gram matrices, where every factor used to be a chain
// of ten launches of its own on a nearly idle device: partial Gram matrices over slices of d, their sums, y = G^-1 x, and the
// result with its scale and diagonal in the product's epilogue (it is written once and read never).  Deep fp32 tiles
// (gemm_deep.hpp); the last launch is bound by writing d^2 floats, the others by latency.  Addresses travel in the kernel
// arguments.  SKFAC step of a ResNet-18 (14 low-rank factors): host time of the inverses 1.5 -> 0.3 ms.
#include <algorithm>
#include "gemm_f32.hpp"

namespace ak {

constexpr int SG_ITEMS = 24;
constexpr int SG_SLICE = 512;            // columns of x per partial Gram matrix: four chunks of a deep tile

struct SgItem {
  const float* x;                        // [n][d]
  float* gram;
  const float* ginv;
  float* y;                              // [n][d]; before that the partial Gram tiles
  float* out;
  const float* lam;
  float* lam_n;
  int n, d, first, slices;
};
struct SgArgs {
  int count;
  SgItem item[SG_ITEMS];
};

__device__ __forceinline__ const SgItem& sg_item_of(const SgArgs& a, int w) {
  int i = 0;
  while (i + 1 < a.count && a.item[i + 1].first <= w) ++i;
  return a.item[i];
}
__device__ __forceinline__ GemmParams sg_params(const float* A, int64_t lda, int transA, const float* B, int64_t ldb, int transB,
                                                float* C, int64_t ldc, int M, int N, int K) {
  GemmParams p;
  p.A = A; p.B = B; p.C = C;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc;
  p.M = M; p.N = N; p.K = K;
  p.transA = transA; p.transB = transB;
  p.alpha = 1.f; p.beta = 0.f;
  p.kmode = K_FULL; p.tile_mode = TILE_ALL;
  return p;
}

// Work group: slice (of d) x tile on or below the diagonal of x x^T; partial tile [64][64] number w - first.
static __global__ __launch_bounds__(256) void sg_gram_kernel(SgArgs a) {
  __shared__ __attribute__((aligned(16))) float lds[deep_lds_floats<64, 64, 128>()];
  const SgItem& m = sg_item_of(a, blockIdx.x);
  const int T = (m.n + 63) / 64, tiles = T * (T + 1) / 2, local = blockIdx.x - m.first;
  const int slice = local / tiles;
  int ti, tj;
  decode_lower_tile(local - slice * tiles, ti, tj);
  const int k0 = slice * SG_SLICE;
  float* part = m.y + static_cast<int64_t>(local) * 4096 - (ti * 64 * 64 + tj * 64);
  gemm_deep_tile<64, 64, 128>(sg_params(m.x + k0, m.d, 0, m.x + k0, m.d, 1, part, 64, m.n, m.n, min(SG_SLICE, m.d - k0)), ti, tj, 0, lds);
}

// Work group: one tile, summed over the slices in order; both triangles.
static __global__ __launch_bounds__(256) void sg_sum_kernel(SgArgs a) {
  const SgItem& m = sg_item_of(a, blockIdx.x);
  const int T = (m.n + 63) / 64, tiles = T * (T + 1) / 2, local = blockIdx.x - m.first;
  if (local == 0 && threadIdx.x == 0) m.lam_n[0] = static_cast<float>(m.n) * m.lam[0];
  int ti, tj;
  decode_lower_tile(local, ti, tj);
  const float* __restrict__ part = m.y + static_cast<int64_t>(local) * 4096;
  for (int e = threadIdx.x; e < 4096; e += 256) {
    const int i = ti * 64 + e / 64, j = tj * 64 + e % 64;
    if (i >= m.n || j >= m.n || j > i) continue;
    float s = 0.f;
    for (int k = 0; k < m.slices; ++k) s += part[static_cast<int64_t>(k) * tiles * 4096 + e];
    m.gram[static_cast<int64_t>(i) * m.n + j] = s;
    m.gram[static_cast<int64_t>(j) * m.n + i] = s;
  }
}

// y <- G^-1 x
static __global__ __launch_bounds__(256) void sg_solve_kernel(SgArgs a) {
  __shared__ __attribute__((aligned(16))) float lds[deep_lds_floats<64, 64, 128>()];
  const SgItem& m = sg_item_of(a, blockIdx.x);
  const int tn = (m.d + 63) / 64, local = blockIdx.x - m.first;
  gemm_deep_tile<64, 64, 128>(sg_params(m.ginv, m.n, 0, m.x, m.d, 0, m.y, m.d, m.n, m.d, m.n), local / tn, local % tn, 0, lds);
}

// out <- (I - x^T y) / lam, lower tiles and their mirror images
static __global__ __launch_bounds__(256) void sg_out_kernel(SgArgs a) {
  __shared__ __attribute__((aligned(16))) float lds[deep_lds_floats<64, 64, 128>()];
  const SgItem& m = sg_item_of(a, blockIdx.x);
  int ti, tj;
  decode_lower_tile(blockIdx.x - m.first, ti, tj);
  GemmParams p = sg_params(m.x, m.d, 1, m.y, m.d, 0, m.out, m.d, m.d, m.d, m.n);
  p.diag = 1.f / m.lam[0];
  p.alpha = -p.diag;
  p.tile_mode = TILE_LOWER_MIRROR;
  gemm_deep_tile<64, 64, 128>(p, ti, tj, 0, lds);
}

static int64_t sg_lower(int64_t n) { const int64_t T = (n + 63) / 64; return T * (T + 1) / 2; }
static int64_t sg_slices(int64_t d) { return (d + SG_SLICE - 1) / SG_SLICE; }

}  // namespace ak

extern "C" size_t ak_smw_group_y_floats(int64_t n, int64_t d) {
  if (n <= 0 || d <= 0) return 0;
  return static_cast<size_t>(std::max(n * d, ak::sg_slices(d) * ak::sg_lower(n) * 4096));
}

extern "C" int ak_smw_group(const int64_t* items, int count, int phase, ak_stream_t stream) {
  using namespace ak;
  if (items == nullptr || count <= 0 || (phase != 0 && phase != 1)) return AK_ERR_ARG;
  for (int i = 0; i < count; ++i) {
    const int64_t* r = items + 9 * i;
    for (int k = 0; k < 7; ++k)
      if (r[k] == 0) return AK_ERR_ARG;
    if (r[7] <= 0 || r[8] <= 0 || r[7] > 32768 || r[8] > (1 << 16)) return AK_ERR_ARG;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  for (int at = 0; at < count; at += SG_ITEMS) {
    SgArgs a;
    a.count = std::min(SG_ITEMS, count - at);
    auto launch = [&](void (*kernel)(SgArgs), auto groups_of) {
      int64_t w = 0;
      for (int i = 0; i < a.count; ++i) {
        a.item[i].first = static_cast<int>(w);
        w += groups_of(static_cast<int64_t>(a.item[i].n), static_cast<int64_t>(a.item[i].d));
      }
      if (w > (1 << 30)) return AK_ERR_TOO_LARGE;
      hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(w)), dim3(256), 0, s, a);
      return AK_OK;
    };
    for (int i = 0; i < a.count; ++i) {
      const int64_t* r = items + 9 * (at + i);
      SgItem& m = a.item[i];
      m.x = reinterpret_cast<const float*>(r[0]); m.gram = reinterpret_cast<float*>(r[1]);
      m.ginv = reinterpret_cast<const float*>(r[2]); m.y = reinterpret_cast<float*>(r[3]);
      m.out = reinterpret_cast<float*>(r[4]); m.lam = reinterpret_cast<const float*>(r[5]);
      m.lam_n = reinterpret_cast<float*>(r[6]);
      m.n = static_cast<int>(r[7]); m.d = static_cast<int>(r[8]);
      m.slices = static_cast<int>(sg_slices(r[8]));
    }
    int rc;
    if (phase == 0) {
      rc = launch(sg_gram_kernel, [](int64_t n, int64_t d) { return sg_lower(n) * sg_slices(d); });
      if (rc == AK_OK) rc = launch(sg_sum_kernel, [](int64_t n, int64_t) { return sg_lower(n); });
    } else {
      rc = launch(sg_solve_kernel, [](int64_t n, int64_t d) { return ((n + 63) / 64) * ((d + 63) / 64); });
      if (rc == AK_OK) rc = launch(sg_out_kernel, [](int64_t, int64_t d) { return sg_lower(d); });
    }
    if (rc != AK_OK) return rc;
  }
  return check_launch();
}
