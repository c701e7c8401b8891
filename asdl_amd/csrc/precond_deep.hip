// Kronecker preconditioning G <- s B_inv G A_inv, b <- s B_inv b of many small modules in two launches: 64 x 64 fp32 tiles
// (gemm_wave.hpp) for all products, the bias products and the 2 x 2 blocks of normalisation layers in work groups beside them.
//
// Bound by latency: a few dozen 64 x 64 tiles, K of a few hundred.  The split kernel's 128 x 128 tiles take 44 us for one
// product of 512 x 784 on a nearly idle device and need the operands' ranges first (two more launches); a tile of
// gemm_wave.hpp takes 2.3 us per 128 k.  The addresses travel in the kernel arguments: no table has to be built and uploaded per step.
// Any size and alignment; the gradients of a call have to be distinct (nothing orders two items of a launch).  MLP 784-512-512-10
// (three modules with bias): 8 launches, 160 us -> 2 launches, 17 and 22 us
// (25 and 34 with tiles staged through the LDS).
#include <algorithm>
#include "gemm_f32.hpp"

namespace ak {

constexpr int KP_ITEMS = 24;             // modules of one launch
// Sizes of a module and of a unit (24 of each stay far below 2^31 work groups).  Wider ones are left to the caller's other paths.
constexpr int64_t KP_MAX_ROWS = 32768, KP_MAX_COLUMNS = 1 << 20, KP_MAX_UNIT = 1 << 24;
constexpr int KP_GEMV_ROWS = 16;         // rows of a bias product per work group

struct KpItem {
  const float* B;
  const float* A;
  float* G;
  float* b;                              // null: no bias
  float* T;                              // B_inv G
  float* tb;                             // B_inv b
  int dB, dA;
  int first, bias_first;                 // first work group of the products' tiles, and of the bias' rows behind them
};
struct KpUnit {
  const float* inv;                      // [F][2][2]
  float* gw;
  float* gb;
  int F, first;
};
struct KpArgs {
  int count, units, end;                 // end: work groups of the modules; those of the units follow
  float scale;
  const int* fail0;                      // device words: nothing is written if one of them is not zero
  const int* fail1;
  KpItem item[KP_ITEMS];
  KpUnit unit[KP_ITEMS];
};

__device__ __forceinline__ GemmParams kp_product(const float* A, const float* B, float* C, int M, int N, int K,
                                                 float alpha) {
  GemmParams p;
  p.A = A; p.B = B; p.C = C;
  p.lda = K; p.ldb = N; p.ldc = N;
  p.M = M; p.N = N; p.K = K;
  p.transA = 0; p.transB = 0;
  p.alpha = alpha; p.beta = 0.f;
  p.kmode = K_FULL; p.tile_mode = TILE_ALL;
  return p;
}

__device__ __forceinline__ int kp_item_of(const KpArgs& a, int w) {
  int i = 0;
  while (i + 1 < a.count && a.item[i + 1].first <= w) ++i;
  return i;
}

// T <- B_inv G, tb <- B_inv b
static __global__ __launch_bounds__(64 * GEMM_WAVES, 2) void kp_first_kernel(KpArgs a) {
  __shared__ __attribute__((aligned(16))) float lds[wave_lds_floats<GEMM_WAVES>()];
  const int w = blockIdx.x;
  const KpItem& m = a.item[kp_item_of(a, w)];
  if (w < m.bias_first) {
    const int tn = (m.dA + 63) / 64, local = w - m.first;
    gemm_wave_tile<GEMM_WAVES>(kp_product(m.B, m.G, m.T, m.dB, m.dA, m.dB, 1.f), local / tn, local % tn, 0, lds);
    return;
  }
  constexpr int ROWS = KP_GEMV_ROWS / GEMM_WAVES;
  const int lane = threadIdx.x & 63, row0 = (w - m.bias_first) * KP_GEMV_ROWS + (threadIdx.x >> 6) * ROWS;
  float s[ROWS] = {};
  for (int k = lane; k < m.dB; k += 64) {
    const float x = m.b[k];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) s[r] += m.B[static_cast<int64_t>(min(row0 + r, m.dB - 1)) * m.dB + k] * x;
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s[r] += __shfl_xor(s[r], o);
    if (lane == 0 && row0 + r < m.dB) m.tb[row0 + r] = s[r];
  }
}

// G <- s T A_inv, b <- s tb
static __global__ __launch_bounds__(64 * GEMM_WAVES, 2) void kp_second_kernel(KpArgs a) {
  __shared__ __attribute__((aligned(16))) float lds[wave_lds_floats<GEMM_WAVES>()];
  if ((a.fail0 != nullptr && *a.fail0 != 0) || (a.fail1 != nullptr && *a.fail1 != 0)) return;
  const int w = blockIdx.x;
  if (w >= a.end) {
    int i = 0;
    while (i + 1 < a.units && a.unit[i + 1].first <= w) ++i;
    const KpUnit& u = a.unit[i];
    const int f = (w - u.first) * 256 + threadIdx.x;
    if (threadIdx.x >= 256 || f >= u.F) return;
    const floatx4 v = *reinterpret_cast<const floatx4*>(u.inv + 4 * static_cast<int64_t>(f));
    const float x = u.gw[f] * a.scale, y = u.gb[f] * a.scale;
    u.gw[f] = v[0] * x + v[1] * y;
    u.gb[f] = v[2] * x + v[3] * y;
    return;
  }
  const KpItem& m = a.item[kp_item_of(a, w)];
  if (w < m.bias_first) {
    const int tn = (m.dA + 63) / 64, local = w - m.first;
    gemm_wave_tile<GEMM_WAVES>(kp_product(m.T, m.A, m.G, m.dB, m.dA, m.dA, a.scale), local / tn, local % tn, 0, lds);
    return;
  }
  const int row = (w - m.bias_first) * KP_GEMV_ROWS + threadIdx.x;
  if (threadIdx.x < KP_GEMV_ROWS && row < m.dB) m.b[row] = a.scale * m.tb[row];
}

static int64_t kp_tiles(int64_t dB, int64_t dA) { return ((dB + 63) / 64) * ((dA + 63) / 64); }

// The rule: microseconds of both products on 64 x 64 tiles against those on the split kernel, whose rates gemm_f32.hpp and
// chol_group.hip use too (64 x 64: 2 us per chunk of 128 k; split: 1.6 us per k-tile of 32, 1 us once the device is full, and
// 20 us for the ranges of its operands).  784-512-512-10 39 us here and 132 split, 2000^3 172 us a product here and 85 split.
static bool kp_faster(const int64_t* items, int count) {
  double longest = 0, chunks = 0, long_tile = 0, ktiles = 0;
  for (int i = 0; i < count; ++i) {
    const int64_t dB = items[6 * i + 4], dA = items[6 * i + 5];
    for (const int64_t K : {dB, dA}) {
      const double c = static_cast<double>((K + 127) / 128), t = static_cast<double>((K + 31) / 32);
      longest = std::max(longest, c);
      long_tile = std::max(long_tile, t);
      chunks += c * static_cast<double>(kp_tiles(dB, dA));
      ktiles += t * static_cast<double>(((dB + 127) / 128) * ((dA + 127) / 128));
    }
  }
  return 2.0 * std::max(2 * longest, chunks / 256) <= std::max(2 * 1.6 * long_tile, ktiles / 256) + 20;
}

}  // namespace ak

extern "C" size_t ak_kron_precond_deep_ws_bytes(const int64_t* items, int count) {
  size_t floats = 0;
  for (int i = 0; i < count; ++i) floats += static_cast<size_t>(items[6 * i + 4]) * items[6 * i + 5] + items[6 * i + 4];
  return floats * sizeof(float);
}

extern "C" int ak_kron_precond_deep_faster(const int64_t* items, int count) {
  if (count < 0 || (count > 0 && items == nullptr)) return AK_ERR_ARG;
  for (int i = 0; i < count; ++i)
    if (items[6 * i + 4] <= 0 || items[6 * i + 5] <= 0) return AK_ERR_ARG;
  return ak::kp_faster(items, count) ? 1 : 0;
}

extern "C" int ak_kron_precond_deep(const int64_t* items, int count, const int64_t* units, int unit_count, float grad_scale,
                                    const int* fail0, const int* fail1, int only_if_faster, void* ws, size_t ws_bytes,
                                    ak_stream_t stream) {
  using namespace ak;
  if (count < 0 || unit_count < 0 || (count > 0 && items == nullptr) || (unit_count > 0 && units == nullptr)) return AK_ERR_ARG;
  for (int i = 0; i < count; ++i) {
    const int64_t* r = items + 6 * i;
    if (r[0] == 0 || r[1] == 0 || r[2] == 0 || r[4] <= 0 || r[5] <= 0) return AK_ERR_ARG;
    if (r[4] > KP_MAX_ROWS || r[5] > KP_MAX_COLUMNS) return AK_ERR_UNSUPPORTED;
  }
  for (int i = 0; i < unit_count; ++i) {        // (all of them before the first launch)
    const int64_t* r = units + 4 * i;
    if (r[0] == 0 || r[1] == 0 || r[2] == 0 || r[3] <= 0) return AK_ERR_ARG;
    if (r[3] > KP_MAX_UNIT) return AK_ERR_UNSUPPORTED;
  }
  if (only_if_faster && !kp_faster(items, count)) return AK_ERR_UNSUPPORTED;
  if (count > 0 && (ws == nullptr || ws_bytes < ak_kron_precond_deep_ws_bytes(items, count))) return AK_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* t = static_cast<float*>(ws);
  int at = 0, unit_at = 0;
  while (at < count || unit_at < unit_count) {
    KpArgs a;
    a.count = std::min(KP_ITEMS, count - at);
    a.units = std::min(KP_ITEMS, unit_count - unit_at);
    a.scale = grad_scale; a.fail0 = fail0; a.fail1 = fail1;
    int64_t w = 0;
    for (int i = 0; i < a.count; ++i, ++at) {
      const int64_t* r = items + 6 * at;
      KpItem& m = a.item[i];
      m.B = reinterpret_cast<const float*>(r[0]); m.A = reinterpret_cast<const float*>(r[1]);
      m.G = reinterpret_cast<float*>(r[2]); m.b = reinterpret_cast<float*>(r[3]);
      m.dB = static_cast<int>(r[4]); m.dA = static_cast<int>(r[5]);
      m.T = t; t += r[4] * r[5];
      m.tb = t; t += r[4];
      m.first = static_cast<int>(w);
      w += kp_tiles(r[4], r[5]);
      m.bias_first = static_cast<int>(w);
      if (m.b != nullptr) w += (r[4] + KP_GEMV_ROWS - 1) / KP_GEMV_ROWS;
    }
    a.end = static_cast<int>(w);
    for (int i = 0; i < a.units; ++i, ++unit_at) {
      const int64_t* r = units + 4 * unit_at;
      KpUnit& u = a.unit[i];
      u.inv = reinterpret_cast<const float*>(r[0]); u.gw = reinterpret_cast<float*>(r[1]); u.gb = reinterpret_cast<float*>(r[2]);
      u.F = static_cast<int>(r[3]); u.first = static_cast<int>(w);
      w += (r[3] + 255) / 256;
    }
    if (a.end > 0) hipLaunchKernelGGL(kp_first_kernel, dim3(a.end), dim3(64 * GEMM_WAVES), 0, s, a);
    if (w > 0) hipLaunchKernelGGL(kp_second_kernel, dim3(static_cast<unsigned>(w)), dim3(64 * GEMM_WAVES), 0, s, a);
  }
  return check_launch();
}
