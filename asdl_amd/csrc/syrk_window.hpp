// Input factor of a convolution of any window, stride and padding on an fp32 NCHW input, without an unfolded copy and without
// staging: syrk_wave.hpp's work groups (64 x 64 tile, a quarter of the positions per wave) whose operand loads gather.
//
// Element (position k, column i) of the unfolded matrix is x[base(k) + column(i)], or zero where the window's tap lies in the
// padding.  A work group writes base(k) and the mask of valid taps of its positions to the LDS once; a lane owns columns, so it
// has their offsets and tap bits in registers, and a load costs two additions, a test and a select.  Loads go through a buffer
// descriptor: an offset out of range reads as zero.  Bound by these gathers (a lane's 4 bytes each) beside the fp32 matrix
// instruction.  us, staged (conv_syrk_kernel) and here: 3 x 3 / 2 of
// 128 x 64 x 32 x 32 273 and 229, 128 x 256 x 8 x 8 484 and 185, 64 x 128 x 56 x 56 1974 and 1103; 3 x 3 of 64 x 48 x 20 x 20 153
// and 86; 1 x 1 / 2 of 128 x 256 x 8 x 8 76 and 20.
#pragma once
#include "syrk_wave.hpp"

namespace ak {

constexpr int SWIN_MAX_K = 4096;                 // positions of a work group: 8 bytes each

struct SyrkWindowParams {
  SyrkWaveParams w;                              // K: positions, per_split: positions of a work group
  int64_t image;                                 // elements of an image
  int64_t images_bytes;                          // bytes of the whole input
  int H, W, Ho, Wo, kh, kw, sh, sw, ph, pw;
  uint32_t mWo, mHo;                             // fastdiv: positions of a work group, rows
};

template <bool DIAG>
__device__ __forceinline__ void syrk_window_sum(floatx16 (&tot)[2][2], __amdgpu_buffer_rsrc_t rsrc, const uint32_t* table, int k, int k1,
                                                const uint32_t (&col)[4], const uint32_t (&tap)[4], int g) {
  constexpr int NC = DIAG ? 2 : 4, CHUNK = 8;
  struct Entries { uint32_t v[16]; };            // (base, mask) of this half's 8 of the batch's 16 positions
  struct Batch { float x[8][NC]; };
  auto entries = [&](Entries& e, int at) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint4 q = *reinterpret_cast<const uint4*>(table + 2 * (at + 8 * t + 4 * g + 2 * h));
        e.v[8 * t + 4 * h] = q.x; e.v[8 * t + 4 * h + 1] = q.y; e.v[8 * t + 4 * h + 2] = q.z; e.v[8 * t + 4 * h + 3] = q.w;
      }
  };
  auto fetch = [&](Batch& f, const Entries& e) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const uint32_t off = (e.v[2 * u + 1] & tap[c]) != 0 ? e.v[2 * u] + col[c] : 0xFFFFFF00u;
        f.x[u][c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, 0, 0));
      }
  };
  floatx16 acc[2][2];
  auto clear = [&] {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
  };
  auto flush = [&] {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[a][b][r] += acc[a][b][r];
  };
  auto multiply = [&](const Batch& f) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          if (!DIAG || a <= b) acc[a][b] = mfma_f32(f.x[u][a], f.x[u][NC - 2 + b], acc[a][b]);
  };
  const int batches = k < k1 ? (k1 - k + 15) / 16 : 0;       // (positions beyond the last one have an empty mask)
  if (batches == 0) return;
  Entries e;
  Batch f0, f1;
  entries(e, k);
  fetch(f0, e);
  entries(e, k + 16 * min(1, batches - 1));
  for (int b0 = 0; b0 < batches; b0 += CHUNK) {
    clear();
    const int b1 = min(b0 + CHUNK, batches);
    int b = b0;
    for (; b + 2 <= b1; b += 2) {                // (always a fetch, at the end of the last batch again)
      fetch(f1, e);
      entries(e, k + 16 * min(b + 2, batches - 1));
      __builtin_amdgcn_sched_barrier(0);
      multiply(f0);
      __builtin_amdgcn_sched_barrier(0);
      fetch(f0, e);
      entries(e, k + 16 * min(b + 3, batches - 1));
      __builtin_amdgcn_sched_barrier(0);
      multiply(f1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (b < b1) multiply(f0);                    // (the last batch of an odd number)
    flush();
  }
}

static __global__ __launch_bounds__(256, 2) void syrk_window_kernel(SyrkWindowParams q) {
  __shared__ __attribute__((aligned(16))) uint32_t smem[16384];       // the positions' table, then the waves' sums
  const SyrkWaveParams& p = q.w;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t id = xcd_contiguous_id(blockIdx.x, gridDim.x), ntiles = static_cast<uint32_t>(p.T * (p.T + 1) / 2);
  const uint32_t split = id / ntiles, tile = id - split * ntiles;
  int ti, tj;
  decode_upper_tile(static_cast<int>(tile), p.T, ti, tj);
  const bool diag = ti == tj;
  const int i0 = 64 * ti, j0 = 64 * tj;
  const int64_t first = static_cast<int64_t>(split) * p.per_split;
  const int per = static_cast<int>(p.per_split), count = static_cast<int>(p.K - first < per ? p.K - first : per);
  // positions first ... first + per - 1, from the image of the first one on
  const int HoWo = q.Ho * q.Wo;
  const int64_t n0 = first / HoWo;
  const int rest0 = static_cast<int>(first - n0 * HoWo);
  for (int k = tid; k < per; k += 256) {
    uint32_t base = 0, mask = 0;
    if (k < count) {
      const uint32_t pos = static_cast<uint32_t>(rest0 + k), row = fastdiv(pos, q.mWo, static_cast<uint32_t>(q.Wo));
      const uint32_t n = fastdiv(row, q.mHo, static_cast<uint32_t>(q.Ho));
      const int y = static_cast<int>(row - n * q.Ho) * q.sh - q.ph, x = static_cast<int>(pos - row * q.Wo) * q.sw - q.pw;
      uint32_t xs = 0;
      for (int kx = 0; kx < q.kw; ++kx) xs |= static_cast<uint32_t>(x + kx >= 0 && x + kx < q.W) << kx;
      for (int ky = 0; ky < q.kh; ++ky)
        if (y + ky >= 0 && y + ky < q.H) mask |= xs << (ky * q.kw);
      base = (n * static_cast<uint32_t>(q.image) + static_cast<uint32_t>(y * q.W + x)) * 4u;     // (wraps where the taps make up for it)
    }
    smem[2 * k] = base;
    smem[2 * k + 1] = mask;
  }
  // the descriptor begins at the first position's image; the launcher has checked that the images of a work group fit
  const int64_t left = q.images_bytes - n0 * q.image * 4;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(p.X) + n0 * q.image, 0, static_cast<int>(left < 0x7FFFFFFF ? left : 0x7FFFFFFF), 0x00020000);
  uint32_t col[4], tap[4];
  const uint32_t KK = static_cast<uint32_t>(q.kh * q.kw);
#pragma unroll
  for (int c = 0; c < 4; ++c) {                  // columns beyond the matrix read the last one: their sums are not stored
    const uint32_t i = static_cast<uint32_t>(min((c < 2 ? i0 : j0) + 32 * (c & 1) + l32, p.d - 1));
    const uint32_t ch = i / KK, t = i - ch * KK, ky = t / static_cast<uint32_t>(q.kw), kx = t - ky * static_cast<uint32_t>(q.kw);
    col[c] = (ch * static_cast<uint32_t>(q.H * q.W) + ky * static_cast<uint32_t>(q.W) + kx) * 4u;
    tap[c] = 1u << t;
  }
  floatx16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
  __syncthreads();
  const int quarter = per / 4, k = wave * quarter, k1 = min(k + quarter, count);
  if (diag) syrk_window_sum<true>(acc, rsrc, smem, k, k1, col, tap, g);
  else syrk_window_sum<false>(acc, rsrc, smem, k, k1, col, tap, g);
  __syncthreads();
  syrk_wave_finish(acc, reinterpret_cast<floatx4(*)[4][4][64]>(smem), p, id, i0, j0, diag);
}

// Positions of a work group, at most what the table holds, and at most 1024 where the partial sums stay below 64 MB: two work groups
// of a CU hide each other's gathers, and a matrix of a round or less would have one.  Even parts: the model of syrk_wave_split
// chooses among the splits that fit (a split of its own choice, cut to 4096, left a short one as a round of its own).
// us, staged, cut to 4096 and here: 3 x 3 of 64 x 100 x 14 x 14 without padding 168, 220 and 138; 128 x 256 x 8 x 8 550, 586 and 335;
// with padding 128 x 96 x 8 x 8 110, 112 and 103; 5 x 5 of 16 x 24 x 56 x 56 332, 379 and 295.
inline int64_t syrk_window_per_split(int64_t d, int64_t K, int64_t* nsplit) {
  const int64_t T = (d + 63) / 64, tiles = T * (T + 1) / 2;
  const int64_t most = tiles * ((K + 1023) / 1024) <= 4096 ? 1024 : SWIN_MAX_K;
  const int64_t s = syrk_wave_split(d, K, (K + most - 1) / most);
  const int64_t per = ((K + s - 1) / s + 63) / 64 * 64;
  *nsplit = (K + per - 1) / per;
  return per;
}
inline bool syrk_window_ok(int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int64_t Ho, int64_t Wo) {
  // (32-bit arithmetic of a work group: its positions span (4096 / (Ho Wo) + 2) images)
  const int64_t image = C * H * W, span = SWIN_MAX_K / (Ho * Wo) + 2;
  return kh * kw <= 32 && Ho > 0 && Wo > 0 && Ho * Wo < (1 << 24) && (Ho * Wo + SWIN_MAX_K) * std::max(Ho, Wo) < (1ll << 32) && span * image * 4 < (1ll << 31) - 4096 && C * kh * kw < (1 << 20) &&
         N * Ho * Wo < (1ll << 40);
}
// The staged kernel stays for strided 1 x 1 windows of many products: a lane's every load is a line of its own there (staged and
// here, us: 32 x 300 x 14 x 14 86 and 18 (15 tiles), 32 x 1024 x 14 x 14 132 and 143, 64 x 256 x 56 x 56 124 and 147).  Of 241 other
// windows (3 x 3 and 5 x 5, strides 1 and 2, 24 to 256 channels) none is more than 1 % slower here (3 x 3 of 32 x 96 x 16 x 16 117.3
// and 117.5).
inline bool syrk_window_faster(int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int64_t Ho, int64_t Wo) {
  if (!syrk_window_ok(N, C, H, W, kh, kw, Ho, Wo)) return false;
  const int64_t T = (C * kh * kw + 63) / 64, work = T * (T + 1) / 2 * N * Ho * Wo;
  return kh * kw > 1 || (sh == 1 && sw == 1) || work <= 700 * 256;
}
inline size_t syrk_window_ws_bytes(int64_t d, int64_t K) {
  int64_t s;
  syrk_window_per_split(d, K, &s);
  const int64_t T = (d + 63) / 64;
  return s > 1 ? static_cast<size_t>(s) * (T * (T + 1) / 2) * 4096 * sizeof(float) : 0;
}

inline int launch_syrk_window(const float* X, int64_t N, int64_t C, int64_t H, int64_t W, int kh, int kw, int sh, int sw, int ph, int pw,
                              int64_t Ho, int64_t Wo, float alpha, float beta, float* A, int64_t lda, void* ws, size_t ws_bytes,
                              hipStream_t stream) {
  SyrkWindowParams q;
  SyrkWaveParams& p = q.w;
  const int64_t d = C * kh * kw, K = N * Ho * Wo, T = (d + 63) / 64, tiles = T * (T + 1) / 2;
  int64_t s;
  p.per_split = syrk_window_per_split(d, K, &s);
  if (s > 1 && (ws == nullptr || ws_bytes < static_cast<size_t>(s) * tiles * 4096 * sizeof(float))) return AK_ERR_WORKSPACE;
  if (tiles * s >= (1ll << 31)) return AK_ERR_UNSUPPORTED;
  p.X = X; p.ld = 0; p.sn = 0; p.K = K; p.d = static_cast<int>(d); p.run = 0; p.T = static_cast<int>(T); p.nsplit = static_cast<int>(s);
  p.alpha = alpha; p.beta = beta; p.C = A; p.ldc = lda; p.ws = static_cast<float*>(ws);
  q.image = C * H * W; q.images_bytes = N * q.image * 4;
  q.H = static_cast<int>(H); q.W = static_cast<int>(W); q.Ho = static_cast<int>(Ho); q.Wo = static_cast<int>(Wo);
  q.kh = kh; q.kw = kw; q.sh = sh; q.sw = sw; q.ph = ph; q.pw = pw;
  q.mWo = make_magic(q.Wo); q.mHo = make_magic(q.Ho);
  hipLaunchKernelGGL(syrk_window_kernel, dim3(static_cast<unsigned>(tiles * s)), dim3(256), 0, stream, q);
  if (s > 1) launch_syrk_finalize<1>(p.ws, p.nsplit, tiles, p.T, A, lda, d, alpha, beta, stream);
  return check_launch();
}

}  // namespace ak
