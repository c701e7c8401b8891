// C <- beta C + alpha sum over k of x_k x_k^T in true fp32 for fp32 rows, straight from memory to the matrix instruction.
//
// A work group owns a 64 x 64 tile of the upper triangle and a range of k, each of its four waves a quarter of the range and
// the whole tile: 2 + 2 operand values per lane feed four v_mfma_f32_32x32x2_f32 (256 cycles), which the L1 delivers in a fraction
// of that, so that there is no staging, no barrier before the sums and every load of a batch is in flight at once.  The four
// waves' tiles are added through the LDS.  Two ways the k lie in memory:
//   rows     element (k, i) at X[k ld + i]  (Linear inputs, G^T G): a lane of half g takes k = 2 u + g of column i
//   runs     element (k, i) at X[n sn + i ld + p], k = n run + p, runs of a multiple of 8 (1 x 1 windows of NCHW, G G^T): a lane
//            takes four consecutive k, k = 8 t + 4 g + e
//
// Bound by latency for few k (launch 2 us, one round of loads 2, 0.85 us of matrix instructions per 64 k of a work group, sums and
// stores 1.5), by the fp32 matrix instruction else.  Measured, before (128 x 128 tiles staged through the LDS) and now, us: rows of
// 128 x 784 18 and 7, 1000 x 1021 33 and 25, 4096 x 512 31 and 19, 70000 x 40 42 and 14; 1 x 1 windows of 128 x 64 x 32 x 32
// 32 and 17, 128 x 512 x 4 x 4 35 and 13, one 512 x 784 matrix 55 and 14, 128 x 512 x 32 x 32 607 and 349.
#pragma once
#include <algorithm>
#include "common.hpp"

namespace ak {

struct SyrkWaveParams {
  const float* X;
  int64_t ld, sn, K, per_split;      // per_split: k of a work group, a multiple of 64
  int d, run, T, nsplit;             // run: 0 for rows
  float alpha, beta;
  float* C;
  int64_t ldc;
  float* ws;
};

// One wave's 64 x 64 sums over k in [k, k1), in chunks of 128 k that are added to a running total (a sum of hundreds of
// roundings in a row shows).  at[c]: lane offsets of the two column blocks of the tile's rows and the two of its columns.
template <bool RUNS, bool DIAG>
__device__ __forceinline__ void syrk_wave_sum(floatx16 (&tot)[2][2], const SyrkWaveParams& p, int64_t k, int64_t k1, const uint32_t (&at)[4],
                                              int g) {
  constexpr int NC = DIAG ? 2 : 4, U = 8, CHUNK = 8;      // a batch is 16 k: U pairs (rows), two groups of 8 (runs); batches of a chunk
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
  auto products = [&](const float (&x)[NC]) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        if (!DIAG || a <= b) acc[a][b] = mfma_f32(x[a], x[NC - 2 + b], acc[a][b]);      // (the lower block of a diagonal tile: below)
  };
  int64_t n = 0;
  int pos = 0;
  const float* __restrict__ src = p.X;
  if constexpr (RUNS) {
    n = k / p.run;
    pos = static_cast<int>(k - n * p.run);
    src += n * p.sn;
  } else {
    src += k * p.ld;
  }
  struct Batch { float x[2 * U][NC]; };          // rows: x[u] pair u; runs: x[4 t + e] element e of group t
  auto fetch_group = [&](Batch& f, int t) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const floatx4 v = *reinterpret_cast<const floatx4*>(src + pos + at[c]);
#pragma unroll
      for (int e = 0; e < 4; ++e) f.x[4 * t + e][c] = v[e];
    }
    pos += 8;
    if (pos == p.run) {
      pos = 0;
      src += p.sn;
    }
  };
  auto fetch = [&](Batch& f) {
    if constexpr (RUNS) {
      fetch_group(f, 0);
      fetch_group(f, 1);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < NC; ++c) f.x[u][c] = (src + 2 * u * p.ld)[at[c]];
      src += 2 * U * p.ld;
    }
  };
  auto multiply = [&](const Batch& f, int steps) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < steps) products(f.x[u]);
  };
  const int batches = k < k1 ? static_cast<int>((k1 - k) / 16) : 0, rest = k < k1 ? static_cast<int>((k1 - k) % 16) : 0;
  Batch f0, f1;
  if (batches > 0) fetch(f0);
  for (int b0 = 0; b0 < batches; b0 += CHUNK) {
    clear();
    const int b1 = min(b0 + CHUNK, batches);
    int b = b0;
    for (; b + 2 <= b1; b += 2) {
      const float* __restrict__ src1 = src;
      const int pos1 = pos;
      fetch(f1);
      __builtin_amdgcn_sched_barrier(0);         // (all loads of a batch leave before the products of the one before)
      multiply(f0, U);
      __builtin_amdgcn_sched_barrier(0);
      // (always a fetch, at the end of f1's batch again: one under a condition would make every use wait for all loads)
      const float* __restrict__ src2 = src;
      const int pos2 = pos;
      const bool last = b + 2 == batches;
      if (last) { src = src1; pos = pos1; }
      fetch(f0);
      if (last) { src = src2; pos = pos2; }
      __builtin_amdgcn_sched_barrier(0);
      multiply(f1, U);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (b < b1) multiply(f0, U);                  // (the last batch of an odd number)
    flush();
  }
  if (rest > 0) {
    clear();
    if constexpr (RUNS) {                         // a group of 8
      fetch_group(f0, 0);
      multiply(f0, 4);
    } else {                                      // rows beyond the range read its last one and count as zeros
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float* __restrict__ row = src + min(2 * u, rest - 1) * p.ld;
        const uint32_t back = 2 * u + 1 >= rest && g == 1 ? static_cast<uint32_t>(p.ld) : 0u;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const float v = row[at[c] - back];
          f0.x[u][c] = 2 * u + g < rest ? v : 0.f;
        }
      }
      multiply(f0, U);
    }
    flush();
  }
}

// Adds the four waves' sums of a tile and stores them: wave w block w.  part: 64 KB of LDS; id: the tile's place in the partial sums.
__device__ __forceinline__ void syrk_wave_finish(const floatx16 (&acc)[2][2], floatx4 (*part)[4][4][64], const SyrkWaveParams& p, uint32_t id,
                                                 int i0, int j0, bool diag) {
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        part[wave][2 * a + b][q][lane] = floatx4{acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]};
  __syncthreads();
  const int wr = wave >> 1, wc = wave & 1;
  floatx16 sum[1][1];
  if (diag && wave == 2) {           // block (1, 0) of a diagonal tile is block (0, 1) transposed: element (r, c) is its (c, r)
    const float* flat = reinterpret_cast<const float*>(&part[0][1][0][0]);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      // element (row l32, column 8 (r / 4) + 4 g + r % 4) of block (0, 1): quad l32 / 8, lane 32 (l32 / 4 % 2) + column, entry l32 % 4
      const int at01 = ((l32 >> 3) * 64 + 32 * ((l32 >> 2) & 1) + 8 * (r >> 2) + 4 * g + (r & 3)) * 4 + (l32 & 3);
      sum[0][0][r] = (flat[at01] + flat[at01 + 4096]) + (flat[at01 + 8192] + flat[at01 + 12288]);
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const floatx4 v = (part[0][wave][q][lane] + part[1][wave][q][lane]) + (part[2][wave][q][lane] + part[3][wave][q][lane]);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum[0][0][4 * q + e] = v[e];
    }
  }
  if (p.nsplit == 1) syrk_epilogue<1, 1>(sum, p.C, p.ldc, p.d, i0 + 32 * wr, j0 + 32 * wc, diag, p.alpha, p.beta, lane);
  else store_partial<1, 1>(sum, p.ws + static_cast<size_t>(id) * 4096, tid);
}

template <bool RUNS>
static __global__ __launch_bounds__(256, 2) void syrk_wave_kernel(SyrkWaveParams p) {
  __shared__ __attribute__((aligned(16))) floatx4 part[4][4][4][64];
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the tiles of one split, which read the same rows, share an L2
  const uint32_t id = xcd_contiguous_id(blockIdx.x, gridDim.x), ntiles = static_cast<uint32_t>(p.T * (p.T + 1) / 2);
  const uint32_t split = id / ntiles, tile = id - split * ntiles;
  int ti, tj;
  decode_upper_tile(static_cast<int>(tile), p.T, ti, tj);
  const bool diag = ti == tj;
  const int i0 = 64 * ti, j0 = 64 * tj;
  const int64_t quarter = p.per_split / 4;
  const int64_t k = static_cast<int64_t>(split) * p.per_split + wave * quarter;
  const int64_t k1 = k + quarter < p.K ? k + quarter : p.K;
  // columns beyond the matrix read the last one: their sums are not stored
  uint32_t at[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int col = min((c < 2 ? i0 : j0) + 32 * (c & 1) + l32, p.d - 1);
    at[c] = RUNS ? static_cast<uint32_t>(col * static_cast<int>(p.ld) + 4 * g) : static_cast<uint32_t>(g * static_cast<int>(p.ld) + col);
  }
  floatx16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
  if (diag) syrk_wave_sum<RUNS, true>(acc, p, k, k1, at, g);
  else syrk_wave_sum<RUNS, false>(acc, p, k, k1, at, g);
  syrk_wave_finish(acc, part, p, id, i0, j0, diag);
}

// The same result with the staged kernels' order of sums (AK_F32_IN_ORDER): their splits of K, one accumulator over each of
// them, the k of an instruction paired as there (rows: 2 u and 2 u + 1; runs: 16 t + m and 16 t + 8 + m).  A work group owns a
// 64 x 64 tile of one split, a wave a 32 x 32 block of it.  Bound by the chain of matrix instructions (64 cycles per two k) behind
// one way to memory, 64 k of both operands in flight.  us, staged and here:
// one 512 x 784 matrix 55 and 14, 767 x 3072 53 and 46, rows of 512 x 512 18.7 and 11.6.
template <bool RUNS, bool MASK>
__device__ __forceinline__ void syrk_chain_fetch(float (&x)[32], const float* __restrict__ X, int64_t ld, uint32_t at, int64_t k, int64_t k1,
                                                 int g) {
  if constexpr (RUNS) {                       // X: the matrix, at: the lane's row and 8 g; k1 - k a multiple of 8
    const float* __restrict__ src = X + k;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int over = MASK ? 16 * t + 8 * g - static_cast<int>(k1 - k - 8) : 0;       // beyond the range: its last eight
      const int back = over > 0 ? over : 0;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const floatx4 v = *reinterpret_cast<const floatx4*>(src + 16 * t + 4 * h + (static_cast<int64_t>(at) - back));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[8 * t + 4 * h + e] = back > 0 ? 0.f : v[e];
      }
    }
  } else {                                    // at: the lane's column and g rows
    const float* __restrict__ src = X + k * ld;
#pragma unroll
    for (int u = 0; u < 32; ++u) {
      const int over = MASK ? 2 * u + g - static_cast<int>(k1 - k - 1) : 0;
      const int back = over > 0 ? over : 0;
      const float v = (src + 2 * u * ld)[static_cast<int64_t>(at) - back * ld];
      x[u] = back > 0 ? 0.f : v;
    }
  }
}

template <bool RUNS>
static __global__ __launch_bounds__(256, 2) void syrk_chain_kernel(SyrkWaveParams p) {
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 1, wc = wave & 1;
  const uint32_t ntiles = static_cast<uint32_t>(p.T * (p.T + 1) / 2), split = blockIdx.x / ntiles, tile = blockIdx.x - split * ntiles;
  int ti, tj;
  decode_upper_tile(static_cast<int>(tile), p.T, ti, tj);
  const int i0 = 64 * ti + 32 * wr, j0 = 64 * tj + 32 * wc;
  const int64_t k0 = static_cast<int64_t>(split) * p.per_split, k1 = k0 + p.per_split < p.K ? k0 + p.per_split : p.K;
  auto lane_offset = [&](int c0) {            // columns beyond the matrix read the last one: their sums are not stored
    const int col = min(c0 + l32, p.d - 1);
    return RUNS ? static_cast<uint32_t>(col) * static_cast<uint32_t>(p.ld) + 8 * g : g * static_cast<uint32_t>(p.ld) + col;
  };
  const uint32_t ai = lane_offset(i0), aj = lane_offset(j0);
  floatx16 acc[1][1];
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[0][0][r] = 0.f;
  struct Batch { float a[32], b[32]; };
  auto fetch = [&](Batch& f, int64_t k) {
    syrk_chain_fetch<RUNS, false>(f.a, p.X, p.ld, ai, k, k1, g);
    syrk_chain_fetch<RUNS, false>(f.b, p.X, p.ld, aj, k, k1, g);
  };
  auto multiply = [&](const Batch& f) {
#pragma unroll
    for (int u = 0; u < 32; ++u) acc[0][0] = mfma_f32(f.a[u], f.b[u], acc[0][0]);
  };
  const int batches = static_cast<int>((k1 - k0) / 64);
  Batch f0, f1;
  if (batches > 0) {
    // (always a fetch, of the last batch again at the end: one under a condition would make every use wait for all loads)
    fetch(f0, k0);
    int b = 0;
    for (; b + 2 <= batches; b += 2) {
      fetch(f1, k0 + 64 * (b + 1));
      __builtin_amdgcn_sched_barrier(0);
      multiply(f0);
      __builtin_amdgcn_sched_barrier(0);
      fetch(f0, k0 + 64 * static_cast<int64_t>(min(b + 2, batches - 1)));
      __builtin_amdgcn_sched_barrier(0);
      multiply(f1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (b < batches) multiply(f0);
  }
  if (k0 + 64 * batches < k1) {
    const int64_t k = k0 + 64 * batches;
    syrk_chain_fetch<RUNS, true>(f0.a, p.X, p.ld, ai, k, k1, g);
    syrk_chain_fetch<RUNS, true>(f0.b, p.X, p.ld, aj, k, k1, g);
    multiply(f0);
  }
  if (p.nsplit == 1) syrk_epilogue<1, 1>(acc, p.C, p.ldc, p.d, i0, j0, ti == tj, p.alpha, p.beta, lane);
  else store_partial<1, 1>(acc, p.ws + static_cast<size_t>(blockIdx.x) * 4096, tid);
}

// Rows: up to 176 k of tiles a CU; beyond that the loads of 32 columns of a row count (staged and here, us: 512 x 767 28 and 21,
// 700 x 600 24 and 22, 1000 x 700 27.5 and 28, 2000 x 512 24 and 27, 2000 x 700 38 and 47).  Runs, read in 16-byte loads, go to the
// chain at every size: of 55 matrices of 30 to 4096 x 784 to 16384 one of 1536 x 1536 and one of 1536 x 2304 lose 5 % (81 and 86 us,
// 110 and 115), 767 and 1024 x 16384 4 and 3 %, the others gain (512 x 784 55 and 14, 1024 x 3072 77 and 74, 3072 x 3072 591 and
// 510, 4096 x 16384 6006 and 4350).
inline bool syrk_chain_rows(int64_t d, int64_t K) {
  const int64_t T = (d + 63) / 64;
  return T * (T + 1) / 2 * K <= 176 * 256;
}

// The staged kernels' plan: nsplit ranges of per_split k.  runs: rows of K contiguous elements (K and per_split multiples of 8, the
// base 16-byte aligned), else K rows; the caller has checked that d ld and 4 ld fit 32 bits and that ws holds the partial tiles.
inline int launch_syrk_chain(const float* X, int64_t d, int64_t K, int64_t ld, bool runs, int nsplit, int64_t per_split, float alpha,
                             float beta, float* C, int64_t ldc, void* ws, hipStream_t stream) {
  SyrkWaveParams p;
  const int64_t T = (d + 63) / 64, tiles = T * (T + 1) / 2;
  p.X = X; p.ld = ld; p.sn = 0; p.K = K; p.per_split = per_split; p.d = static_cast<int>(d); p.run = 0;
  p.T = static_cast<int>(T); p.nsplit = nsplit; p.alpha = alpha; p.beta = beta; p.C = C; p.ldc = ldc; p.ws = static_cast<float*>(ws);
  const dim3 grid(static_cast<unsigned>(tiles * nsplit));
  if (runs) hipLaunchKernelGGL(syrk_chain_kernel<true>, grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL(syrk_chain_kernel<false>, grid, dim3(256), 0, stream, p);
  if (nsplit > 1) launch_syrk_finalize<1>(p.ws, nsplit, tiles, p.T, C, ldc, d, alpha, beta, stream, true);
  return check_launch();
}

// The split of K, into `fewest` parts at least, whose estimated time is shortest: matrix instructions, and for more than one part
// their way through memory and the second launch.
inline int64_t syrk_wave_split(int64_t d, int64_t K, int64_t fewest = 1) {
  const int64_t T = (d + 63) / 64, tiles = T * (T + 1) / 2;
  int64_t best = fewest;
  double least = 1e30;
  for (int64_t s = fewest; s <= std::max<int64_t>(512, fewest); s = s < 8 ? s + 1 : s + s / 8) {
    if (s > fewest && K / s < 64) break;
    const double rounds = static_cast<double>((tiles * s + 255) / 256);
    double t = 5.0 + 0.0133 * static_cast<double>((K + s - 1) / s + 32) * rounds;
    if (s > 1) t += 4.0 + static_cast<double>(tiles * s) * 16384.0 * 2 / 4e6;
    if (t < least) { least = t; best = s; }
  }
  return best;
}

// Rows: while the busiest CU has no more than 1536 of K, or the matrix is at most two tiles wide.  Beyond that the work groups'
// loads of the same rows (each 32 columns of one row at a time) count, and the staged kernel with its 128 x 128 tiles is the
// faster one: staged and here, us: 4096 x 700 (1408 a CU) 45 and 33, 333 x 1999 (999) 47 and 35; 2000 x 1000 (2000) 41 and 50,
// 1000 x 1500 (2000) 50 and 76, 100000 x 256 (4096) 113 and 107; two tiles wide 200000 x 128 87 and 56, 300000 x 64 130 and 29.
inline bool syrk_wave_rows(int64_t d, int64_t K) {
  if (d < 1 || K < 1) return false;
  const int64_t T = (d + 63) / 64, tiles = T * (T + 1) / 2, s = syrk_wave_split(d, K);
  return d <= 128 || (tiles * s + 255) / 256 * ((K + s - 1) / s) <= 1536;
}
inline size_t syrk_wave_ws_bytes(int64_t d, int64_t K) {
  const int64_t T = (d + 63) / 64, s = syrk_wave_split(d, K);
  return s > 1 ? static_cast<size_t>(s) * (T * (T + 1) / 2) * 4096 * sizeof(float) : 0;
}

// run == 0: rows.  The caller has checked alignment (runs: 16-byte loads) and that lane offsets fit 32 bits.
inline int launch_syrk_wave(const float* X, int64_t d, int64_t K, int64_t ld, int64_t sn, int run, float alpha, float beta, float* C,
                            int64_t ldc, void* ws, size_t ws_bytes, hipStream_t stream) {
  SyrkWaveParams p;
  const int64_t T = (d + 63) / 64, tiles = T * (T + 1) / 2;
  int64_t s = syrk_wave_split(d, K);
  p.per_split = ((K + s - 1) / s + 63) / 64 * 64;
  s = (K + p.per_split - 1) / p.per_split;
  if (s > 1 && (ws == nullptr || ws_bytes < static_cast<size_t>(s) * tiles * 4096 * sizeof(float))) return AK_ERR_WORKSPACE;
  p.X = X; p.ld = ld; p.sn = sn; p.K = K; p.d = static_cast<int>(d); p.run = run; p.T = static_cast<int>(T);
  p.nsplit = static_cast<int>(s); p.alpha = alpha; p.beta = beta; p.C = C; p.ldc = ldc; p.ws = static_cast<float*>(ws);
  const dim3 grid(static_cast<unsigned>(tiles * s));        // (d > 2^20 would pass 2^31 - 1: no such matrix fits)
  if (run > 0) hipLaunchKernelGGL(syrk_wave_kernel<true>, grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL(syrk_wave_kernel<false>, grid, dim3(256), 0, stream, p);
  if (s > 1) launch_syrk_finalize<1>(p.ws, p.nsplit, tiles, p.T, C, ldc, d, alpha, beta, stream);
  return check_launch();
}

}  // namespace ak
