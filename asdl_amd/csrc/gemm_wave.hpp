// fp32 product tile for products that leave most of the device idle: true fp32 products (v_mfma_f32_32x32x2_f32), operands
// straight from memory to the matrix instruction.  Included by gemm_f32.hpp; same interface (GemmParams).
//
// A work group owns a 64 x 64 tile; each of its eight waves sums the whole tile over every eighth batch of 16 k, and the waves'
// sums are added through the LDS.  No staging, no barrier before the sums, and every load of the next batch is in flight while
// the 32 matrix instructions of this one run (2048 cycles, two waves per SIMD).  The k of a batch are dealt so that an operand
// with contiguous contraction comes in 16-byte loads and one with contiguous rows in 8-byte loads, two rows per lane (whole rows
// of the tile per load, which is the faster of the two: A B^T at 1024^3 30 us, A B 25).  Loads need 4-byte alignment only.
//
// Bound by the fp32 matrix instruction (1.75 us per 128 k and CU) and the way of 64 + 64 operand rows per tile from the L2.
// Errors against 64 bits of 60 products of 8 to 2048 x 8 to 2048 x 8 to 4096: 0.93 of the staged tile's in the mean, 1.08 at most.
// Measured against the tile staged through the LDS (gemm_deep.hpp), us: 64^3 9.3 and 7.7, 512 x 784 x 784 41 and 21,
// 1153 x 512 x 1153 45 and 29, 577 x 1000 x 1000 47 and 26, 1000^3 57 and 27, 300 x 300 x 20000 1084 and 557.
#pragma once
#include "common.hpp"

namespace ak {

template <int WAVES> constexpr int wave_lds_floats() { return WAVES * 4096; }

// Where a lane finds its rows of an operand: block c's row 32 c + l (contiguous contraction), or 2 l + c (contiguous rows: both
// blocks' rows in one 8-byte load).
struct WaveRows {
  uint32_t at[2];            // offsets of the rows of both blocks
  int pair;                  // and of the 8-byte load: -1 (the last row of the tile before) where one row is left
  bool odd;                  // the load's second half is block 0's row: the operand ends there
};
template <bool KC>
__device__ __forceinline__ WaveRows wave_rows(int64_t ld, int left, int l32, int g) {
  // rows beyond the operand (left: of it from the tile's first on) read its last one: their sums are not stored
  WaveRows w;
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int row = min(KC ? 32 * c + l32 : 2 * l32 + c, left - 1);
    w.at[c] = KC ? static_cast<uint32_t>(row) * static_cast<uint32_t>(ld) + 4 * g : 4 * g * static_cast<uint32_t>(ld) + row;
  }
  w.odd = 2 * l32 == left - 1;
  w.pair = 4 * g * static_cast<int>(ld) + min(2 * l32, left - 2);
  return w;
}

typedef float floatx2u __attribute__((ext_vector_type(2), aligned(4)));

// 16 k of both blocks: x[c][4 t + e] is k = 8 t + 4 g + e.  src: uniform, the operand at (first k, first row of the tile)
struct WaveBatch { float x[2][8]; };
template <bool KC>
__device__ __forceinline__ void wave_fetch(WaveBatch& f, const float* __restrict__ src, int64_t ld, const WaveRows& w) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
    if constexpr (KC) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const floatx4 v = *reinterpret_cast<const floatx4u*>(src + 8 * t + w.at[c]);
#pragma unroll
        for (int e = 0; e < 4; ++e) f.x[c][4 * t + e] = v[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const floatx2u v = *reinterpret_cast<const floatx2u*>(src + (8 * t + e) * ld + w.pair);
        f.x[0][4 * t + e] = v[0];
        f.x[1][4 * t + e] = v[1];
      }
    }
}
template <bool KC>
__device__ __forceinline__ void wave_settle(WaveBatch& f, const WaveRows& w) {
  if constexpr (!KC)
#pragma unroll
    for (int u = 0; u < 8; ++u) f.x[0][u] = w.odd ? f.x[1][u] : f.x[0][u];
}

// One element at a time: the last, incomplete batch (elements beyond its `rest` k read the last k and count as zeros) and
// operands of a single row.
template <bool KC>
__device__ __forceinline__ void wave_fetch_rest(WaveBatch& f, const float* __restrict__ src, int64_t ld, const WaveRows& w, int rest, int g) {
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = 8 * t + 4 * g + e, back = k < rest ? 0 : k - (rest - 1);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const float* __restrict__ q = KC ? src + 8 * t + e : src + (8 * t + e) * ld;
        const float v = q[static_cast<int64_t>(w.at[c]) - back * (KC ? 1 : ld)];
        f.x[c][4 * t + e] = k < rest ? v : 0.f;
      }
    }
}

// Wave `wave` of WAVES sums the batches of 16 k number wave, wave + WAVES, ...: the waves read the same cache lines of an operand
// with contiguous contraction at about the same time.
template <int WAVES, bool A_KC, bool B_KC>
__device__ __forceinline__ void wave_sum(floatx16 (&tot)[2][2], const float* __restrict__ A, int64_t lda, const float* __restrict__ B, int64_t ldb,
                                         int left_a, int left_b, bool single, int kbeg, int kend, int wave, int l32, int g) {
  const WaveRows ra = wave_rows<A_KC>(lda, left_a, l32, g), rb = wave_rows<B_KC>(ldb, left_b, l32, g);
  const int full = max(kend - kbeg, 0) / 16, k = kbeg + 16 * wave;
  int batches = full > wave ? (full - wave + WAVES - 1) / WAVES : 0;
  const int rest = full % WAVES == wave ? max(kend - kbeg, 0) % 16 : 0;
  const float* __restrict__ sa = A_KC ? A + k : A + k * lda;
  const float* __restrict__ sb = B_KC ? B + k : B + k * ldb;
  const int64_t step_a = A_KC ? 16 * WAVES : 16 * WAVES * lda, step_b = B_KC ? 16 * WAVES : 16 * WAVES * ldb;
  struct Pair { WaveBatch a, b; };
  // (always a load, of the last batch again at the end: a fetch under a condition makes every use wait for all loads)
  auto fetch = [&](Pair& f, int batch) {
    const int at = min(batch, batches - 1);
    wave_fetch<A_KC>(f.a, sa + at * step_a, lda, ra);
    wave_fetch<B_KC>(f.b, sb + at * step_b, ldb, rb);
  };
  auto multiply = [&](floatx16 (&acc)[2][2], Pair& f) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = mfma_f32(f.a.x[a][u], f.b.x[b][u], acc[a][b]);
  };
  auto clear = [&](floatx16 (&acc)[2][2]) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
  };
  auto flush = [&](const floatx16 (&acc)[2][2]) {
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[a][b][r] += acc[a][b][r];
  };
  floatx16 acc[2][2];
  Pair f0, f1;
  // A batch by itself, on two accumulators: it is a wave's whole sum where the contraction is short, and eight instructions in a row
  // that round at its magnitude show there (zero-mean operands, 15, 25, 52 k: 7.0, 7.5, 8.6e-8 on one, 5.6, 6.2, 6.9e-8 so, 5.5, 6.1,
  // 7.2e-8 on the four of gemm_deep.hpp; 0.15 us)
  auto by_itself = [&](Pair& f) {
    floatx16 odd[2][2];
    clear(acc);
    clear(odd);
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          if (u & 1) odd[a][b] = mfma_f32(f.a.x[a][u], f.b.x[b][u], odd[a][b]);
          else acc[a][b] = mfma_f32(f.a.x[a][u], f.b.x[b][u], acc[a][b]);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) tot[a][b][r] += acc[a][b][r] + odd[a][b][r];
  };
  auto fetch_few = [&](int batch, int n) {
    wave_fetch_rest<A_KC>(f0.a, sa + batch * step_a, lda, ra, n, g);
    wave_fetch_rest<B_KC>(f0.b, sb + batch * step_b, ldb, rb, n, g);
  };
  auto settle = [&](Pair& f) {
    wave_settle<A_KC>(f.a, ra);
    wave_settle<B_KC>(f.b, rb);
  };
  if (single) {
    for (int b = 0; b < batches; ++b) {
      fetch_few(b, 16);
      clear(acc);
      multiply(acc, f0);
      flush(acc);
    }
  } else if (batches > 0) {
    fetch(f0, 0);
    int b = 0;
    for (; b + 2 <= batches; b += 2) {
      fetch(f1, b + 1);
      __builtin_amdgcn_sched_barrier(0);         // (all loads of a batch leave before the products of the one before)
      clear(acc);
      settle(f0);
      multiply(acc, f0);
      __builtin_amdgcn_sched_barrier(0);
      fetch(f0, b + 2);
      __builtin_amdgcn_sched_barrier(0);
      settle(f1);
      multiply(acc, f1);
      flush(acc);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (b < batches) {                            // (the last batch of an odd number)
      settle(f0);
      by_itself(f0);
    }
  }
  if (rest > 0) {
    fetch_few(batches, rest);
    by_itself(f0);
  }
}

// One 64 x 64 tile (ti, tj) of batch entry z of the product described by p; lds: wave_lds_floats() floats, all waves of the
// work group.
template <int WAVES>
__device__ __forceinline__ void gemm_wave_tile(const GemmParams& p, int ti, int tj, int z, float* lds) {
  if (p.active != nullptr && p.active[static_cast<int64_t>(z) * p.active_stride] == 0) return;
  const int i0 = ti * 64, j0 = tj * 64;
  if (p.tile_mode != TILE_ALL && i0 + 64 <= j0) return;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int kbeg = 0, kend = p.K;
  switch (p.kmode) {     // ranges rounded outwards to multiples of the tile; the operands are zero outside their triangle
    case K_LE_J: kend = min(p.K, j0 + 64); break;
    case K_GE_J: kbeg = j0; break;
    case K_LE_I: kend = min(p.K, i0 + 64); break;
    case K_GE_MAXIJ: kbeg = max(i0, j0); break;
    default: break;
  }
  const bool a_kc = (p.transA == 0), b_kc = (p.transB != 0);
  const float* __restrict__ A = p.A + static_cast<int64_t>(z) * p.sA + (a_kc ? i0 * p.lda : i0);
  const float* __restrict__ B = p.B + static_cast<int64_t>(z) * p.sB + (b_kc ? j0 * p.ldb : j0);
  float* __restrict__ C = p.C_list != nullptr ? p.C_list[z] : p.C + static_cast<int64_t>(z) * p.sC;
  floatx16 tot[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) tot[a][b][r] = 0.f;
  const int left_a = p.M - i0, left_b = p.N - j0;
  const bool single = (!a_kc && p.M == 1) || (!b_kc && p.N == 1);      // (no second row to load eight bytes from)
  if (a_kc) {
    if (b_kc) wave_sum<WAVES, true, true>(tot, A, p.lda, B, p.ldb, left_a, left_b, single, kbeg, kend, wave, l32, g);
    else wave_sum<WAVES, true, false>(tot, A, p.lda, B, p.ldb, left_a, left_b, single, kbeg, kend, wave, l32, g);
  } else {
    if (b_kc) wave_sum<WAVES, false, true>(tot, A, p.lda, B, p.ldb, left_a, left_b, single, kbeg, kend, wave, l32, g);
    else wave_sum<WAVES, false, false>(tot, A, p.lda, B, p.ldb, left_a, left_b, single, kbeg, kend, wave, l32, g);
  }
  floatx4* part = reinterpret_cast<floatx4*>(lds);
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        part[((wave * 4 + 2 * a + b) * 4 + q) * 64 + lane] = floatx4{tot[a][b][4 * q], tot[a][b][4 * q + 1], tot[a][b][4 * q + 2], tot[a][b][4 * q + 3]};
  __syncthreads();
  // wave w finishes QUADS register quads of block w % 4
  constexpr int QUADS = 16 / WAVES;
  const int block = wave & 3, q0 = (wave >> 2) * QUADS, wr = block >> 1, wc = block & 1;
  floatx4 acc[QUADS];
#pragma unroll
  for (int q = 0; q < QUADS; ++q) {
    floatx4 v[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v[w] = part[((w * 4 + block) * 4 + q0 + q) * 64 + lane];
#pragma unroll
    for (int h = WAVES / 2; h > 0; h >>= 1)
#pragma unroll
      for (int w = 0; w < h; ++w) v[w] += v[w + h];
    acc[q] = v[0];
  }

  // mirrored results are exactly symmetric: a tile on the diagonal keeps its lower triangle and mirrors it as well
  const bool lower_only = p.tile_mode != TILE_ALL;
  const bool mirror = p.tile_mode == TILE_LOWER_MIRROR;
  float* __restrict__ C2 = p.C2 != nullptr ? p.C2 + static_cast<int64_t>(z) * p.sC2 : nullptr;
  float vmax = 0.f;
  const int gj = j0 + (b_kc ? 32 * wc + l32 : 2 * l32 + wc);
  const int gi0 = i0 + (a_kc ? 32 * wr + 8 * q0 + 4 * g : 2 * (8 * q0 + 4 * g) + wr), di = a_kc ? 1 : 2;
  auto row = [&](int r) { return gi0 + di * (8 * (r >> 2) + (r & 3)); };
  if (gj < p.N) {
    if (p.beta != 0.f) {
      // all reads of the old result before the first store, so that they are in flight together
      float old[4 * QUADS];
#pragma unroll
      for (int r = 0; r < 4 * QUADS; ++r) old[r] = C[static_cast<int64_t>(min(row(r), p.M - 1)) * p.ldc + gj];
#pragma unroll
      for (int r = 0; r < 4 * QUADS; ++r) acc[r >> 2][r & 3] = p.alpha * acc[r >> 2][r & 3] + p.beta * old[r];
    } else {
#pragma unroll
      for (int r = 0; r < 4 * QUADS; ++r) {
        acc[r >> 2][r & 3] *= p.alpha;
        if (row(r) == gj) acc[r >> 2][r & 3] += p.diag;
      }
    }
#pragma unroll
    for (int r = 0; r < 4 * QUADS; ++r) {
      const int gi = row(r);
      const float v = acc[r >> 2][r & 3];
      if (gi >= p.M || (lower_only && gi < gj)) continue;
      C[static_cast<int64_t>(gi) * p.ldc + gj] = v;
      vmax = gemm_fold_absmax(vmax, v, gi == gj, p.absmax_identity);
      if (C2 != nullptr) C2[static_cast<int64_t>(gi) * p.ldc2 + gj] = p.c2_scale * v + (gi == gj ? p.c2_diag : 0.f);
      if (mirror && gi > gj) {
        C[static_cast<int64_t>(gj) * p.ldc + gi] = v;
        if (C2 != nullptr) C2[static_cast<int64_t>(gj) * p.ldc2 + gi] = p.c2_scale * v;
      }
    }
  }
  if (p.absmax_out != nullptr) gemm_store_absmax(p.absmax_out + static_cast<int64_t>(z) * p.absmax_stride, vmax, lane);
}

constexpr int GEMM_WAVES = 8;

// Offsets inside a tile's operand rows are kept in 32 bits.
inline bool gemm_wave_ok(const GemmParams& p) { return p.lda < (1 << 24) && p.ldb < (1 << 24); }

static __global__ __launch_bounds__(64 * GEMM_WAVES, 2) void gemm_wave_kernel(GemmParams p) {
  __shared__ __attribute__((aligned(16))) float wave_lds[wave_lds_floats<GEMM_WAVES>()];
  // rows of tiles, which read the same rows of A, side by side on one XCD
  const uint32_t id = xcd_contiguous_id((blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x, gridDim.x * gridDim.y * gridDim.z);
  const uint32_t row = id / gridDim.x;
  gemm_wave_tile<GEMM_WAVES>(p, row % gridDim.y, id % gridDim.x, row / gridDim.y, wave_lds);
}

}  // namespace ak
