// fp32 product tile for products that leave most of the device idle: true fp32 products (v_mfma_f32_32x32x2_f32), small
// tiles, deep k-chunks.  Included by gemm_f32.hpp; same interface (GemmParams).
// (Most products take gemm_wave.hpp, without the LDS; this form stays for short contractions over more tiles than CUs, A B^T
// over many tiles, the inverses' small products and those of the low-rank inverses.)
//
// A product of a few hundred rows is bound by memory latency, not by the matrix pipes: with k-tiles of 16 or 32 and one
// of them in flight, every k-tile waits for the L2 or the device memory once (about a microsecond when the operands were
// just written by another XCD).  Here a work group requests a whole chunk of KC columns of both operands (KC = 128: 16
// 16-byte loads per thread) before it touches the first, and the next chunk while the matrix instructions of this one run
// (4096 cycles for 64 x 64 x 128).  K = 128: 11.5 us -> 7.3 us per launch against the 128 x 128 split tile; K = 784, 28
// tiles of 128: 45 -> 27 us.  Loads of 16 bytes need 4-byte alignment only, so ragged leading dimensions take the
// same path.
//
// One work group = 4 waves of one 32 x 32 block each (BM x BN = 64 x 64 or 32 x 128).  An operand whose contraction index
// is contiguous in memory is kept in the LDS as [row][KC + 4] and read four k at a time (ds_read_b128), one whose row
// index is contiguous as [k][rows + 8]; lane group g of a wave takes k = 8 q + 4 g + e in step 4 q + e of either.
#pragma once
#include "common.hpp"

namespace ak {

typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

template <int R, int KC> struct DeepPanel {
  static constexpr int KC_LD = KC + 4, IC_LD = R + 8;
  static constexpr int FLOATS = R * KC_LD > KC * IC_LD ? R * KC_LD : KC * IC_LD;
  static constexpr int CHUNKS = R * KC / 4 / 256;       // 16-byte loads per thread
  typedef floatx4 Regs[CHUNKS];
};

// No branch around a load (a load under a lane's own condition is waited for before the next one leaves): a panel inside the
// operand is read as it lies, from a uniform address per load and one lane offset; a chunk beyond an edge reads the last one
// inside, shifts it and counts as zeros from the edge on.  1000^3: 57 -> 40 us; 300 x 75 x 300: 20 -> 17.
template <int R, int KC>
__device__ __forceinline__ void deep_fetch(typename DeepPanel<R, KC>::Regs& reg, const float* __restrict__ P,
                                           int64_t ld, bool kcontig, int r0, int r_end, int k0, int k_end, int tid) {
  const int o0 = kcontig ? r0 : k0, i0 = kcontig ? k0 : r0, o_end = kcontig ? r_end : k_end, i_end = kcontig ? k_end : r_end;
  const int row_chunks = kcontig ? KC / 4 : R / 4, step = 256 / row_chunks;       // chunks of a memory row; rows per 256 chunks
  const int outer = tid / row_chunks, inner = 4 * (tid % row_chunks);
  const float* __restrict__ base = P + static_cast<int64_t>(o0) * ld + i0;
  if (o0 + (kcontig ? R : KC) <= o_end && i0 + (kcontig ? KC : R) <= i_end) {
    const int64_t at = static_cast<int64_t>(outer) * ld + inner;
#pragma unroll
    for (int u = 0; u < DeepPanel<R, KC>::CHUNKS; ++u) reg[u] = *reinterpret_cast<const floatx4u*>(base + u * step * ld + at);
  } else if (i_end >= 4) {
    const int first = i_end - 4 < i0 + inner ? i_end - 4 : i0 + inner, shift = i0 + inner - first;
#pragma unroll
    for (int u = 0; u < DeepPanel<R, KC>::CHUNKS; ++u) {
      const int row = o0 + outer + u * step;
      reg[u] = *reinterpret_cast<const floatx4u*>(P + static_cast<int64_t>(row < o_end ? row : o_end - 1) * ld + first);
    }
#pragma unroll
    for (int u = 0; u < DeepPanel<R, KC>::CHUNKS; ++u) {
      const floatx4 w = reg[u];
      const bool in = o0 + outer + u * step < o_end;
      floatx4 v;
      v[0] = shift == 0 ? w[0] : shift == 1 ? w[1] : shift == 2 ? w[2] : w[3];
      v[1] = shift == 0 ? w[1] : shift == 1 ? w[2] : w[3];
      v[2] = shift == 0 ? w[2] : w[3];
      v[3] = w[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) reg[u][e] = in && shift + e < 4 ? v[e] : 0.f;
    }
  } else {
#pragma unroll
    for (int u = 0; u < DeepPanel<R, KC>::CHUNKS; ++u) {
      const int row = o0 + outer + u * step;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        reg[u][e] = row < o_end && i0 + inner + e < i_end ? P[static_cast<int64_t>(row) * ld + i0 + inner + e] : 0.f;
    }
  }
}

template <int R, int KC>
__device__ __forceinline__ void deep_stash(const typename DeepPanel<R, KC>::Regs& reg, float* __restrict__ lds,
                                           bool kcontig, int tid) {
  using P = DeepPanel<R, KC>;
#pragma unroll
  for (int u = 0; u < P::CHUNKS; ++u) {
    const int c = tid + 256 * u;
    const int off = kcontig ? (c / (KC / 4)) * P::KC_LD + 4 * (c % (KC / 4)) : (c / (R / 4)) * P::IC_LD + 4 * (c % (R / 4));
    *reinterpret_cast<floatx4*>(lds + off) = reg[u];
  }
}

// acc += the product of the chunk in the LDS, for this wave's 32 x 32 block.  pa / pb: its first operand element.
template <int BM, int BN, int KC, bool A_KC, bool B_KC>
__device__ __forceinline__ void deep_chunk(floatx16 (&acc)[4], const float* __restrict__ pa, const float* __restrict__ pb) {
  constexpr int LA = A_KC ? 1 : DeepPanel<BM, KC>::IC_LD, LB = B_KC ? 1 : DeepPanel<BN, KC>::IC_LD;
#pragma unroll 4
  for (int q = 0; q < KC / 8; ++q) {
    floatx4 a, b;
    if constexpr (A_KC) a = *reinterpret_cast<const floatx4*>(pa + 8 * q);
    else
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = pa[(8 * q + e) * LA];
    if constexpr (B_KC) b = *reinterpret_cast<const floatx4*>(pb + 8 * q);
    else
#pragma unroll
      for (int e = 0; e < 4; ++e) b[e] = pb[(8 * q + e) * LB];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = mfma_f32(a[e], b[e], acc[e]);
  }
}

template <int BM, int BN, int KC>
constexpr int deep_lds_floats() { return DeepPanel<BM, KC>::FLOATS + DeepPanel<BN, KC>::FLOATS; }

// One BM x BN tile (ti, tj) of batch entry z of the product described by p; lds: deep_lds_floats() floats.  The sum is
// always taken in chunks: a fresh accumulator for every KC of the contraction, added to a running total.  The rounding
// error of a long sum stays near that of one rounding instead of growing with the number of matrix instructions.
template <int BM, int BN, int KC>
__device__ __forceinline__ void gemm_deep_tile(const GemmParams& p, int ti, int tj, int z, float* lds) {
  static_assert((BM / 32) * (BN / 32) == 4, "four waves");
  using PA = DeepPanel<BM, KC>;
  using PB = DeepPanel<BN, KC>;
  if (p.active != nullptr && p.active[static_cast<int64_t>(z) * p.active_stride] == 0) return;
  const int i0 = ti * BM, j0 = tj * BN;
  if (p.tile_mode != TILE_ALL && i0 + BM <= j0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = wave / (BN / 32), wc = wave % (BN / 32), g = lane >> 5, l32 = lane & 31;

  int kbeg = 0, kend = p.K;
  switch (p.kmode) {     // ranges rounded outwards to multiples of the tile; the operands are zero outside their triangle
    case K_LE_J: kend = min(p.K, j0 + BN); break;
    case K_GE_J: kbeg = j0; break;
    case K_LE_I: kend = min(p.K, i0 + BM); break;
    case K_GE_MAXIJ: kbeg = max(i0, j0); break;
    default: break;
  }
  const float* __restrict__ A = p.A + static_cast<int64_t>(z) * p.sA;
  const float* __restrict__ B = p.B + static_cast<int64_t>(z) * p.sB;
  float* __restrict__ C = p.C_list != nullptr ? p.C_list[z] : p.C + static_cast<int64_t>(z) * p.sC;
  const bool a_kc = (p.transA == 0), b_kc = (p.transB != 0);
  float* ldsA = lds;
  float* ldsB = lds + PA::FLOATS;
  const int ra0 = 32 * wr + l32, rb0 = 32 * wc + l32;
  const float* pa = ldsA + (a_kc ? ra0 * PA::KC_LD + 4 * g : 4 * g * PA::IC_LD + ra0);
  const float* pb = ldsB + (b_kc ? rb0 * PB::KC_LD + 4 * g : 4 * g * PB::IC_LD + rb0);

  // Four accumulators per block, added up after every chunk: the matrix instruction rounds its accumulator once per two
  // k, and a sum of K / 2 roundings in a row shows in the inverses of ill-conditioned factors.
  floatx16 part[4], acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = part[0][r] = part[1][r] = part[2][r] = part[3][r] = 0.f;
  typename PA::Regs ra;
  typename PB::Regs rb;
  if (kbeg < kend) {
    deep_fetch<BM, KC>(ra, A, p.lda, a_kc, i0, p.M, kbeg, kend, tid);
    deep_fetch<BN, KC>(rb, B, p.ldb, b_kc, j0, p.N, kbeg, kend, tid);
  }
  for (int k0 = kbeg; k0 < kend; k0 += KC) {
    if (k0 != kbeg) __syncthreads();
    deep_stash<BM, KC>(ra, ldsA, a_kc, tid);
    deep_stash<BN, KC>(rb, ldsB, b_kc, tid);
    __syncthreads();
    if (k0 + KC < kend) {
      deep_fetch<BM, KC>(ra, A, p.lda, a_kc, i0, p.M, k0 + KC, kend, tid);
      deep_fetch<BN, KC>(rb, B, p.ldb, b_kc, j0, p.N, k0 + KC, kend, tid);
    }
    if (a_kc) {
      if (b_kc) deep_chunk<BM, BN, KC, true, true>(part, pa, pb);
      else deep_chunk<BM, BN, KC, true, false>(part, pa, pb);
    } else {
      if (b_kc) deep_chunk<BM, BN, KC, false, true>(part, pa, pb);
      else deep_chunk<BM, BN, KC, false, false>(part, pa, pb);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[r] += (part[0][r] + part[1][r]) + (part[2][r] + part[3][r]);
      part[0][r] = part[1][r] = part[2][r] = part[3][r] = 0.f;
    }
  }

  // mirrored results are exactly symmetric: a tile on the diagonal keeps its lower triangle and mirrors it as well
  const bool lower_only = p.tile_mode != TILE_ALL;
  const bool mirror = p.tile_mode == TILE_LOWER_MIRROR;
  float* __restrict__ C2 = p.C2 != nullptr ? p.C2 + static_cast<int64_t>(z) * p.sC2 : nullptr;
  float vmax = 0.f;
  const int gj = j0 + 32 * wc + l32;
  if (gj < p.N) {
    const int gi0 = i0 + 32 * wr + 4 * g;
    if (p.beta != 0.f) {
      // all reads of the old result before the first store, so that they are in flight together
      float old[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int gi = gi0 + 8 * (r >> 2) + (r & 3);
        old[r] = C[static_cast<int64_t>(min(gi, p.M - 1)) * p.ldc + gj];
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = p.alpha * acc[r] + p.beta * old[r];
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[r] *= p.alpha;
        if (gi0 + 8 * (r >> 2) + (r & 3) == gj) acc[r] += p.diag;
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int gi = gi0 + 8 * (r >> 2) + (r & 3);
      if (gi >= p.M || (lower_only && gi < gj)) continue;
      C[static_cast<int64_t>(gi) * p.ldc + gj] = acc[r];
      vmax = gemm_fold_absmax(vmax, acc[r], gi == gj, p.absmax_identity);
      if (C2 != nullptr) C2[static_cast<int64_t>(gi) * p.ldc2 + gj] = p.c2_scale * acc[r] + (gi == gj ? p.c2_diag : 0.f);
    }
    if (mirror) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int gi = gi0 + 8 * q;
        const floatx4 v = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
        float* dst = C + static_cast<int64_t>(gj) * p.ldc + gi;
        if (gi > gj && gi + 4 <= p.M) *reinterpret_cast<floatx4u*>(dst) = v;
        else
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (gi + e > gj && gi + e < p.M) dst[e] = v[e];
        if (C2 != nullptr) {
          float* dst2 = C2 + static_cast<int64_t>(gj) * p.ldc2 + gi;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (gi + e > gj && gi + e < p.M) dst2[e] = p.c2_scale * v[e];
        }
      }
    }
  }
  if (p.absmax_out != nullptr) gemm_store_absmax(p.absmax_out + static_cast<int64_t>(z) * p.absmax_stride, vmax, lane);
}

static __global__ __launch_bounds__(256) void gemm_deep_kernel(GemmParams p) {
  __shared__ __attribute__((aligned(16))) float deep_lds[deep_lds_floats<64, 64, 128>()];
  // rows of tiles, which read the same rows of A, side by side on one XCD
  const uint32_t id = xcd_contiguous_id((blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x, gridDim.x * gridDim.y * gridDim.z);
  const uint32_t row = id / gridDim.x;
  gemm_deep_tile<64, 64, 128>(p, row % gridDim.y, id % gridDim.x, row / gridDim.y, deep_lds);
}

}  // namespace ak
