// What one step of the block eliminations of chol_sweep.hpp and chol_chain.hpp is made of: a work group of 16 waves forms
//   v_i = Y_i M^T  (Y_i, M: 128 x 128, M lower triangular)   and   X_ij -+ v_i v_j^T
// on the bf16 matrix instructions at the accuracy of fp32, and factors the next diagonal block (chol_leaf.hpp).
//
// Every operand element is split into three bf16 pieces (hi + mid + lo == x: gemm_x3.hpp) once, on its way into the LDS; six
// of the nine piece products count, the five small ones on an accumulator of their own, so that a sum over 128 k rounds
// the large one eight times.  A 128 x 128 x 128 product takes 2.7 us of a CU so, 6.8 on the fp32 matrix instruction, which
// was the most of a step.  Bound by the matrix instructions and the LDS reads of 32 x 32 blocks alike (16 waves: one
// fragment per instruction and operand piece), then by the operands' way from memory.
//
// LDS: an operand's half of 64 k is three planes of [128 rows][64 bf16], 16-byte chunks permuted inside a row by the row (xor
// with row / 2: 16 rows are two lines of banks), which leaves reads of 32 rows and writes of whole chunks without conflicts.
#pragma once
#include "gemm_f32.hpp"
#include "chol_leaf.hpp"
#include <type_traits>

namespace ak {

// A work group of 16 waves takes all vector registers of its CU (128 of each wave), so that no other kernel's waves run there.
// 16-bit matrix instructions disturb some kernels beside them: the host framework's sums over the rows of a bf16 matrix
// (bias gradients), on another stream, lost what 16 lanes of a wave had summed in 479 of 480 runs beside a loop of v_mfma_f32_32x32x16_bf16 or
// _f16, in 278 of 720 beside the framework's own product of 2048 x 2048, and in 311 of 6000 beside inverses of 2 x 4096 whose products left
// half a CU free.  In none of 480 where the loop held the CU's registers or its LDS, nor beside fp32 matrix
// instructions, FMA or LDS loops; alone in none of 6000.  Everything here may run on a stream beside the framework's.
__device__ __forceinline__ void hold_cu() { asm volatile("" ::: "v127"); }

constexpr int ST_TILE = LEAF * LEAF;
constexpr int ST_PLANE = LEAF * 128;                 // bytes of one plane of a half
constexpr int ST_HALF = 3 * ST_PLANE;
constexpr int ST_LDS = 3 * ST_HALF;                  // both halves of M, one of Y; later v_i and v_j, a half each
typedef float st_floatx8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ void st_split(st_floatx8 x, bf16x8 (&o)[3]) {
  o[0] = __builtin_convertvector(x, bf16x8);
  x -= __builtin_convertvector(o[0], st_floatx8);
  o[1] = __builtin_convertvector(x, bf16x8);
  x -= __builtin_convertvector(o[1], st_floatx8);
  o[2] = __builtin_convertvector(x, bf16x8);
}

// One thread's part of a 128 x 128 operand on its way to the LDS: eight consecutive k of one row per half.
struct StPart {
  st_floatx8 v[2];
};

// Element (r, k) at P[r * ld + k], zeros outside rows x cols.
__device__ __forceinline__ void st_fetch(StPart& s, const float* __restrict__ P, int ld, int rows, int cols, int tid) {
  const int r = tid >> 3, c = 8 * (tid & 7);
  if (rows >= LEAF && cols >= LEAF) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const floatx4 q = *reinterpret_cast<const floatx4u*>(P + 64 * h + 4 * u + static_cast<uint32_t>(r * ld + c));      // (128 rows of at most 32768)
#pragma unroll
        for (int e = 0; e < 4; ++e) s.v[h][4 * u + e] = q[e];
      }
    return;
  }
  const float* __restrict__ src = P + static_cast<int64_t>(min(r, rows - 1)) * ld;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = 64 * h + c + e;
      const float x = src[min(k, cols - 1)];         // (loads without conditions; what lies outside is replaced)
      s.v[h][e] = r < rows && k < cols ? x : 0.f;
    }
}
// Element (r, k) at P[k * ld + r]; rows: at least 128.
__device__ __forceinline__ void st_fetch_t(StPart& s, const float* __restrict__ P, int ld, int cols, int tid) {
  const int r = tid & 127, c = 8 * (tid >> 7);
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = 64 * h + c + e;
      const float x = P[static_cast<int64_t>(min(k, cols - 1)) * ld + r];
      s.v[h][e] = k < cols ? x : 0.f;
    }
}
__device__ __forceinline__ void st_stash(const st_floatx8& x, AK_LDS3 unsigned char* half, bool transposed, int tid) {
  const int row = transposed ? tid & 127 : tid >> 3, chunk = transposed ? tid >> 7 : tid & 7;
  bf16x8 o[3];
  st_split(x, o);
  AK_LDS3 unsigned char* dst = half + row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4);
#pragma unroll
  for (int q = 0; q < 3; ++q) *reinterpret_cast<AK_LDS3 bf16x8*>(dst + q * ST_PLANE) = o[q];
}

struct StSum {          // the largest piece products, the five others
  floatx16 big, small;
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int r = 0; r < 16; ++r) big[r] = small[r] = 0.f;
  }
  __device__ __forceinline__ floatx16 value() const {
    floatx16 v;
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = big[r] + small[r];
    return v;
  }
};

// 32 x 32 block: rows `arow` + l % 32 of operand half A, rows `brow` + l % 32 of B, the first STEPS steps of 16 k of the half.
template <int STEPS>
__device__ __forceinline__ void st_mma(StSum& s, AK_LDS3 const unsigned char* A, int arow, AK_LDS3 const unsigned char* B, int brow,
                                       int lane) {
  const int g = lane >> 5, a = arow + (lane & 31), b = brow + (lane & 31);
  AK_LDS3 const unsigned char* pa = A + a * 128;
  AK_LDS3 const unsigned char* pb = B + b * 128;
#pragma unroll 1
  for (int t = 0; t < STEPS; ++t) {             // (four waves a SIMD: fragments read ahead gain nothing and cost 24 registers)
    const int ca = ((2 * t + g) ^ ((a >> 1) & 7)) << 4, cb = ((2 * t + g) ^ ((b >> 1) & 7)) << 4;
    bf16x8 x[3], y[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      x[q] = *reinterpret_cast<AK_LDS3 const bf16x8*>(pa + ca + q * ST_PLANE);
      y[q] = *reinterpret_cast<AK_LDS3 const bf16x8*>(pb + cb + q * ST_PLANE);
    }
    s.small = mfma_bf16(x[1], y[1], s.small);
    s.big = mfma_bf16(x[0], y[0], s.big);
    s.small = mfma_bf16(x[0], y[2], s.small);
    s.small = mfma_bf16(x[2], y[0], s.small);
    s.small = mfma_bf16(x[0], y[1], s.small);
    s.small = mfma_bf16(x[1], y[0], s.small);
  }
}

// v = Y M^T of the staged M (both halves at lds) and of Y, which passes through the third half.  The wave's block comes out
// transposed: register r of lane l is v[32 wr + l % 32][32 wc + 8 (r / 4) + 4 (l / 32) + r % 4].  M is lower triangular: column
// block wc sums k < 32 (wc + 1).  Everybody calls it; the third half is free again after the next barrier.
__device__ __forceinline__ floatx16 st_panel(const StPart& y, bool transposed, AK_LDS3 unsigned char* lds, int wr, int wc, int tid) {
  const int lane = tid & 63;
  AK_LDS3 unsigned char* half = lds + 2 * ST_HALF;
  StSum s;
  s.clear();
  st_stash(y.v[0], half, transposed, tid);
  __syncthreads();
  if (wc == 0) st_mma<2>(s, lds, 0, half, 32 * wr, lane);
  else st_mma<4>(s, lds, 32 * wc, half, 32 * wr, lane);
  __syncthreads();
  st_stash(y.v[1], half, transposed, tid);
  __syncthreads();
  if (wc == 2) st_mma<2>(s, lds + ST_HALF, 64, half, 32 * wr, lane);
  else if (wc == 3) st_mma<4>(s, lds + ST_HALF, 96, half, 32 * wr, lane);
  return s.value();
}

// A wave's block of st_panel() as rows of an operand half (of the half that its columns belong to).
__device__ __forceinline__ void st_put(const floatx16& v, AK_LDS3 unsigned char* half, int wr, int wc, int lane) {
  typedef __bf16 bf16x4v __attribute__((ext_vector_type(4)));
  typedef float floatx4v __attribute__((ext_vector_type(4)));
  const int g = lane >> 5, row = 32 * wr + (lane & 31);
  AK_LDS3 unsigned char* dst = half + row * 128 + 8 * g;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    floatx4v x = {v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
    const int at = ((4 * (wc & 1) + q) ^ ((row >> 1) & 7)) << 4;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const bf16x4v o = __builtin_convertvector(x, bf16x4v);
      *reinterpret_cast<AK_LDS3 bf16x4v*>(dst + at + p * ST_PLANE) = o;
      x -= __builtin_convertvector(o, floatx4v);
    }
  }
}

// This thread's part of M^T, which is v_k of the step's own column, in the registers of a block of st_panel().
__device__ __forceinline__ floatx16 st_own(const float* __restrict__ M, int tid) {
  StPart p;
  st_fetch_t(p, M, LEAF, LEAF, tid);
  floatx16 v;
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = p.v[r >> 3][r & 7];
  return v;
}

// v_i v_j^T: register r of lane l of wave (wr, wc) is element (32 wr + 8 (r / 4) + 4 (l / 32) + r % 4, 32 wc + l % 32).
// own_i, own_j: that operand comes from st_own(); same: v_j = v_i.
__device__ __forceinline__ floatx16 st_outer(const floatx16& vi, bool own_i, const floatx16& vj, bool own_j, bool same,
                                             AK_LDS3 unsigned char* lds, int wr, int wc, int tid) {
  const int lane = tid & 63;
  StSum s;
  s.clear();
  auto half = [&](auto h_tag) {
    constexpr int h = decltype(h_tag)::value;
    auto put = [&](const floatx16& v, bool own, AK_LDS3 unsigned char* dst) {
      if (own) {
        st_floatx8 x;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = v[8 * h + e];
        st_stash(x, dst, true, tid);
      } else if ((wc >> 1) == h) {
        st_put(v, dst, wr, wc, lane);
      }
    };
    __syncthreads();
    put(vi, own_i, lds);
    if (!same) put(vj, own_j, lds + ST_HALF);
    __syncthreads();
    st_mma<4>(s, lds, 32 * wr, same ? lds : lds + ST_HALF, 32 * wc, lane);
  };
  half(std::integral_constant<int, 0>{});
  half(std::integral_constant<int, 1>{});
  return s.value();
}

// The next diagonal block is updated by blocks (a, b) of 32 x 32, a <= b, one to each of the first ten waves, on its way to
// the leaf: register 4 q + e of lane l stands for element (32 b + l % 32, 32 a + 8 q + 4 (l / 32) + e) of its lower triangle.
__device__ __forceinline__ void st_leaf_block(int wave, int& a, int& b) {      // (integers only: branches on them have to be scalar)
  b = wave >= 10 ? 4 : (wave >= 1) + (wave >= 3) + (wave >= 6);
  a = wave - b * (b + 1) / 2;
}

// The wave's block before the update; n: columns of the diagonal block inside the matrix; old(i, j) gives elements
// (i, j ... j + 3) of its lower triangle, i and j below n.  Called before the products, so that it is under way while they run.
template <class Old>
__device__ __forceinline__ void st_leaf_fetch(floatx16& upd, Old&& old, int n, int tid) {
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int a, b;
  st_leaf_block(wave, a, b);
#pragma unroll
  for (int r = 0; r < 16; ++r) upd[r] = 0.f;
  if (b < 4 && 32 * b < n) {
    const int i = 32 * b + (lane & 31), j = 32 * a + 4 * (lane >> 5);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const floatx4 x = old(min(i, n - 1), min(j + 8 * q, n - 1 & ~3));
#pragma unroll
      for (int e = 0; e < 4; ++e) upd[4 * q + e] = x[e];
    }
  }
}

// The next diagonal block, updated by v (has_v: the wave's block of st_panel() of its row) and factored.  M = L^-1 goes to
// Mn [128][128] and through store_t(i, j, four) its transpose: elements (i + l % 16, j + 4 (l / 16) ... + 3) of M^T, the zeros
// below its diagonal included.  Returns the first bad pivot, 0 if none.
template <class StoreT>
__device__ __forceinline__ int st_leaf(floatx16& upd, StoreT&& store_t, const floatx16& v, bool has_v, int n, float* __restrict__ Mn,
                                       AK_LDS3 unsigned char* lds, LeafShared& sh, int wr, int wc, int tid) {
  asm volatile("" : "+v"(tid));       // (keeps the address arithmetic below the products)
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g4 = lane >> 4, c = lane & 15;
  const int nb = (n + LT - 1) / LT;
  int a, b;
  st_leaf_block(wave, a, b);
  if (has_v) {
    __syncthreads();
    st_put(v, lds + (wc >> 1) * ST_HALF, wr, wc, lane);
    __syncthreads();
  }
  AK_LDS3 floatx4* handed = reinterpret_cast<AK_LDS3 floatx4*>(lds + 2 * ST_HALF);      // (36 KB of the third half)
  if (b < 4 && 32 * b < n) {
    if (has_v) {
      StSum s;
      s.clear();
      st_mma<4>(s, lds, 32 * a, lds, 32 * b, lane);
      st_mma<4>(s, lds + ST_HALF, 32 * a, lds + ST_HALF, 32 * b, lane);
#pragma unroll
      for (int r = 0; r < 16; ++r) upd[r] -= s.big[r] + s.small[r];
    }
    const int i = 32 * b + (lane & 31), g = lane >> 5;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = 32 * a + 8 * q + 4 * g, ts = 2 * a + (q >> 1), tc = 2 * b + ((lane >> 4) & 1);
      floatx4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = upd[4 * q + e];
        if (i >= n) x[e] = i == j + e ? 1.f : 0.f;      // identity padding
        if (j + e > i) x[e] = 0.f;
      }
      // tile (ts, tc) of 16 x 16 of U's side: element (16 ts + 4 g4 + e, 16 tc + c) by lane 16 g4 + c
      if (ts <= tc) handed[(tc * (tc + 1) / 2 + ts) * 64 + 16 * (2 * (q & 1) + g) + c] = x;
    }
  }
  __syncthreads();
  const int bad = leaf_eliminate(
      nb, sh, wave, lane, [&](int s, int col) { return handed[(col * (col + 1) / 2 + s) * 64 + lane]; },
      [&](int s, int col, const floatx4& x) {
        // (addresses as a uniform part and a 32-bit one of the lane, which all tiles share: as 64-bit ones of the lane they were
        // formed ahead of the elimination and took its registers)
        float* __restrict__ to = Mn + LT * s * LEAF + LT * col;
#pragma unroll
        for (int r = 0; r < 4; ++r) to[static_cast<uint32_t>((4 * g4 + r) * LEAF + c)] = x[r];
        store_t(LT * col, LT * s, x);
        if (s != col) {
          const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
          *reinterpret_cast<floatx4*>(Mn + LT * col * LEAF + LT * s + static_cast<uint32_t>(c * LEAF + 4 * g4)) = zero;
          store_t(LT * s, LT * col, zero);
        }
      });
  if (nb < LEAF_TILES) {         // the identity beyond the matrix
    for (int e = tid; e < ST_TILE; e += LEAF_THREADS) {
      const int i = e / LEAF, j = e % LEAF;
      if (i >= LT * nb || j >= LT * nb) Mn[e] = i == j ? 1.f : 0.f;
    }
  }
  return bad;
}

}  // namespace ak
